"""A download whose helper thread fails reports the failure and has waited for
the kernels it started, also when the helper held the last outstanding chunk."""
import os
import subprocess

import pytest

from tests.conftest import ROOT


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = tmp_path_factory.mktemp("download") / "download_failures"
    cpp = os.path.join(ROOT, "tests", "cpp")
    r = subprocess.run(["g++", "-O2", "-std=c++17", "-pthread", "-I", os.path.join(cpp, "host_hip"),
                        os.path.join(cpp, "download_failures.cc"), "-o", str(out)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return str(out)


@pytest.mark.parametrize("mode", ["none", "pack", "record"])
def test_failed_chunk_is_an_error(exe, mode):
    r = subprocess.run([exe, mode], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr
    trials, errors, silent, wrong, unwaited = map(int, r.stdout.split())
    assert errors == (0 if mode == "none" else trials)
    assert silent == wrong == unwaited == 0
