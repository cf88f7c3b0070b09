"""A download whose helper thread fails reports the failure and has waited for
the kernels it started, also when the helper held the last outstanding chunk.
Helpers come once the stream's earlier work is done: they would wait for it on
CPUs that the program's own threads may want."""
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


def run(exe, mode):
    r = subprocess.run([exe, mode], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr
    print(mode, r.stdout)
    return map(int, r.stdout.split())


@pytest.mark.parametrize("mode", ["pack", "record"])
def test_failed_chunk_is_an_error(exe, mode):
    trials, helped, errors, silent, unwaited = run(exe, mode)
    if helped == 0:
        pytest.skip("no idle CPU for a helper")
    assert errors == helped
    assert silent == unwaited == 0


@pytest.mark.parametrize("mode", ["none", "late"])
def test_helpers_come_late(exe, mode):
    trials, helped, errors, silent, unwaited = run(exe, mode)
    assert helped == errors == silent == 0
