"""The memory that models keep of dropped field copies is bounded over the process
and given back with the model."""
import threading

import numpy as np
import pytest

from akantu2_amd.model import _Spare


@pytest.fixture
def limit(monkeypatch):
    before = _Spare._bytes
    monkeypatch.setattr(_Spare, "LIMIT", before + 1000)
    yield before
    assert _Spare._bytes == before


def test_bounded_over_models_and_given_back(limit):
    a, b = _Spare(), _Spare()
    u, s = np.zeros(50), np.zeros(50)  # 400 bytes each
    a.put("u", u, s)
    assert _Spare._bytes == limit + 800
    b.put("u", np.zeros(50), None)  # over the limit: not kept
    assert b.take("u") == (None, None)
    b.put("v", np.zeros(25), None)
    assert _Spare._bytes == limit + 1000
    assert a.take("u") == (u, s) and a.take("u") == (None, None)
    b.put("v", np.zeros(10), np.zeros(10))  # in the place of the one before
    assert _Spare._bytes == limit + 160
    del b
    assert _Spare._bytes == limit


def test_threads(limit):
    def work():
        s = _Spare()
        for k in range(500):
            s.put(k % 3, np.zeros(4), None)
            s.take(k % 2)

    threads = [threading.Thread(target=work) for _ in range(8)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
