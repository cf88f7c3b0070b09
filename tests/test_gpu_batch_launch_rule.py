"""The library's own launch shape of an FP64 batch (small Hex8 tiles, one wave per
workgroup) stays in force when only graphs are switched, when the shape read from
an untouched batch is set again, and after the autotuner unless it finds a faster
one; a tile of 2,048 elements per workgroup takes over ten times as long here."""
import numpy as np
import pytest

from akantu2_amd import mesh as M

pytestmark = pytest.mark.gpu


def _batch():
    from akantu2_amd.batch import Batch

    m = M.box_mesh("_hexahedron_8", 30, 30, 30, jitter=0.1, seed=3)
    b = Batch("fp64", nodes=m.nb_nodes + 255, hexes=m.nb_elements + 64)
    i = b.add(m, "neohookean", blocked=M.clamped_face_x0(m),
              velocity=M.initial_velocity(m, 1e-3, 5))
    return b, i


def _pass_ms(b):
    """Fastest of some element passes."""
    best = 1e9
    for _ in range(4):
        b.enableKernelTiming(True)
        b.solveStep(5)
        ms, n = b.kernelTiming(0)
        best = min(best, ms / n)
        b.enableKernelTiming(False)
    return best


@pytest.mark.parametrize("change", ["graph off", "read back", "autotuned"])
def test_the_rule_stays(change):
    ref, i = _batch()
    want = _pass_ms(ref)
    b, k = _batch()
    if change == "graph off":
        b.setLaunch(graph=False)
        assert not b.launch()["graph"]
    elif change == "read back":
        s = b.launch()
        b.setLaunch(**s)
        assert b.launch() == s
    else:
        best = b.autotune(repeats=3)
        assert best["element_pass_ms"] <= 1.5 * want
    got = _pass_ms(b)
    print(change, "element pass", want, "->", got, flush=True)
    assert got <= 2 * want
    assert np.array_equal(ref.get(i, "displacement"), b.get(k, "displacement"))
