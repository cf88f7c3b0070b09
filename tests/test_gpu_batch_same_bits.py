"""An FP32 instance keeps its bits whatever else the batch holds: alone its group
has a launch of its own, beside another group the batch's groups share one, and
which it is changes while it runs, as others are admitted and retired.  All
element types and laws, with strains that reach every branch of theirs.  So does
an FP32 model whose steps take one launch or two."""
import numpy as np
import pytest

from akantu2_amd import SolidMechanicsModel
from akantu2_amd import mesh as M

pytestmark = pytest.mark.gpu

TET, HEX = "_tetrahedron_4", "_hexahedron_8"
PLASTIC = "plastic_linear_isotropic_hardening"
LAWS = ("elastic", "elastic_fd", "neohookean", PLASTIC)
KINDS = [(t, law) for t in (TET, HEX) for law in LAWS]
FIELDS = ("displacement", "velocity", "acceleration", "internal_force")


def _mesh(etype, cells, seed=3):
    return M.box_mesh(etype, *cells, jitter=0.1, seed=seed)


def _batch(plastic=True):
    from akantu2_amd.batch import Batch

    return Batch("fp32", nodes=40000, tets=60000, hexes=8000, plastic=plastic)


def _add(b, etype, law, cells, amplitude, seed=4):
    m = _mesh(etype, cells)
    return b.add(m, law, E=1.1, nu=0.31, sigma_y=2e-3, h=0.05, blocked=M.clamped_face_x0(m),
                 velocity=M.initial_velocity(m, amplitude, seed))


def _get(b, i):
    return [b.get(i, f) for f in FIELDS]


def _same(got, want):
    for f, g, w in zip(FIELDS, got, want):
        assert np.isfinite(w).all() and np.abs(w).max() > 0
        assert np.array_equal(g, w), f


# amplitudes: small strains, and strains beyond the log1p series' 1/16
@pytest.mark.parametrize("amplitude", [1e-3, 2e-1])
def test_alone_and_beside_every_other_group(amplitude):
    cells = {TET: (9, 5, 4), HEX: (9, 6, 5)}
    b = _batch()
    ids = [_add(b, t, law, cells[t], amplitude) for t, law in KINDS]
    b.solveStep(21)
    b.solveStep(4)
    for i, (t, law) in zip(ids, KINDS):
        alone = _batch()
        k = _add(alone, t, law, cells[t], amplitude)
        alone.solveStep(25)
        _same(_get(b, i), _get(alone, k))


@pytest.mark.parametrize("kind", KINDS, ids=lambda k: k[0][1:4] + k[1][:10])
def test_others_come_and_go(kind):
    cells = {TET: (13, 5, 4), HEX: (17, 6, 5)}
    others = [k for k in KINDS if k != kind]
    b = _batch()
    i = _add(b, *kind, cells[kind[0]], 1e-2)
    b.solveStep(7)
    more = [_add(b, *k, (4, 3, 2), 1e-2, 7) for k in others[::3]]
    b.solveStep(10)
    for k in more:
        b.remove(k)
    b.solveStep(3)
    _add(b, *others[1], (3, 3, 3), 1e-2, 9)
    b.solveStep(5)
    alone = _batch()
    k = _add(alone, *kind, cells[kind[0]], 1e-2)
    alone.solveStep(25)
    _same(_get(b, i), _get(alone, k))


@pytest.mark.parametrize("etype,law", [k for k in KINDS if k[1] != PLASTIC])
def test_one_and_two_launches_a_step(etype, law):
    mesh = _mesh(etype, (13, 7, 6))
    out = []
    for timing in (False, True):  # kernel timing: two launches
        m = SolidMechanicsModel(mesh)
        m.addMaterial(law, E=1.1, nu=0.31)
        m.setPrecision("fp32")
        m.initFull()
        m.getBlockedDOFs()[:] = M.clamped_face_x0(mesh)
        m.getVelocity()[:] = M.initial_velocity(mesh, 5e-2, 4)
        m.setTimeStep(0.3 * m.getStableTimeStep())
        m.enableKernelTiming(timing)
        m.solveSteps(21)
        m.solveSteps(4)
        out.append([np.array(f()) for f in (m.getDisplacement, m.getVelocity, m.getAcceleration,
                                            m.getInternalForce)])
    _same(*out)
