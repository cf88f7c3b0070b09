"""FP32 Hex8 block passes at the edges of their 63-element blocks: one element,
one block, one more, ragged last blocks, every law; the single model and a
batch of the same instances against the FP64 oracle.  Bounds are the FP32
form's: 1e-5 of the largest displacement, and 1e-4 for the forces."""
import numpy as np
import pytest

import oracle
from akantu2_amd import SolidMechanicsModel
from akantu2_amd import mesh as M

pytestmark = pytest.mark.gpu

PL = "plastic_linear_isotropic_hardening"
CELLS = [(1, 1, 1), (62, 1, 1), (63, 1, 1), (64, 1, 1), (7, 3, 6), (127, 1, 1), (5, 5, 11)]
LAWS = ["elastic", "elastic_fd", "neohookean", PL]
STEPS = 25


def _velocity(m):
    """U(-1e-2, 1e-2) on the free nodes (the sine envelope of the other tests
    vanishes on every node of a mesh one cell long)."""
    v = np.random.default_rng(7).uniform(-1e-2, 1e-2, (m.nb_nodes, 3))
    return v * (1 - M.clamped_face_x0(m))


@pytest.mark.parametrize("law", LAWS)
def test_block_edges(law):
    from akantu2_amd.batch import Batch
    mat = dict(rho=1.0, E=1.3, nu=0.27)
    if law == PL:
        mat.update(sigma_y=2e-3, h=0.05)
    meshes = [M.box_mesh("_hexahedron_8", *c, jitter=0.1, seed=6) for c in CELLS]
    b = Batch("fp32", nodes=sum(m.nb_nodes + 255 for m in meshes),
              hexes=sum(m.nb_elements for m in meshes), plastic=law == PL)
    ids = [b.add(m, law, blocked=M.clamped_face_x0(m),
                 velocity=_velocity(m), **mat) for m in meshes]
    b.solveStep(STEPS)
    for m, iid in zip(meshes, ids):
        o = oracle.OracleModel(oracle.HEX8, m.nodes, m.conn, law, **mat)
        o.init_full()
        o.blocked[:] = M.clamped_face_x0(m)
        o.v[:] = _velocity(m)
        o.set_time_step(b.timeStep(iid)[0])
        o.solve_steps(STEPS)
        g = SolidMechanicsModel(m)
        g.addMaterial(law, **mat)
        g.setPrecision("fp32")
        g.initFull()
        g.getBlockedDOFs()[:] = M.clamped_face_x0(m)
        g.getVelocity()[:] = _velocity(m)
        g.setTimeStep(b.timeStep(iid)[0])
        g.solveSteps(STEPS)
        for u, f in ((g.getDisplacement(), g.getInternalForce()),
                     (b.getDisplacement(iid), b.getInternalForce(iid))):
            assert np.abs(u - o.u).max() <= 1e-5 * np.abs(o.u).max(), m.shape
            assert np.abs(f - o.f_int).max() <= 1e-4 * np.abs(o.f_int).max(), m.shape
