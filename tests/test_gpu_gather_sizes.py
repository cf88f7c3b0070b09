"""The gather at the node count where it changes its load order (131,072 nodes:
the nodal state first and the table entries eight at a time up to there, one
entry after another above) and at half of it: the FP64 path equals the oracle
bit for bit on both sides, with nodes of 1 to 24 elements, blocked nodes, an
external force and a partly filled last slice; and where a step's bytes no
longer fit the cache (310 MB) and the table is read with non-temporal loads."""
import numpy as np
import pytest

import oracle
from akantu2_amd import SolidMechanicsModel
from akantu2_amd import mesh as M

pytestmark = pytest.mark.gpu

# 65,536 and 66,560 nodes; the third Hex8 box (65,533 nodes) has a last slice of
# 253; 131,072 and 133,120 nodes; more than 310 MB a step
CELLS = {"_tetrahedron_4": [(63, 31, 31), (64, 31, 31), (63, 31, 63), (64, 31, 63), (79, 66, 66)],
         "_hexahedron_8": [(63, 31, 31), (64, 31, 31), (12, 70, 70), (63, 31, 63), (64, 31, 63),
                           (79, 62, 62)]}


@pytest.mark.parametrize("etype,cells", [(t, c) for t in CELLS for c in CELLS[t]])
def test_gather_matches_oracle_around_the_switch(etype, cells):
    mesh = M.box_mesh(etype, *cells, jitter=0.1, seed=2)
    blocked = M.clamped_face_x0(mesh)
    v0 = M.initial_velocity(mesh, 1e-3, 3)
    fext = 1e-4 * np.random.default_rng(5).standard_normal((mesh.nb_nodes, 3))
    g = SolidMechanicsModel(mesh)
    g.addMaterial("elastic", E=1.2, nu=0.28)
    g.initFull()
    g.getBlockedDOFs()[:] = blocked
    g.getVelocity()[:] = v0
    g.getExternalForce()[:] = fext
    dt = 0.5 * g.getStableTimeStep()
    g.setTimeStep(dt)
    o = oracle.OracleModel(mesh.etype, mesh.nodes, mesh.conn, "elastic", E=1.2, nu=0.28)
    o.init_full()
    o.blocked[:] = blocked
    o.v[:] = v0
    o.f_ext[:] = fext
    o.set_time_step(dt)
    o.solve_steps(3)
    g.solveSteps(3)
    for got, want in ((g.getDisplacement(), o.u), (g.getVelocity(), o.v),
                      (g.getAcceleration(), o.a), (g.getInternalForce(), o.f_int)):
        assert np.array_equal(got, want)
