"""An instance's tables are made on the device when it joins a batch: block
lists by a sort, table rows by arrival and rank.  FP64: every corner has its
place in element order, so the results equal the oracle's bit for bit.  FP32:
block partials; the forces stay within float rounding of the oracle's (a sum of
some 24 terms of 6e-8 each: 1e-5 of the largest force), and the tables do not
depend on what the arenas held before or on the arrival order: an instance added
again after another left has the same bits."""
import dataclasses

import numpy as np
import pytest

import oracle
from akantu2_amd import mesh as M

pytestmark = pytest.mark.gpu

TET, HEX = "_tetrahedron_4", "_hexahedron_8"
# one element's worth; around one and two blocks (256 Tet4, 63 Hex8) and one
# slice (256 nodes); many blocks around a node (random numbering)
CELLS = [(TET, (1, 1, 1)), (TET, (42, 1, 1)), (TET, (43, 1, 1)), (TET, (63, 1, 1)),
         (TET, (64, 1, 1)), (TET, (13, 9, 8)), (HEX, (1, 1, 1)), (HEX, (62, 1, 1)),
         (HEX, (63, 1, 1)), (HEX, (64, 1, 1)), (HEX, (11, 9, 8))]


def shuffled(mesh, seed):
    rng = np.random.default_rng(seed)
    to = rng.permutation(mesh.nb_nodes)
    nodes = np.empty_like(mesh.nodes)
    nodes[to] = mesh.nodes
    conn = to[mesh.conn][rng.permutation(mesh.nb_elements)]
    return dataclasses.replace(mesh, nodes=nodes, conn=np.ascontiguousarray(conn, np.int32))


@pytest.mark.parametrize("order", ["grid", "random"])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("etype,cells", CELLS)
def test_admitted_instance(etype, cells, precision, order):
    from akantu2_amd.batch import Batch

    mesh = M.box_mesh(etype, *cells, jitter=0.1, seed=2)
    if order == "random":
        mesh = shuffled(mesh, 3)
    rng = np.random.default_rng(4)
    blocked = rng.random((mesh.nb_nodes, 3)) < 0.1
    v0 = 0.05 * rng.standard_normal((mesh.nb_nodes, 3))
    other = M.box_mesh(TET, 5, 4, 3, jitter=0.1, seed=5)
    pad = 64 * 256  # slices as wide as their largest row
    hexes = mesh.nb_elements if etype == HEX else 0
    tets = other.nb_elements + pad + (mesh.nb_elements if etype == TET else 0)
    b = Batch(precision, nodes=mesh.nb_nodes + other.nb_nodes + 512, tets=tets, hexes=hexes)

    def run():
        i = b.add(mesh, "elastic", E=1.2, nu=0.28, blocked=blocked, velocity=v0)
        b.solveStep(3)
        return i, [b.get(i, f) for f in ("displacement", "velocity", "internal_force")]

    gone = b.add(other, "elastic", E=2.0)
    b.solveStep(2)
    b.remove(gone)
    i, got = run()
    o = oracle.OracleModel(mesh.etype, mesh.nodes, mesh.conn, "elastic", E=1.2, nu=0.28)
    o.init_full()
    o.blocked[:] = blocked
    o.v[:] = v0
    o.set_time_step(b.timeStep(i)[0])
    o.solve_steps(3)
    for g, w in zip(got, (o.u, o.v, o.f_int)):
        if precision == "fp64":
            assert np.array_equal(g, w)
        else:
            assert np.abs(g - w).max() <= 1e-5 * np.abs(w).max()
    b.remove(i)
    b.add(other, "elastic", E=2.0)
    for g, w in zip(run()[1], got):
        assert np.array_equal(g, w)
