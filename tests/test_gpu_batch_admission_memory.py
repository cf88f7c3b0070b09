"""Device memory of a batch and its instances: an admission allocates none (what
it needs beside the arenas is held from the batch's creation), an instance that
fills a batch takes what akx_batch_footprint says, and a refused one gives back
every range."""
import pytest
import torch

from akantu2_amd import _native as N
from akantu2_amd import mesh as M
from akantu2_amd.batch import Batch, footprint

pytestmark = pytest.mark.gpu

TET, HEX = "_tetrahedron_4", "_hexahedron_8"
PLASTIC = "plastic_linear_isotropic_hardening"
MB = 1 << 20


def _used():
    torch.cuda.synchronize()
    free, total = torch.cuda.mem_get_info()
    return total - free


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("etype,cells,law", [(HEX, (110, 100, 100), "neohookean"),
                                             (TET, (64, 50, 50), PLASTIC)])
def test_admission_allocates_nothing(etype, cells, law, precision):
    m = M.box_mesh(etype, *cells, jitter=0.1, seed=1)
    small = M.box_mesh(etype, 2, 2, 2)
    nel = m.nb_elements + small.nb_elements
    tets, hexes = (nel + 4096, 0) if etype == TET else (0, nel + 4096)
    warm = Batch(precision, nodes=512, tets=4096, hexes=512, plastic=True)
    warm.add(small, law, sigma_y=1e-2, h=0.1)  # the runtime and the kernels' code
    warm.close()
    first = _used()
    b = Batch(precision, nodes=m.nb_nodes + 512, tets=tets, hexes=hexes, plastic=law == PLASTIC)
    b.add(small, law, sigma_y=1e-2, h=0.1)
    b.synchronize()
    before = _used()
    b.add(m, law, sigma_y=1e-2, h=0.1, blocked=M.clamped_face_x0(m),
          velocity=M.initial_velocity(m, 1e-3, 2))
    after = _used()
    want = footprint(precision, m.etype, law, m.nb_nodes, m.nb_elements)
    print(f"{precision} {etype} {m.nb_elements}: add {(after - before) / MB:.1f} MB, batch "
          f"{(after - first) / MB:.1f} MB, footprint {want / MB:.1f} MB", flush=True)
    assert after - before <= 4 * MB
    # the 4,096 elements more, the small instance, a fixed part (a round of nodes'
    # input 6.4 MB, tables) and the allocator's granularity
    assert after - first <= 1.01 * want + 32 * MB


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_refused_instance_gives_its_ranges_back(precision):
    m = M.box_mesh(TET, 12, 10, 9, jitter=0.1, seed=1)
    filler = M.box_mesh(HEX, 5, 5, 5, jitter=0.1, seed=1)
    for nodes, tets, hexes, what in ((m.nb_nodes - 256, 10 * m.nb_elements, 0, "node"),
                                     (4 * m.nb_nodes, m.nb_elements - 1, 0, "element"),
                                     (4 * m.nb_nodes, m.nb_elements, 0, None)):
        b = Batch(precision, nodes=nodes, tets=tets, hexes=filler.nb_elements)
        left = b.capacityLeft()
        try:
            b.remove(b.add(m, "elastic"))
        except N.AkantuError as e:
            assert e.code == -4
            assert what is None or what + " arena full" in str(e)
        else:
            assert what is None
        assert b.capacityLeft() == left
        b.add(filler, "elastic")
        b.solveStep(2)


def test_too_many_elements_around_a_node_is_refused_and_gives_back():
    import numpy as np

    n = 300  # tetrahedra around one edge
    t = np.linspace(0, 2 * np.pi, n, endpoint=False)
    ring = np.stack([np.cos(t), np.sin(t), 0.5 + 0 * t], 1)
    nodes = np.concatenate([[[0, 0, 0], [0, 0, 1]], ring])
    k = np.arange(n)
    conn = np.stack([0 * k, 2 + k, 1 + 0 * k, 2 + (k + 1) % n], 1).astype(np.int32)
    if np.linalg.det(nodes[conn[0]][1:] - nodes[conn[0]][0]) < 0:
        conn = conn[:, [0, 2, 1, 3]]
    fan = M.BoxMesh(0, nodes, np.ascontiguousarray(conn, np.int32), (n, 1, 1))
    b = Batch("fp64", nodes=4096, tets=1 << 16)
    left = b.capacityLeft()
    with pytest.raises(N.AkantuError, match="more than 255"):
        b.add(fan, "elastic")
    assert b.capacityLeft() == left
    b.add(M.box_mesh(TET, 3, 3, 3), "elastic")
    b.solveStep(2)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_more_nodes_than_one_round(precision):
    """140,608 nodes: their input goes up in two rounds of up to 131,072."""
    import numpy as np

    import oracle

    mesh = M.box_mesh(HEX, 51, 51, 51, jitter=0.1, seed=2)
    rng = np.random.default_rng(4)
    blocked = rng.random((mesh.nb_nodes, 3)) < 0.1
    v0 = 0.05 * rng.standard_normal((mesh.nb_nodes, 3))
    b = Batch(precision, nodes=mesh.nb_nodes + 512, hexes=mesh.nb_elements + 4096)
    i = b.add(mesh, "elastic", E=1.2, nu=0.28, blocked=blocked, velocity=v0)
    b.solveStep(2)
    o = oracle.OracleModel(mesh.etype, mesh.nodes, mesh.conn, "elastic", E=1.2, nu=0.28)
    o.init_full()
    o.blocked[:] = blocked
    o.v[:] = v0
    o.set_time_step(b.timeStep(i)[0])
    o.solve_steps(2)
    for f, w in (("nodes", mesh.nodes), ("displacement", o.u), ("velocity", o.v),
                 ("internal_force", o.f_int)):
        g = b.get(i, f)
        if precision == "fp64" or f == "nodes":
            assert np.array_equal(g, w), f
        else:
            assert np.abs(g - w).max() <= 1e-5 * np.abs(w).max(), f
