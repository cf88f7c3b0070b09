"""Which models step in one launch, at the limits of each kind, and when a batch
replays a graph: what the tests of their results compare."""
import ctypes as C

import numpy as np
import pytest

from akantu2_amd import _native as N
from akantu2_amd import SolidMechanicsModel
from akantu2_amd import mesh as M
from akantu2_amd.batch import Batch

pytestmark = pytest.mark.gpu

TET, HEX = "_tetrahedron_4", "_hexahedron_8"
PLASTIC = "plastic_linear_isotropic_hardening"


def workgroups(m):
    n = C.c_int64(-1)
    N.check(N.lib().akx_model_get_step_workgroups(m._h, C.byref(n)))
    return n.value


def model(etype, cells, law, precision="fp64", elements=None, numbering="grid"):
    mesh = M.box_mesh(etype, *cells, jitter=0.1, seed=2)
    if numbering == "random":
        conn = np.random.default_rng(3).permutation(mesh.nb_nodes)[mesh.conn]
        nodes = np.empty_like(mesh.nodes)
        nodes[np.random.default_rng(3).permutation(mesh.nb_nodes)] = mesh.nodes
        mesh = M.BoxMesh(mesh.etype, nodes, np.ascontiguousarray(conn, np.int32), mesh.shape)
    m = SolidMechanicsModel(mesh)
    if elements is None:
        m.addMaterial(law, E=1.2, nu=0.28, sigma_y=2e-3, h=0.1)
    else:
        ids = np.arange(mesh.nb_elements)
        m.addMaterial(law, E=1.2, nu=0.28, elements=ids[:elements])
        m.addMaterial(law, E=1.4, nu=0.28, elements=ids[elements:])
    m.setPrecision(precision)
    m.initFull()
    m.setTimeStep(0.3 * m.getStableTimeStep())
    return m


# the largest mesh of each kind and one above
@pytest.mark.parametrize("etype,law,precision,last,above", [
    (TET, "elastic", "fp64", (39, 15, 15), (40, 15, 15)),
    (TET, "neohookean", "fp32", (39, 15, 15), (40, 15, 15)),
    (TET, PLASTIC, "fp64", (31, 15, 15), (32, 15, 15)),
    (HEX, "elastic", "fp64", (19, 15, 7), (20, 15, 7)),
    (HEX, "neohookean", "fp64", (15, 11, 7), (16, 11, 7)),
    (HEX, "elastic_fd", "fp32", (47, 15, 15), (48, 15, 15)),
])
def test_largest_one_launch_models(etype, law, precision, last, above):
    small, large = model(etype, last, law, precision), model(etype, above, law, precision)
    assert workgroups(small) > 0
    assert workgroups(large) == 0
    small.enableKernelTiming(True)
    assert workgroups(small) == 0
    small.enableKernelTiming(False)
    assert workgroups(small) > 0


def test_models_that_take_two_launches():
    assert workgroups(model(TET, (5, 4, 4), "elastic", "fp64_fast")) == 0
    assert workgroups(model(TET, (5, 4, 4), PLASTIC, "fp32")) == 0
    assert workgroups(model(HEX, (5, 4, 4), PLASTIC)) == 0
    assert workgroups(model(TET, (5, 4, 4), "elastic", elements=100)) == 0


@pytest.mark.parametrize("etype,precision", [(TET, "fp64"), (TET, "fp32"), (HEX, "fp64"),
                                             (HEX, "fp32")])
def test_random_numbering_has_a_plan(etype, precision):
    """Runs of nodes without locality: more elements around them, as many as the
    workgroup takes (the results are compared for such meshes too)."""
    assert workgroups(model(etype, (6, 5, 4), "elastic", precision, numbering="random")) > 0


def graph_steps(b):
    n = C.c_int(-1)
    N.check(N.lib().akx_batch_get_graph_steps(b._h, C.byref(n)))
    return n.value


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_batch_graphs(precision):
    mesh = M.box_mesh(TET, 5, 3, 2, jitter=0.1, seed=1)
    b = Batch(precision, nodes=2048, tets=32768)
    b.add(mesh, "elastic")
    b.solveStep(511)
    assert graph_steps(b) == 0
    b.solveStep(40)  # the lists have not lasted 512 steps when it starts
    assert graph_steps(b) == 0
    b.solveStep(16)  # a replay leaves no step for the call's end
    assert graph_steps(b) == 0
    b.solveStep(17)
    assert graph_steps(b) == 16
    b.add(mesh, "elastic")
    b.solveStep(20)
    assert graph_steps(b) == 0
    b.setLaunch(graph=False)
    for _ in range(40):
        b.solveStep(20)
    assert graph_steps(b) == 0
    b.setLaunch(graph=True)
    b.solveStep(520)
    b.solveStep(20)
    assert graph_steps(b) == 16
