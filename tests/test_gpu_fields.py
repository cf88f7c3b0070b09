"""Downloads of nodal fields: one wait for several fields, chunks of 1 MB
(43,690 rows of three doubles) taken by several threads above that.  Sizes on
both sides of a chunk, ragged last chunks, second destinations, the one-byte
field, fields of a batch, and the arrays a model hands out again."""
import ctypes as C

import numpy as np
import pytest

from akantu2_amd import SolidMechanicsModel
from akantu2_amd import _native as N
from akantu2_amd import mesh as M

pytestmark = pytest.mark.gpu

# a chunk is 43,690 rows.  Nodes: 8, 43,690 (one chunk), 43,692 (two rows more),
# 87,380 (two chunks), 262,144 (six chunks and four rows)
CELLS = [(1, 1, 1), (4368, 4, 1), (10922, 1, 1), (8737, 4, 1), (63, 63, 63)]


@pytest.mark.parametrize("cells", CELLS)
def test_fields_come_back_as_set(cells):
    mesh = M.box_mesh("_hexahedron_8", *cells)
    g = SolidMechanicsModel(mesh)
    g.addMaterial("elastic")
    g.initFull()
    nn = mesh.nb_nodes
    rng = np.random.default_rng(1)
    u, v = rng.standard_normal((2, nn, 3))
    blocked = (rng.random((nn, 3)) < 0.3).astype(np.uint8)
    g.getDisplacement()[:] = u
    g.getVelocity()[:] = v
    g.getBlockedDOFs()[:] = blocked
    g.synchronize()
    g._push()
    ids = [N.FIELD_DISPLACEMENT, N.FIELD_BLOCKED_DOFS, N.FIELD_VELOCITY, N.FIELD_MASS,
           N.FIELD_EXTERNAL_FORCE, N.FIELD_NODES]
    host = [np.full((nn, 3), 9, np.uint8 if i == N.FIELD_BLOCKED_DOFS else float) for i in ids]
    copy = [np.full_like(h, 8) if k % 2 == 0 else None for k, h in enumerate(host)]
    ptrs = (C.c_void_p * len(ids))(*[h.ctypes.data for h in host])
    dups = (C.c_void_p * len(ids))(*[None if c is None else c.ctypes.data for c in copy])
    N.check(N.lib().akx_model_get_fields(g._h, len(ids), (C.c_int * len(ids))(*ids), ptrs, dups))
    mass = np.repeat(np.asarray(g.getMass())[:, :1], 3, axis=1)
    for k, want in enumerate((u, blocked, v, mass, np.zeros((nn, 3)), mesh.nodes)):
        assert np.array_equal(host[k], want), ids[k]
        if copy[k] is not None:
            assert np.array_equal(copy[k], want), ids[k]
    # arrays handed out again after their copy was dropped: the current values,
    # and edits through them are still seen
    for step in range(3):
        w = g.getDisplacement()
        assert np.array_equal(w, u)
        w[-1, 2] = u[-1, 2] = float(step)
        del w
        g._push()
        assert not g._mirrors
    kept = g.getVelocity()
    assert np.array_equal(kept, v)
    again = g.getVelocity()
    assert again is kept


def test_batch_fields():
    from akantu2_amd.batch import Batch
    meshes = [M.box_mesh("_hexahedron_8", *c, jitter=0.1, seed=3) for c in CELLS[:4]]
    b = Batch("fp64", nodes=sum(m.nb_nodes + 255 for m in meshes),
              hexes=sum(m.nb_elements for m in meshes))
    vel = [np.random.default_rng(k).standard_normal((m.nb_nodes, 3))
           for k, m in enumerate(meshes)]
    ids = [b.add(m, "elastic", velocity=v) for m, v in zip(meshes, vel)]
    for i, m, v in zip(ids, meshes, vel):
        assert np.array_equal(b.get(i, "velocity"), v)
        assert np.array_equal(b.get(i, "nodes"), m.nodes)
