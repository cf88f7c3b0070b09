"""The groups of an FP32 batch run in one launch when there are several, up to
20,480 tiles (256 Tet4 or 63 Hex8 each).  Every instance gives what it gives
alone (its group's own launch), up to float rounding of its element forces
(the compiler contracts each kernel's products on its own: 1e-5 of the largest
force, 1e-6 of the displacements after these steps)."""
import numpy as np
import pytest

from akantu2_amd import mesh as M

pytestmark = pytest.mark.gpu

TET, HEX = "_tetrahedron_4", "_hexahedron_8"
PLASTIC = "plastic_linear_isotropic_hardening"
SMALL = [(TET, (7, 3, 2), "elastic"), (HEX, (5, 3, 3), "neohookean"),
         (TET, (43, 1, 1), "elastic_fd"), (HEX, (9, 7, 1), PLASTIC), (TET, (1, 1, 1), PLASTIC),
         (HEX, (64, 1, 1), "elastic"), (TET, (9, 5, 4), "neohookean"), (HEX, (1, 1, 1), "elastic_fd")]


def run(insts):
    from akantu2_amd.batch import Batch

    meshes = [M.box_mesh(t, *c, jitter=0.1, seed=3) for t, c, _ in insts]
    tets = sum(m.nb_elements for m, i in zip(meshes, insts) if i[0] == TET)
    hexes = sum(m.nb_elements for m, i in zip(meshes, insts) if i[0] == HEX)
    b = Batch("fp32", nodes=sum(m.nb_nodes + 256 for m in meshes), tets=2 * tets + 20000,
              hexes=hexes, plastic=any(i[2] == PLASTIC for i in insts))
    ids = [b.add(m, law, E=1.0, nu=0.3, sigma_y=2e-3, h=0.05, blocked=M.clamped_face_x0(m),
                 velocity=M.initial_velocity(m, 1e-2, 4)) for m, (_, _, law) in zip(meshes, insts)]
    b.solveStep(5)
    b.solveStep(2)
    return [[b.get(i, f) for f in ("displacement", "internal_force")] for i in ids]


def check(got, want):
    for g, w, bound in zip(got, want, (1e-6, 1e-5)):
        assert np.isfinite(g).all()
        assert np.abs(g - w).max() <= bound * np.abs(w).max()


@pytest.mark.parametrize("members", [range(8), (0, 2), (1, 5), (0, 1), (3, 4), (6, 7)],
                         ids=lambda m: "".join(map(str, m)))
def test_merged_groups_equal_groups_alone(members):
    insts = [SMALL[k] for k in members]
    for inst, got in zip(insts, run(insts)):
        check(got, run([inst])[0])


def test_more_tiles_than_one_launch_takes():
    many = (HEX, (127, 102, 100), "elastic")  # 20,563 tiles of 63
    got = run([many, SMALL[0]])
    check(got[1], run([SMALL[0]])[0])
    assert all(np.isfinite(f).all() for f in got[0])
