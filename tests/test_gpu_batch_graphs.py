"""Steps of a batch whose lists have lasted 512 steps are replayed from a graph
of 16: the same bits as launches one by one, at step counts around one and two
replays, with odd counts (history parity) and reads of the fields in between,
and after the lists change."""
import numpy as np
import pytest

from akantu2_amd import mesh as M

pytestmark = pytest.mark.gpu

PLASTIC = "plastic_linear_isotropic_hardening"


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_replayed_steps_equal_launched_ones(precision):
    from akantu2_amd.batch import Batch

    meshes = [M.box_mesh("_tetrahedron_4", 5, 3, 2, jitter=0.1, seed=1),
              M.box_mesh("_hexahedron_8", 4, 3, 3, jitter=0.1, seed=2)]

    def run(graph):
        b = Batch(precision, nodes=2048, tets=32768, hexes=1024, plastic=True)
        b.setLaunch(graph=graph)
        out = []

        def add(m, law, seed):
            return b.add(m, law, E=1.0, nu=0.3, sigma_y=2e-3, h=0.05,
                         blocked=M.clamped_face_x0(m), velocity=M.initial_velocity(m, 1e-2, seed))

        ids = [add(meshes[0], PLASTIC, 3), add(meshes[1], "neohookean", 4)]
        for steps in (511, 40, 17, 16, 33, 18, 1, 50):
            b.solveStep(steps)
            out += [b.get(i, f) for i in ids for f in ("displacement", "internal_force")]
        ids.append(add(meshes[0], "elastic", 5))
        for steps in (20, 500, 35):
            b.solveStep(steps)
            out += [b.get(i, f) for i in ids for f in ("displacement", "internal_force")]
        return out

    for got, want in zip(run(True), run(False)):
        assert np.isfinite(got).all()
        assert np.array_equal(got, want)
