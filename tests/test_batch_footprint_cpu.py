"""akx_batch_footprint against the arenas' bytes per node and element: what the
server's memory budget is divided by."""
import pytest

from akantu2_amd.batch import footprint

TET, HEX = 0, 1
PLASTIC = "plastic_linear_isotropic_hardening"


def _bytes(precision, etype, law, nn, nel):
    f32 = precision == "fp32"
    nnpe, nqp, block, entries = ((4, 1, 256, 2), (8, 8, 63, 8))[etype]
    slices = -(-nn // 256)
    real = 4 if f32 else 8
    # node records, v, a, f_int, mass, blocked bits, degree; FP32: X and u apart,
    # compensation terms
    node = 48 + 3 * 24 + 8 + 2 + (2 * 24 + 2 * 12 if f32 else 0)
    # connectivity, 1.25 force-table entries of three values per corner
    elem = nnpe * (4 + 1.25 * 3 * real)
    if f32:  # local corners and slots; per block entry node, place and slot end
        elem += nnpe * 4 + entries * 10
    else:  # places in the table
        elem += nnpe * 4
    if law == PLASTIC:
        elem += nqp * 2 * (7 if f32 else 28) * real
    blocks = -(-nel // block) if f32 else 0
    # slices: row start; admission: widths / counts (4), offsets (8), block ranges (16)
    return slices * (256 * node + 8 + 12) + nel * elem + blocks * 28


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("etype", [TET, HEX])
@pytest.mark.parametrize("law", ["elastic", PLASTIC])
def test_footprint_is_what_the_arenas_hold(precision, etype, law):
    for nn, nel in ((1000, 5000), (300000, 1000000)):
        want = _bytes(precision, etype, law, nn, nel)
        assert abs(footprint(precision, etype, law, nn, nel) - want) <= 1
