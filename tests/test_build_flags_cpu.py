"""Floating-point contraction is fixed by the sources: no translation unit is
built with -ffp-contract=fast, which lets the optimiser choose, kernel by kernel,
which products are fused into which sums.  The same element functions, compiled
into the launch of one group of a batch and into the launch of all, could then
round differently, and an FP32 instance's bits would depend on the others in
the batch."""
from akantu2_amd import build


def test_contraction_does_not_depend_on_the_kernel():
    assert set(build.SOURCES) == {"akx_model.hip", "akx_fast.hip", "akx_batch.hip"}
    assert set(build.SOURCES.values()) <= {"off", "on"}
    assert not any("fast" in f for f in build.FLAGS)
