// akx_fast.hpp -- entry points of the fast element pass (akx_fast.hip).
#pragma once
#include "akx_args.hpp"
#include "akx_batch.hpp"
#include <hip/hip_runtime.h>

namespace akxf {
// copy dN_n/dxi_m at the 8 Hex8 Gauss points ([q][m][n]) to the device
hipError_t upload_hex8_dnds(const double *dnds);
// elements per workgroup of the FP32 / FP64-fast element passes (bpa: the
// FP32 block-partial passes)
int64_t elements_per_block(int etype, bool bpa = false);
// launch the element pass of one material (etype 0 = Tet4, 1 = Hex8)
hipError_t launch_elements(int etype, int law, bool fp32, const akx::ElemArgs &A,
                           hipStream_t stream);
// launch one step of a small FP32 model (akx_step.hpp)
hipError_t launch_step(int etype, int law, const akx::StepArgs &S, size_t lds, hipStream_t stream);
// launch the FP32-form batched element pass (block-partial assembly) of one
// (element type, law) group, or of all groups: the Tet4 and the Hex8 tiles
hipError_t launch_batch_elements_f32(int etype, int law, const akx::BatchElemArgs &A,
                                     hipStream_t stream);
hipError_t launch_batch_all_f32(const akx::BatchElemArgs &tets, const akx::BatchElemArgs &hexes,
                                hipStream_t stream);
} // namespace akxf
