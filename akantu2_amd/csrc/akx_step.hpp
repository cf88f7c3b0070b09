// akx_step.hpp -- one step of a small model in one launch: what the Tet4 and
// Hex8 kernels of the strict and the fast translation unit share.
//
// A mesh of up to a few thousand nodes leaves most of the chip idle, so a step
// costs its launches and the round trips of each kernel, not its work.  Here
// every workgroup owns a few nodes, computes all elements around
// them (each element in up to nnpe workgroups) and updates its nodes from
// forces that never leave its LDS: no force table, no second launch, and the
// predictor of a call's first step is applied to the nodes as they are read.
// Only u is read across workgroups, so only u alternates between two arrays
// (in a call's first step, whose predictor reads v and a too, these do as
// well).  Values and summation orders are those of the element pass and the
// gather.
#pragma once
#include "akx_args.hpp"
#include "akx_math.hpp"
#include <hip/hip_runtime.h>

namespace AKX_MATH_NS {

using akx::StepArgs;

// Predictor of one component
template <bool COMP>
__device__ __forceinline__ void step_predict(double dt, double a, double &v, float &cv,
                                             double &u, float &cu) {
  if constexpr (COMP)
    half_step_predict(a, dt, v, cv, u, cu);
  else
    reference_predict(a, dt, v, u);
}

// {X, u} records of the workgroup's node list.  The caller synchronises.
template <bool COMP>
__device__ __forceinline__ void step_stage(const StepArgs &S, int64_t b, double2 *s_rec) {
  for (int k = threadIdx.x; k < S.max_nodes; k += blockDim.x) {
    const int32_t n = S.lnode[b * S.max_nodes + k];
    if (n < 0)
      continue;
    double x[3], u[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      x[c] = S.X[c * S.nn + n];
      u[c] = S.u[c * S.nn + n];
    }
    if (S.first) {
      const uint8_t blk = S.blocked[n];
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const int64_t o = c * S.nn + n;
        double v = S.v[o], up = u[c];
        const double a = S.a[o];
        float cv = 0.f, cu = 0.f;
        if constexpr (COMP) {
          cv = S.cv[o];
          cu = S.cu[o];
        }
        step_predict<COMP>(S.dt, a, v, cv, up, cu);
        u[c] = (blk >> c) & 1 ? u[c] : up;
      }
    }
    s_rec[3 * k] = make_double2(x[0], x[1]);
    s_rec[3 * k + 1] = make_double2(x[2], u[0]);
    s_rec[3 * k + 2] = make_double2(u[1], u[2]);
  }
}

// One component of one owned node: lane t < 3 own takes component t / own of
// node t % own.  load() is called ahead of the staging, so that its round trip
// overlaps it; update() after the elements' forces are in their slots.
template <bool COMP> struct StepDof {
  int64_t o, n;
  double M, fx, u, v, a;
  float cu, cv;
  int c, s0, s1;
  bool on, held;

  __device__ __forceinline__ void load(const StepArgs &S, int64_t b) {
    const int t = threadIdx.x;
    c = t / S.own;
    const int k = t - c * S.own;
    n = c < 3 ? S.onode[b * S.own + k] : -1;
    on = n >= 0;
    if (!on)
      return;
    o = c * S.nn + n;
    s0 = k == 0 ? 0 : S.send[b * S.own + k - 1];
    s1 = S.send[b * S.own + k];
    M = S.mass[n];
    held = (S.blocked[n] >> c) & 1;
    u = S.u[o];
    v = S.v[o];
    // the FP32 form's a is the last step's only
    a = !COMP || S.first ? S.a[o] : 0.;
    fx = S.fext ? S.fext[o] : 0.;
    if constexpr (COMP) {
      cu = S.cu[o];
      cv = S.cv[o];
    }
  }

  template <bool PREDICT, class FT>
  __device__ __forceinline__ void finish(const StepArgs &S, double f) {
    if (!held) {
      if constexpr (COMP)
        half_step_gather<PREDICT>(fx + f, M, S.dt, v, cv, u, cu, a);
      else
        reference_gather<PREDICT>(fx, f, M, S.dt, a, v, u);
    }
  }

  // f = (0 + -1 e_0) + -1 e_1 ... over the node's slots, or over their partial
  // sums (s_run: the slot ends one) where the element pass leaves these, as
  // sums in FP64 rounded once to FT
  template <bool RUNS, class FT>
  __device__ __forceinline__ double sum(const FT *s_slot, const uint8_t *s_run) const {
    double f = 0., part = 0.;
    constexpr int CH = 8;
    for (int d = s0; d < s1; d += CH) {
      FT e[CH];
      bool end[CH];
#pragma unroll
      for (int j = 0; j < CH; ++j) {
        const int s = d + j < s1 ? d + j : s1 - 1;
        e[j] = s_slot[3 * s + c];
        if constexpr (RUNS)
          end[j] = s_run[s] != 0;
      }
#pragma unroll
      for (int j = 0; j < CH; ++j)
        if (d + j < s1) {
          if constexpr (RUNS) {
            part = part + double(e[j]);
            if (end[j]) {
              f = f + -1. * double(FT(part));
              part = 0.;
            }
          } else {
            f = f + -1. * double(e[j]);
          }
        }
    }
    return f;
  }

  template <bool RUNS, class FT>
  __device__ __forceinline__ void update(const StepArgs &S, const FT *s_slot,
                                         const uint8_t *s_run) {
    if (!on)
      return;
    const double f = sum<RUNS>(s_slot, s_run);
    if (S.first && !held)
      step_predict<COMP>(S.dt, a, v, cv, u, cu);
    if (S.last)
      finish<false, FT>(S, f);
    else
      finish<true, FT>(S, f);
    if (S.fint)
      S.fint[o] = f;
    if (S.u2)
      S.u2[o] = u;
    S.v2[o] = v;
    if constexpr (COMP) {
      S.cu2[o] = cu;
      S.cv2[o] = cv;
      // between the steps of a call a is neither read nor written: the first
      // step carries a held component's over, the last writes the others'
      if (S.first || (S.last && !held))
        S.a2[o] = a;
    } else {
      S.a2[o] = a;
    }
  }
};

} // namespace AKX_MATH_NS
