// akx_fast.hip -- regrouped element pass of the FP32 precision form and of
// the opt-in FP64 "fast" form.  Compiled with -ffp-contract=on, in its own
// translation unit and math namespace: a product is fused into the sum that is
// written in the same expression, so every kernel that an element function is
// part of gives the same bits (the launches of a batch's groups and the one of
// all, one-launch and two-launch steps).
//
// Same mechanics as the reference (material.cc:98-154 + 457-584): gather u,
// grad u at every Gauss point, constitutive law, B^T sigma (small strain) or
// (B_L + B_NL)^T S = (F S) dN/dX (total Lagrangian), times w detJ, summed per
// element.  The arithmetic is regrouped for gfx950:
//   J_q = dN/dxi_q X,  H_q = U dN/dxi_q^T              (natural gradients)
//   grad u_q = H_q J_q^{-1 T}
//   Q_q = w_q detJ_q P_q J_q^{-1}      (P = sigma, or F S for finite strain)
//   r_e(n) = sum_q Q_q dN_n/dxi_q
// which needs no dN/dX array and exchanges 9 numbers per Gauss point instead
// of 24.  In FP64 the results agree with the reference operation order to
// rounding per evaluation; the FP32 form uses a cancellation-free neo-Hookean
// stress.
//
// Hex8: FP32 block passes four lanes per element, two nodes and two Gauss
// points each; otherwise 8 lanes per element (one per Gauss point; in the last
// phase one per node), 32 elements per 256-thread block, nodal data and Q in LDS.
// Tet4: one thread per element (single Gauss point).
// The same element code serves the batched FP32 form (one tile of one instance
// per workgroup, per-instance parameters).
#define AKX_MATH_NS akxf
#include "akx_args.hpp"
#include "akx_math.hpp"
#include "akx_fast.hpp"
#include "akx_step.hpp"

#include <hip/hip_runtime.h>

#include <algorithm>

namespace akxf {

using akx::BatchElemArgs;
using akx::BInst;
using akx::NodesSoA;
using akx::NodesXU;
using akx::BBlk;
using akx::BTile;
using akx::ElemArgs;
using akx::QpCompact;
using akx::QpViewT;
using akx::batch_compact_view;
using akx::FE_W;
using akx::qp_view;
using akx::slot_pos;

constexpr int LAW_ELASTIC = 0, LAW_ELASTIC_FD = 1, LAW_NEOHOOKEAN = 2,
              LAW_PLASTIC = 3;

// dN_n/dxi_m at the 8 Hex8 Gauss points, [q][m][n]
__constant__ double c_dnds[8][3][8];

__device__ __forceinline__ int64_t xcd_block(int64_t nblocks_padded) {
  int64_t b = blockIdx.x;
  int64_t per = nblocks_padded >> 3;
  return (b & 7) * per + (b >> 3);
}

// inverse and determinant by cofactors
template <class R>
__device__ __forceinline__ R inv_det(const R (&m)[3][3], R (&r)[3][3]) {
  R c00 = m[1][1] * m[2][2] - m[1][2] * m[2][1];
  R c10 = m[2][1] * m[0][2] - m[2][2] * m[0][1];
  R c20 = m[0][1] * m[1][2] - m[0][2] * m[1][1];
  R det = c00 * m[0][0] + c10 * m[1][0] + c20 * m[2][0];
  R id = akx_rcp(det);
  r[0][0] = c00 * id;
  r[0][1] = c10 * id;
  r[0][2] = c20 * id;
  r[1][0] = (m[1][2] * m[2][0] - m[1][0] * m[2][2]) * id;
  r[1][1] = (m[2][2] * m[0][0] - m[2][0] * m[0][2]) * id;
  r[1][2] = (m[0][2] * m[1][0] - m[0][0] * m[1][2]) * id;
  r[2][0] = (m[1][0] * m[2][1] - m[1][1] * m[2][0]) * id;
  r[2][1] = (m[2][0] * m[0][1] - m[2][1] * m[0][0]) * id;
  r[2][2] = (m[0][0] * m[1][1] - m[0][1] * m[1][0]) * id;
  return det;
}

// Linear isotropic hardening with the full incremental history of the
// reference (grad u, stress, plastic strain, hardening).
template <class CT, class HT>
__device__ __forceinline__ void plastic_at(const QpViewT<HT> &V, int64_t iq, CT lambda,
                                           CT mu, CT sy, CT hh, const CT (&g)[3][3],
                                           CT (&S)[3][3]) {
  CT pg[3][3], ps[3][3], pe[3][3], eps[3][3], iso;
#pragma unroll
  for (int jj = 0; jj < 3; ++jj)
#pragma unroll
    for (int ii = 0; ii < 3; ++ii) {
      const int64_t o = (int64_t)(ii + 3 * jj) * V.nq_all + iq;
      pg[ii][jj] = CT(V.p_grad[o]);
      ps[ii][jj] = CT(V.p_sig[o]);
      pe[ii][jj] = CT(V.p_eps[o]);
    }
  plastic_lih(lambda, mu, sy, hh, g, pg, ps, CT(V.p_iso[iq]), pe, S, iso, eps);
#pragma unroll
  for (int jj = 0; jj < 3; ++jj)
#pragma unroll
    for (int ii = 0; ii < 3; ++ii) {
      const int64_t o = (int64_t)(ii + 3 * jj) * V.nq_all + iq;
      V.c_grad[o] = HT(g[ii][jj]);
      V.c_sig[o] = HT(S[ii][jj]);
      V.c_eps[o] = HT(eps[ii][jj]);
    }
  V.c_iso[iq] = HT(iso);
  if (V.c_pe) { // afterSolveStep -> updateEnergies (material_plastic.cc:86-99)
    CT dd = CT(0);
#pragma unroll
    for (int jj = 0; jj < 3; ++jj)
#pragma unroll
      for (int ii = 0; ii < 3; ++ii)
        dd += (S[ii][jj] + ps[ii][jj]) * (eps[ii][jj] - pe[ii][jj]);
    V.c_pe[iq] = HT(CT(V.p_pe[iq]) + dd / CT(2));
  }
}

// The total-strain form with the compact state (plastic strain in Voigt
// order and hardening, FP32): the batched FP32 form.
template <class CT>
__device__ __forceinline__ void plastic_at(const QpCompact &V, int64_t iq, CT lambda,
                                           CT mu, CT sy, CT hh, const CT (&g)[3][3],
                                           CT (&S)[3][3]) {
  CT pe[6], pn[6], iso;
#pragma unroll
  for (int k = 0; k < 6; ++k)
    pe[k] = CT(V.p_eps[(int64_t)k * V.nq_all + iq]);
  plastic_lih_total(lambda, mu, sy, hh, g, pe, CT(V.p_iso[iq]), S, pn, iso);
#pragma unroll
  for (int k = 0; k < 6; ++k)
    V.c_eps[(int64_t)k * V.nq_all + iq] = float(pn[k]);
  V.c_iso[iq] = float(iso);
}

// Constitutive law at one Gauss point: g -> stress S (sigma or PK2) and the
// tensor P contracted with dN/dX (sigma, or F S for finite deformation).
template <int LAW, class CT, class VT>
__device__ __forceinline__ void law_at(const VT &V, int64_t iq, CT lambda,
                                       CT mu, CT sy, CT hh, const CT (&g)[3][3],
                                       CT (&S)[3][3], CT (&P)[3][3]) {
  if constexpr (LAW == LAW_ELASTIC) {
    elastic_stress(lambda, mu, g, CT(0), S);
  } else if constexpr (LAW == LAW_ELASTIC_FD) {
    CT E[3][3];
    green_strain(g, E);
    elastic_stress(lambda, mu, E, CT(0), S);
  } else if constexpr (LAW == LAW_NEOHOOKEAN) {
    if constexpr (sizeof(CT) == 4)
      neohookean_pk2_stable(lambda, mu, g, S);
    else
      neohookean_pk2(lambda, mu, g, S);
  } else {
    plastic_at(V, iq, lambda, mu, sy, hh, g, S);
  }
  if (V.grad_u) {
#pragma unroll
    for (int jj = 0; jj < 3; ++jj)
#pragma unroll
      for (int ii = 0; ii < 3; ++ii) {
        const int64_t o = (int64_t)(ii + 3 * jj) * V.nq_all + iq;
        V.grad_u[o] = double(g[ii][jj]);
        V.stress[o] = double(S[ii][jj]);
      }
  }
  if constexpr (LAW == LAW_ELASTIC_FD || LAW == LAW_NEOHOOKEAN) {
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
      for (int J = 0; J < 3; ++J) {
        CT s = S[k][J]; // F S = S + grad u S
#pragma unroll
        for (int m = 0; m < 3; ++m)
          s += g[k][m] * S[m][J];
        P[k][J] = s;
      }
  } else {
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
      for (int J = 0; J < 3; ++J)
        P[k][J] = S[k][J];
  }
}

template <class CT>
__device__ __forceinline__ void element_params(const ElemArgs &A, int64_t i,
                                               CT &lambda, CT &mu, CT &sy,
                                               CT &hh) {
  if (sizeof(CT) == 4 && A.lm_f) { // the same FP32 values, one 8-byte load
    const float2 v = A.lm_f[i];
    lambda = CT(v.x);
    mu = CT(v.y);
  } else {
    lambda = CT(A.lam_el ? A.lam_el[i] : A.lambda);
    mu = CT(A.mu_el ? A.mu_el[i] : A.mu);
  }
  sy = CT(A.sy_el ? A.sy_el[i] : A.sigma_y);
  hh = CT(A.h_el ? A.h_el[i] : A.h);
}

// ---------------------------------------------------------------------------
// Hex8: 8 lanes per element.  hex8_group handles EPB elements; every lane of
// the block calls it (it holds barriers), lanes without an element with
// active = false.  sD must hold dN_n/dxi_m ([q][m][n]) before the call.
// ---------------------------------------------------------------------------
constexpr int HEX_EPB = 32; // elements per 256-thread block

template <int LAW, class CT, class FT, class VT, int EPB, class NA, int W = 3>
__device__ __forceinline__ void hex8_group(CT (&sN)[EPB][8][6], CT (&sQ)[EPB][8][9],
                                           const CT (&sD)[8][3][8], int el, int q,
                                           bool active, const int32_t *conn_e,
                                           const NA &nodes_of, CT lambda, CT mu, CT sy,
                                           CT hh, const VT &V, int64_t iq,
                                           const int32_t *pos_e, FT *fe) {
  // lane q stages node q: absolute in FP64; in FP32 relative to node 0 of
  // the element (exact FP64 difference, rounded once; lanes 8 el .. 8 el + 7
  // are one element, so node 0 comes from the first lane of the 8)
  double x[3] = {0., 0., 0.}, d[3] = {0., 0., 0.};
  if (active)
    nodes_of.load(conn_e[q], x, d);
  if constexpr (sizeof(CT) == 4) {
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      x[c] -= __shfl(x[c], 0, 8);
      d[c] -= __shfl(d[c], 0, 8);
    }
  }
  if (active) {
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      sN[el][q][c] = CT(x[c]);
      sN[el][q][3 + c] = CT(d[c]);
    }
  }
  __syncthreads();
  if (active) {
    CT J[3][3], H[3][3];
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int b = 0; b < 3; ++b) {
        J[a][b] = CT(0);
        H[a][b] = CT(0);
      }
#pragma unroll
    for (int n = 0; n < 8; ++n) {
      CT xn[3], un[3];
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        xn[c] = sN[el][n][c];
        un[c] = sN[el][n][3 + c];
      }
#pragma unroll
      for (int m = 0; m < 3; ++m) {
        const CT d = sD[q][m][n];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          J[m][c] += d * xn[c];
          H[c][m] += un[c] * d;
        }
      }
    }
    CT Ji[3][3];
    const CT wJ = inv_det(J, Ji); // Hex8 Gauss weights are 1
    CT g[3][3];
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int b = 0; b < 3; ++b) {
        CT s = CT(0);
#pragma unroll
        for (int m = 0; m < 3; ++m)
          s += H[a][m] * Ji[b][m];
        g[a][b] = s;
      }
    CT S[3][3], P[3][3];
    law_at<LAW, CT>(V, iq, lambda, mu, sy, hh, g, S, P);
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
      for (int m = 0; m < 3; ++m) {
        CT s = CT(0);
#pragma unroll
        for (int J2 = 0; J2 < 3; ++J2)
          s += P[k][J2] * Ji[J2][m];
        sQ[el][q][3 * k + m] = wJ * s;
      }
  }
  __syncthreads();
  if (active) {
    const int n = q; // this lane now owns node n of the element
    CT r[3] = {CT(0), CT(0), CT(0)};
#pragma unroll
    for (int qq = 0; qq < 8; ++qq)
#pragma unroll
      for (int m = 0; m < 3; ++m) {
        const CT d = sD[qq][m][n];
#pragma unroll
        for (int k = 0; k < 3; ++k)
          r[k] += sQ[el][qq][3 * k + m] * d;
      }
    akx::put_entry<W>(fe, (int64_t)pos_e[n], FT(r[0]), FT(r[1]), FT(r[2]));
  }
}

// ---------------------------------------------------------------------------
// Hex8, FP32 form, sum-factorised.  The trilinear shape functions at the
// 2 x 2 x 2 Gauss points factor per natural axis: along an axis, a node pair
// (v-, v+) maps to the two Gauss points by
//   I: alpha v_own + beta v_partner          (interpolation)
//   D: (v+ - v-) / 2                           (derivative)
// with alpha, beta = (1 +- 1/sqrt(3)) / 2.  With the 8 lanes of an element
// indexed by corner bits (bit a set = + side of axis a), node and Gauss point
// of a lane share the bits, so every axis step is a butterfly with the lane
// 1, 2 or 4 away:
//   J, H:   row m of [J|H] = D on axis m, I on the other two      (nodes -> q)
//   force:  F = sum_m (D^T on axis m, I on the other two) Q_m     (q -> nodes)
// The lanes apply the raw steps  I' = v + r p  (r = beta / alpha) and
// D' = v - p (own minus partner).  Then J' = c S J and H' = c H S with
// c = 2 / alpha^2 and S = diag(s_m), s_m = the lane's sign on axis m, so
// grad u = H' J'^-1 = H J^-1 unchanged, and the raw transposed chain applied
// to Q' = (sigma / c^3) det(J') P J'^-1, sigma = s_0 s_1 s_2, gives the
// nodal forces sum_q Q_q dN/dxi_q.  No LDS and no barriers: 14 exchanges
// per component instead of 8 x 3 products over the nodes.
// Bits -> node of the reference's numbering (counter-clockwise faces):
// n(b) = b ^ ((b >> 1) & 1); the Gauss point index is the bits themselves.
// ---------------------------------------------------------------------------
__device__ __forceinline__ float lane_x4(float v) { // value of the lane 4 away (swizzle)
  return __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(v), 0x101F));
}

constexpr float HEX_G = 0.57735026918962576f;          // 1 / sqrt(3)
constexpr float HEX_R = 0.26794919243112270f;          // beta / alpha = (1 - G) / (1 + G)
constexpr float HEX_C3 = 33.243067814700545f;          // c^3, c = 2 / alpha^2

// One butterfly step as one instruction, the partner's value read through
// DPP: acc + r v_partner (v_fmac_f32_dpp) and v - v_partner
// (v_subrev_f32_dpp).  The compiler does not fuse a DPP move into an FMA
// here, so the steps are written out; s_nop 4 gives the wait states a DPP
// read needs after a VALU write of its source (2) or of EXEC (5), which the
// compiler cannot account for inside asm.  Partners are lanes of the same
// element, so they are active whenever the lane is.
#define AKXF_DPP_STEPS(SUFFIX, PERM)                                                      \
  __device__ __forceinline__ float fmac_##SUFFIX(float acc, float v, float r) {           \
    asm("s_nop 4\n\tv_fmac_f32_dpp %0, %1, %2 quad_perm:" PERM                            \
        " row_mask:0xf bank_mask:0xf bound_ctrl:1"                                         \
        : "+v"(acc)                                                                        \
        : "v"(v), "v"(r));                                                                 \
    return acc;                                                                            \
  }                                                                                        \
  __device__ __forceinline__ float diff_##SUFFIX(float v) {                                \
    float d;                                                                               \
    asm("s_nop 4\n\tv_subrev_f32_dpp %0, %1, %1 quad_perm:" PERM                          \
        " row_mask:0xf bank_mask:0xf bound_ctrl:1"                                         \
        : "=v"(d)                                                                          \
        : "v"(v));                                                                         \
    return d;                                                                              \
  }
AKXF_DPP_STEPS(x1, "[1,0,3,2]")
AKXF_DPP_STEPS(x2, "[2,3,0,1]")
#undef AKXF_DPP_STEPS

// r in a vector register (the source operand of v_fmac_f32_dpp)
__device__ __forceinline__ float hex_r_vgpr() {
  float r;
  asm volatile("v_mov_b32 %0, 0x3e8930a3" : "=v"(r)); // HEX_R
  return r;
}

// [J' | H'] rows xi, eta, zeta at this lane's Gauss point, from the node
// values of one component.
__device__ __forceinline__ void hex_sf_grad(float R, float v, float &rx, float &ry,
                                            float &rz) {
  const float p = lane_x4(v);
  const float a = v - p, b = v + p * R;                 // axis 2: D, I
  const float a1 = fmac_x2(a, a, R);                    // axis 1: I, D, I
  const float b1 = diff_x2(b), c1 = fmac_x2(b, b, R);
  rz = fmac_x1(a1, a1, R);                              // axis 0: I, I, D
  ry = fmac_x1(b1, b1, R);
  rx = diff_x1(c1);
}

// One force component of this lane's node from Q'_(xi, eta, zeta).
__device__ __forceinline__ float hex_sf_force(float R, float qx, float qy, float qz) {
  const float A = diff_x1(qx);                          // axis 0: D^T, I, I
  const float B = fmac_x1(qy, qy, R);
  const float C = fmac_x1(qz, qz, R);
  const float E = fmac_x2(A, A, R) + diff_x2(B);        // axis 1: I, D^T; I
  const float Cz = fmac_x2(C, C, R);
  return (E + lane_x4(E) * R) + (Cz - lane_x4(Cz));     // axis 2: I, D^T
}

// corner of the lane with bits b
__device__ __forceinline__ int hex_node_of_lane(int b) {
  const int node = b ^ ((b >> 1) & 1);
  return node;
}

// All 64 lanes of the wave call it (cross-lane steps); lanes 8 e .. 8 e + 7
// are element e, lane bits b = l % 8.  Lanes of elements beyond the range
// pass active = false and compute on zeros.  nd: the node of the lane's
// corner (hex_node_of_lane) in nodes_of; F: the force on it.
template <int LAW, class VT, class NA>
__device__ __forceinline__ void hex8_group_sf(int b, bool active, int32_t nd, const NA &nodes_of,
                                              float lambda, float mu, float sy, float hh,
                                              const VT &V, int64_t iq, float (&F)[3]) {
  double x[3] = {0., 0., 0.}, d[3] = {0., 0., 0.};
  if (active)
    nodes_of.load(nd, x, d);
  const float R = hex_r_vgpr();
  // relative to node 0 (lane bits 0): exact FP64 difference, rounded once
  float J[3][3], H[3][3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const float xr = float(x[c] - __shfl(x[c], 0, 8));
    const float ur = float(d[c] - __shfl(d[c], 0, 8));
    hex_sf_grad(R, xr, J[0][c], J[1][c], J[2][c]);
    hex_sf_grad(R, ur, H[c][0], H[c][1], H[c][2]);
  }
  float Ji[3][3];
  const float dJ = inv_det(J, Ji);
  float g[3][3];
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int bb = 0; bb < 3; ++bb) {
      float s = 0.f;
#pragma unroll
      for (int m = 0; m < 3; ++m)
        s += H[a][m] * Ji[bb][m];
      g[a][bb] = s;
    }
  float S[3][3], P[3][3] = {};
  if (active)
    law_at<LAW, float>(V, iq, lambda, mu, sy, hh, g, S, P);
  // sigma = s_0 s_1 s_2 = +1 when an even number of bits are clear
  const float sig = ((3 - __builtin_popcount(b)) & 1) ? -1.f : 1.f;
  const float w = dJ * (sig / HEX_C3);
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    float q[3];
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      float s = 0.f;
#pragma unroll
      for (int J2 = 0; J2 < 3; ++J2)
        s += P[k][J2] * Ji[J2][m];
      q[m] = w * s;
    }
    F[k] = hex_sf_force(R, q[0], q[1], q[2]);
  }
}

template <int LAW, class FT>
__global__ void __launch_bounds__(256) k_hex8_sf(ElemArgs A) {
  const int t = threadIdx.x, el = t >> 3, b = t & 7;
  const int64_t i = xcd_block(A.nblocks_padded) * HEX_EPB + el;
  const bool active = i < A.n;
  int64_t e = 0;
  float lambda = 0.f, mu = 0.f, sy = 0.f, hh = 0.f;
  if (active) {
    e = A.filter ? (int64_t)A.filter[i] : A.first + i;
    element_params(A, i, lambda, mu, sy, hh);
  }
  int32_t nd = 0, pos = 0;
  if (active) {
    nd = A.conn[e * 8 + hex_node_of_lane(b)];
    pos = A.pos[(A.pos_offset + i) * 8 + hex_node_of_lane(b)];
  }
  float F[3];
  hex8_group_sf<LAW>(b, active, nd, NodesSoA{A.X, A.u, A.nn}, lambda, mu, sy, hh, qp_view(A, 8),
                     i * 8 + b, F);
  if (active)
    akx::put_entry<3>(reinterpret_cast<FT *>(A.fe), (int64_t)pos, FT(F[0]), FT(F[1]), FT(F[2]));
}

// ---------------------------------------------------------------------------
// Hex8, FP32 form, four lanes per element (the block-partial passes).  Lane
// bits (y, z) own the two nodes and the two Gauss points of one x edge: the x
// axis is worked in the lane, y and z as the butterflies above with the lanes
// 1 and 2 away, all within a quad:
//   D: v_own - v_partner,   I: v_own + r v_partner
// With d = v+ - v- and s = v+ + v- along x, the rows of J' and H' at
// xi = +-G are
//   d/dxi = I_y I_z d,  d/deta = D_y I_z (KS s +- KD d),  d/dzeta = I_y D_z (KS s +- KD d)
// KD = G KS: the two Gauss points share every step but one addition per row.
// The rows are c_m s_m times the true ones (c_0 = 2 (1 + r)^2, c_1 = c_2 =
// 4 KS (1 + r), s_0 = 1), which g = H' J'^-1 does not see, and the transposed
// steps (D and I are symmetric) applied to Q' = W s_y s_z P adj(J'),
// W = 1 / (c_0 c_1 c_2), give the nodal forces.  tests/test_hex8_quad_cpu.py
// restates the steps lane by lane.
//
// A constant's rounding shifts the stiffness of every element and step alike:
// 1e-8 of it is 1e-6 of the displacement after 300 steps.  So the constants
// are ones that FP32 holds well: r to 5e-9, KS exactly, KD to 1e-10 (KS is
// free; 1 / 2 with KD = G / 2 would be off by 1.8e-8), and W goes into the Lame
// constants in FP64 (LameF).  Stiffness bias -1e-9, against -3.6e-8 of
// hex8_group_sf (numpy emulation of both).
//
// Bound by FP32 vector issue on large meshes: 700 VALU instructions per wave
// of 16 elements against 2 x 408 with one lane per Gauss point
// (hex8_group_sf), 93% of the cycles busy (SQ_ACTIVE_INST_VALU against
// GRBM_GUI_ACTIVE).  Block pass, neo-Hookean, 2 M elements 163-173 -> 155 us,
// 255,000 33.9 -> 27.6 us, 19,740 16.7 -> 8.8 us and 1,000 16.1 -> 6.9 us (the
// former blocks of 192 elements ran six groups of 32 one after another, on
// 104 workgroups for the 19,740).  Also measured on 2 M elements: one lane
// per element 259 us (181 VGPRs, two waves per SIMD); four lanes with the
// corners read from the X and u arrays 169 us (lanes of a quad lie in four
// rows, so every lane is an L1 access of its own: 110 M per pass against 23 M
// with the records staged in LDS).
// ---------------------------------------------------------------------------
constexpr float HEX_KS = 0.63818359375f;      // 1307 / 2048
constexpr float HEX_KD = 0.36845546964396530f; // HEX_KS / sqrt(3)
constexpr double HEX_W = 1. / (2. * (1. + (double)HEX_R) * (1. + (double)HEX_R) * 16. *
                               (double)HEX_KS * (double)HEX_KS * (1. + (double)HEX_R) *
                               (1. + (double)HEX_R));

// the value of the lane 1 / 2 away, of the quad's first lane
__device__ __forceinline__ float quad_x1(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xf, 0xf, true));
}
__device__ __forceinline__ float quad_x2(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4E, 0xf, 0xf, true));
}
__device__ __forceinline__ double quad_first(double v) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0x00, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0x00, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}

// One component's node values (v0 at x-, v1 at x+ of the lane's edge) ->
// d/dxi and the parts of d/deta = e0 +- KD e1 and d/dzeta = z0 +- KD z1.
__device__ __forceinline__ void quad_grad(float v0, float v1, float &dxi, float &e0, float &e1,
                                          float &z0, float &z1) {
  const float d = v1 - v0, s = HEX_KS * (v0 + v1);
  const float dp = quad_x2(d), sp = quad_x2(s);
  const float dzd = d - dp, izd = d + HEX_R * dp;
  const float dzs = s - sp, izs = s + HEX_R * sp;
  const float ip = quad_x1(izd);
  dxi = izd + HEX_R * ip;
  e0 = izs - quad_x1(izs);
  e1 = izd - ip;
  z0 = dzs + HEX_R * quad_x1(dzs);
  z1 = dzd + HEX_R * quad_x1(dzd);
}

// The transposed steps: one force component of the lane's nodes from the
// rows of Q' at xi = -G (m) and xi = +G (p).
__device__ __forceinline__ void quad_force(const float (&m)[3], const float (&p)[3], float &f0,
                                           float &f1) {
  const float X = p[0] + m[0];
  const float Se = p[1] + m[1], de = p[1] - m[1];
  const float Sz = p[2] + m[2], Z = HEX_KD * (p[2] - m[2]);
  // I a + D b = (a + b) + partner's (r a - b)
  // I_y X + D_y E, E = KD de
  const float da = (X + HEX_KD * de) + quad_x1(HEX_R * X - HEX_KD * de);
  const float db = Z + HEX_R * quad_x1(Z);
  const float d = (da + db) + quad_x2(HEX_R * da - db);
  const float sa = Se - quad_x1(Se);
  const float sb = Sz + HEX_R * quad_x1(Sz);
  const float s = (sa + sb) + quad_x2(HEX_R * sa - sb);
  f0 = HEX_KS * s - d;
  f1 = HEX_KS * s + d;
}

// adjugate: K = det(m) m^-1
__device__ __forceinline__ void adjugate(const float (&m)[3][3], float (&K)[3][3]) {
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const int i1 = (i + 1) % 3, i2 = (i + 2) % 3, j1 = (j + 1) % 3, j2 = (j + 2) % 3;
      K[j][i] = m[i1][j1] * m[i2][j2] - m[i1][j2] * m[i2][j1];
    }
}

// Lame constants times HEX_W and the lane's sign as hi + lo floats: rounded to
// FP32 alone, a material's constants are off by up to 3e-8 in every element
// and step (per-element constants come rounded, theirs scatter).
struct LameF {
  float l, m, l_lo, m_lo;
  __device__ __forceinline__ float times_l(float x) const { return fmaf(l, x, l_lo * x); }
  __device__ __forceinline__ float times_m(float x) const { return fmaf(m, x, m_lo * x); }
  __device__ __forceinline__ float times_m_plus(float x, float c) const {
    return fmaf(m, x, fmaf(m_lo, x, c));
  }
};

// b: the quad lane, s_y s_z = -1 on lanes 1 and 2
__device__ __forceinline__ LameF lame_quad(double lambda, double mu, int b) {
  const double w = (b == 1 || b == 2) ? -HEX_W : HEX_W;
  const double lw = lambda * w, mw = mu * w;
  const float l = float(lw), m = float(mw);
  return LameF{l, m, float(lw - double(l)), float(mw - double(m))};
}

// Q'[k][m] = W s_y s_z (P adj(J'))[k][m] of one Gauss point from the rows
// J'[m][c] = c_m s_m dX_c/dxi_m and H'[m][c] (elastic laws and neo-Hookean);
// lambda, mu: the material's constants, for the stress that is stored.
template <int LAW, class VT>
__device__ __forceinline__ void hex8_point(const float (&J)[3][3], const float (&H)[3][3],
                                           const LameF &L, float lambda, float mu,
                                           const VT &V, int64_t iq, float (&Q)[3][3]) {
  float K[3][3], g[3][3];
  adjugate(J, K);
  const float id = akx_rcp(J[0][0] * K[0][0] + J[0][1] * K[1][0] + J[0][2] * K[2][0]);
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int b = 0; b < 3; ++b)
      g[a][b] = (H[0][a] * K[b][0] + H[1][a] * K[b][1] + H[2][a] * K[b][2]) * id;
  constexpr int I6[6] = {0, 1, 2, 0, 0, 1}, J6[6] = {0, 1, 2, 1, 2, 2};
  float T[3][3], P[3][3];
  if (V.grad_u) { // materialise grad u and the stress
    law_at<LAW, float>(V, iq, lambda, mu, 0.f, 0.f, g, T, P);
  }
  if constexpr (LAW == LAW_NEOHOOKEAN) {
    // on the current configuration: tau = F S F^T = mu (b - I) + lambda ln J I
    // with b - I = g + g^T + g g^T, and det J P J^-1 = (1 / det F) tau
    // adj(J + H): no inverse of C and no product F S, and like the form with
    // S free of cancellation (neohookean_pk2_stable)
    const float tr = g[0][0] + g[1][1] + g[2][2];
    // J - 1 = tr g + (sum of the principal 2 x 2 minors) + det g
    float Kg[3][3];
    adjugate(g, Kg);
    const float dg = g[0][0] * Kg[0][0] + g[0][1] * Kg[1][0] + g[0][2] * Kg[2][0];
    const float jm1 = tr + (Kg[0][0] + Kg[1][1] + Kg[2][2] + dg);
    const float w = akx_rcp(1.f + jm1);
    const float wm = L.times_m(w), wl = w * L.times_l(akx_log1p(jm1));
#pragma unroll
    for (int v = 0; v < 6; ++v) {
      const int i = I6[v], j = J6[v];
      float p = g[i][j] + g[j][i];
#pragma unroll
      for (int k = 0; k < 3; ++k)
        p += g[i][k] * g[j][k];
      T[i][j] = T[j][i] = i == j ? wm * p + wl : wm * p;
    }
    float jc[3][3];
#pragma unroll
    for (int m = 0; m < 3; ++m)
#pragma unroll
      for (int c = 0; c < 3; ++c)
        jc[m][c] = J[m][c] + H[m][c];
    adjugate(jc, K);
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
      for (int m = 0; m < 3; ++m)
        P[k][m] = T[k][m];
  } else {
    // S = lambda tr(e) I + 2 mu e, e the strain (2 e = g + g^T (+ g^T g))
    float e2[6];
#pragma unroll
    for (int v = 0; v < 6; ++v) {
      const int i = I6[v], j = J6[v];
      e2[v] = g[i][j] + g[j][i];
      if constexpr (LAW == LAW_ELASTIC_FD)
#pragma unroll
        for (int k = 0; k < 3; ++k)
          e2[v] += g[k][i] * g[k][j];
    }
    const float sd = 0.5f * L.times_l(e2[0] + e2[1] + e2[2]);
#pragma unroll
    for (int v = 0; v < 6; ++v)
      T[I6[v]][J6[v]] = T[J6[v]][I6[v]] =
          v < 3 ? L.times_m_plus(e2[v], sd) : L.times_m(e2[v]);
    // P = sigma, or F S
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
      for (int m = 0; m < 3; ++m) {
        P[k][m] = T[k][m];
        if constexpr (LAW == LAW_ELASTIC_FD)
#pragma unroll
          for (int c = 0; c < 3; ++c)
            P[k][m] += g[k][c] * T[c][m];
      }
  }
#pragma unroll
  for (int k = 0; k < 3; ++k)
#pragma unroll
    for (int m = 0; m < 3; ++m)
      Q[k][m] = P[k][0] * K[0][m] + P[k][1] * K[1][m] + P[k][2] * K[2][m];
}

// Quad lane b (bit 0 y, bit 1 z) of one element; lc, ls: its two corners'
// indices in the block's node records and their LDS slots.  All four lanes of
// an active element call it.
template <int LAW, class VT, class NA>
__device__ __forceinline__ void hex8_quad(int b, uint32_t lc, uint32_t ls, const NA &nodes_of,
                                          const LameF &L, float lambda, float mu,
                                          const VT &V, int64_t iq0, float *s_f) {
  // nodes of a face run counter-clockwise: (x-, x+) at y-, (x+, x-) at y+
  const int yp = (b & 1) * 16;
  lc = __funnelshift_r(lc, lc, yp);
  ls = __funnelshift_r(ls, ls, yp);
  double x0[3], d0[3], x1[3], d1[3];
  nodes_of.load((int32_t)(lc & 0xffffu), x0, d0);
  nodes_of.load((int32_t)(lc >> 16), x1, d1);
  // relative to node 0 (lane 0, x-): exact FP64 difference, rounded once
  float Jx[3], Hx[3], xe0[3], xe1[3], xz0[3], xz1[3], ue0[3], ue1[3], uz0[3], uz1[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const double xr = quad_first(x0[c]), ur = quad_first(d0[c]);
    quad_grad(float(x0[c] - xr), float(x1[c] - xr), Jx[c], xe0[c], xe1[c], xz0[c], xz1[c]);
    quad_grad(float(d0[c] - ur), float(d1[c] - ur), Hx[c], ue0[c], ue1[c], uz0[c], uz1[c]);
  }
  float Qm[3][3], Qp[3][3];
#pragma unroll
  for (int ix = 0; ix < 2; ++ix) {
    float J[3][3], H[3][3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      J[0][c] = Jx[c];
      H[0][c] = Hx[c];
      const float kd = ix ? HEX_KD : -HEX_KD;
      J[1][c] = xe0[c] + kd * xe1[c];
      H[1][c] = ue0[c] + kd * ue1[c];
      J[2][c] = xz0[c] + kd * xz1[c];
      H[2][c] = uz0[c] + kd * uz1[c];
    }
    hex8_point<LAW>(J, H, L, lambda, mu, V, iq0 + (ix + 2 * b), ix ? Qp : Qm);
  }
  float *o0 = s_f + 3 * (ls & 0xffffu), *o1 = s_f + 3 * (ls >> 16);
#pragma unroll
  for (int k = 0; k < 3; ++k)
    quad_force(Qm[k], Qp[k], o0[k], o1[k]);
}

// The plastic law of a block of n elements goes eight lanes per element, 32
// elements at a time: consecutive lanes then read consecutive Gauss points of
// its history (four lanes per element, two points each, read every second
// value per load: block pass of 150,000 elements 143 -> 233 us).  lconn,
// lslot, iq0: the block's first element and Gauss point; params(i, lambda, mu,
// sy, hh) gives the constants of its i-th element.
template <class VT, class PF>
__device__ __forceinline__ void hex8_plastic_block(int n, const uint16_t *lconn,
                                                   const uint16_t *lslot,
                                                   const akx::NodesLDS &rec, const VT &V,
                                                   int64_t iq0, const PF &params, float *s_f) {
  for (int base = 0; base < n; base += 32) {
    const int el = base + (threadIdx.x >> 3), b = threadIdx.x & 7;
    const bool active = el < n;
    const int ec = active ? el : 0, c = ec * 8 + hex_node_of_lane(b);
    float lambda, mu, sy, hh, F[3];
    params(ec, lambda, mu, sy, hh);
    hex8_group_sf<LAW_PLASTIC>(b, active, lconn[c], rec, lambda, mu, sy, hh, V, iq0 + ec * 8 + b,
                               F);
    if (active) {
      float *o = s_f + 3 * lslot[c];
      o[0] = F[0];
      o[1] = F[1];
      o[2] = F[2];
    }
  }
}

// the slots s0 .. s1 - 1 of one (block, node) in order, FP64, rounded once.
// SPREAD: they lie at slot_pos (Tet4)
template <bool SPREAD>
__device__ __forceinline__ void sum_slots(const float *s_f, int s0, int s1, float *fe,
                                          int64_t entry) {
  double fx = 0., fy = 0., fz = 0.;
  for (int sl = s0; sl < s1; ++sl) {
    const float *f = s_f + 3 * (SPREAD ? slot_pos(sl) : sl);
    fx += (double)f[0];
    fy += (double)f[1];
    fz += (double)f[2];
  }
  akx::put_entry<3>(fe, entry, float(fx), float(fy), float(fz));
}

// FP32 Hex8 with block-partial assembly: each workgroup does one block of
// BPA_HEX8 consecutive elements, four lanes each.  The {X, u} records of the
// block's distinct nodes (ascending ids) are staged in LDS; the lanes put
// their nodes' forces in LDS slots (the corners of one distinct node of the
// block take consecutive slots in ascending element order), then one thread
// per distinct node adds its slots in that order (FP64, rounded once) and
// writes one table entry per (block, node).  The gather adds a node's
// partials in block order.  63 elements: 252 of the 256 lanes, and a block
// inside one row of cells has 4 x 64 distinct nodes, one per lane in the
// staging and summing phases.
// MAT: grad u and the stress are stored (computeAllStresses); a variant of its
// own, whose code kept 60 registers more alive in every step's pass.
template <int LAW, bool MAT>
__global__ void __launch_bounds__(256) k_hex8_bpa(ElemArgs A) {
  extern __shared__ double2 s_xu[]; // [bl_maxu][3] records, then [63 * 8][3] floats
  float *s_f = reinterpret_cast<float *>(s_xu + 3 * A.bl_maxu);
  QpViewT<double> V = qp_view(A, 8);
  if constexpr (!MAT)
    V.grad_u = V.stress = nullptr;
  const int t = threadIdx.x;
  const int64_t blk = xcd_block(A.nblocks_padded);
  const int64_t i0 = blk * akx::BPA_HEX8, i = i0 + (t >> 2);
  if (i0 >= A.n) // padding block: no elements, no node list
    return;
  const bool active = (t >> 2) < akx::BPA_HEX8 && i < A.n;
  // the lane's own streams and its first node of the summing phase first, so
  // that their loads overlap the staging
  uint32_t lc = 0, ls = 0;
  double lambda = A.lambda, mu = A.mu;
  if (LAW != LAW_PLASTIC && active) {
    lc = reinterpret_cast<const uint32_t *>(A.lconn + i * 8)[t & 3];
    ls = reinterpret_cast<const uint32_t *>(A.lslot + i * 8)[t & 3];
    if (A.lm_f) {
      lambda = A.lm_f[i].x;
      mu = A.lm_f[i].y;
    }
  }
  const uint16_t *soff = A.bl_soff + blk * (A.bl_maxu + 1);
  const int32_t *dst = A.bl_pos + blk * A.bl_maxu;
  int32_t d_first = -1;
  int s0_first = 0, s1_first = 0;
  if (t < A.bl_maxu) {
    d_first = dst[t];
    s0_first = soff[t];
    s1_first = soff[t + 1];
  }
  akx::stage_block_records(A, blk, s_xu);
  __syncthreads();
  const akx::NodesLDS rec{reinterpret_cast<const double *>(s_xu)};
  if constexpr (LAW == LAW_PLASTIC)
    hex8_plastic_block((int)min((int64_t)akx::BPA_HEX8, A.n - i0), A.lconn + i0 * 8,
                       A.lslot + i0 * 8, rec, V, i0 * 8,
                       [&](int el, float &l, float &m, float &y, float &h) {
                         element_params(A, i0 + el, l, m, y, h);
                       },
                       s_f);
  else if (active)
    hex8_quad<LAW>(t & 3, lc, ls, rec, lame_quad(lambda, mu, t & 3), float(lambda), float(mu), V,
                   i * 8, s_f);
  __syncthreads();
  float *fe = reinterpret_cast<float *>(A.fe);
  for (int k = t; k < A.bl_maxu; k += 256) {
    const bool first = k == t;
    const int32_t d = first ? d_first : dst[k];
    if (d < 0)
      continue;
    const int s0 = first ? s0_first : soff[k], s1 = first ? s1_first : soff[k + 1];
    sum_slots<false>(s_f, s0, s1, fe, (int64_t)d);
  }
}

template <int LAW, class CT, class FT>
__global__ void __launch_bounds__(256) k_hex8_fast(ElemArgs A) {
  __shared__ CT sN[HEX_EPB][8][6];     // X (0..2) and u (3..5) of the 8 nodes
  __shared__ CT sQ[HEX_EPB][8][9];     // Q of the 8 Gauss points
  __shared__ CT sD[8][3][8];           // dN_n/dxi_m at Gauss point q
  const int t = threadIdx.x, el = t >> 3, q = t & 7;
  for (int k = t; k < 192; k += 256)
    (&sD[0][0][0])[k] = CT((&c_dnds[0][0][0])[k]);
  const int64_t i = xcd_block(A.nblocks_padded) * HEX_EPB + el;
  const bool active = i < A.n;
  int64_t e = 0;
  CT lambda = CT(0), mu = CT(0), sy = CT(0), hh = CT(0);
  if (active) {
    e = A.filter ? (int64_t)A.filter[i] : A.first + i;
    element_params(A, i, lambda, mu, sy, hh);
  }
  hex8_group<LAW, CT, FT, QpViewT<double>, HEX_EPB>(
      sN, sQ, sD, el, q, active, A.conn + e * 8, NodesSoA{A.X, A.u, A.nn}, lambda, mu, sy,
      hh,
      qp_view(A, 8), i * 8 + q, A.pos + (A.pos_offset + (active ? i : 0)) * 8,
      reinterpret_cast<FT *>(A.fe));
}

// ---------------------------------------------------------------------------
// Tet4: one thread per element
// ---------------------------------------------------------------------------
// EARLY_POS: load the table positions beside the connectivity and keep them
// there (the scheduler otherwise places the load at its use, after the element
// math, a third memory round trip per element).  Faster for the one-element-
// per-thread FP32 pass; slower inside the persistent batch loop, and in FP64
// it costs the pass a wave per SIMD.
// J = dX/dxi and H = du/dxi of one Tet4 element, differences of its corners.
// BARRIER: a scheduling barrier after the node loads, so that a load issued
// before the call stays ahead of the math.
template <class CT, class NA, bool BARRIER>
__device__ __forceinline__ void tet4_JH(const int4 nd, const NA &nodes_of, CT (&J)[3][3],
                                        CT (&H)[3][3]) {
  const int32_t nodes[4] = {nd.x, nd.y, nd.z, nd.w};
  double X[4][3], U[4][3];
#pragma unroll
  for (int n = 0; n < 4; ++n)
    nodes_of.load(nodes[n], X[n], U[n]);
  if constexpr (BARRIER)
    __builtin_amdgcn_sched_barrier(0);
  // natural directions: xi -> node 3, eta -> node 1, zeta -> node 2
  const int nm[3] = {3, 1, 2};
#pragma unroll
  for (int m = 0; m < 3; ++m)
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      J[m][c] = CT(X[nm[m]][c] - X[0][c]);
      H[c][m] = CT(U[nm[m]][c] - U[0][c]);
    }
}

// Q = w detJ P J^-1 of one Tet4 element (its corner forces are the columns
// of Q and minus their sum)
template <int LAW, class CT, class VT>
__device__ __forceinline__ void tet4_Q(const CT (&J)[3][3], const CT (&H)[3][3], CT lambda,
                                       CT mu, CT sy, CT hh, const VT &V, int64_t iq,
                                       CT (&Q)[3][3]) {
  CT Ji[3][3];
  const CT detJ = inv_det(J, Ji);
  const CT wJ = detJ * CT(1. / 6.);
  CT g[3][3];
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int b = 0; b < 3; ++b) {
      CT s = CT(0);
#pragma unroll
      for (int m = 0; m < 3; ++m)
        s += H[a][m] * Ji[b][m];
      g[a][b] = s;
    }
  CT S[3][3], P[3][3];
  law_at<LAW, CT>(V, iq, lambda, mu, sy, hh, g, S, P);
#pragma unroll
  for (int k = 0; k < 3; ++k)
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      CT s = CT(0);
#pragma unroll
      for (int J2 = 0; J2 < 3; ++J2)
        s += P[k][J2] * Ji[J2][m];
      Q[k][m] = wJ * s;
    }
}

template <int LAW, class CT, class FT, class VT, class NA, int W = 3, bool EARLY_POS = false>
__device__ __forceinline__ void tet4_one(const int4 nd, const NA &nodes_of,
                                         CT lambda, CT mu, CT sy, CT hh, const VT &V,
                                         int64_t iq, const int32_t *pos_e, FT *fe) {
  int4 pv;
  if constexpr (EARLY_POS)
    pv = *reinterpret_cast<const int4 *>(pos_e);
  CT J[3][3], H[3][3], Q[3][3];
  tet4_JH<CT, NA, EARLY_POS>(nd, nodes_of, J, H);
  tet4_Q<LAW, CT, VT>(J, H, lambda, mu, sy, hh, V, iq, Q);
  if constexpr (!EARLY_POS)
    pv = *reinterpret_cast<const int4 *>(pos_e);
  akx::put_entry<W>(fe, (int64_t)pv.x, FT(-(Q[0][0] + Q[0][1] + Q[0][2])),
                    FT(-(Q[1][0] + Q[1][1] + Q[1][2])), FT(-(Q[2][0] + Q[2][1] + Q[2][2])));
  akx::put_entry<W>(fe, (int64_t)pv.y, FT(Q[0][1]), FT(Q[1][1]), FT(Q[2][1]));
  akx::put_entry<W>(fe, (int64_t)pv.z, FT(Q[0][2]), FT(Q[1][2]), FT(Q[2][2]));
  akx::put_entry<W>(fe, (int64_t)pv.w, FT(Q[0][0]), FT(Q[1][0]), FT(Q[2][0]));
}

template <int LAW, class CT, class FT>
__global__ void __launch_bounds__(256) k_tet4_fast(ElemArgs A) {
  const int64_t i = xcd_block(A.nblocks_padded) * blockDim.x + threadIdx.x;
  if (i >= A.n)
    return;
  const int64_t e = A.filter ? (int64_t)A.filter[i] : A.first + i;
  CT lambda, mu, sy, hh;
  element_params(A, i, lambda, mu, sy, hh);
  tet4_one<LAW, CT, FT, QpViewT<double>, akx::NodesXU, 3, sizeof(CT) == 4>(
      *reinterpret_cast<const int4 *>(A.conn + e * 4), akx::NodesXU{A.xu}, lambda,
                                         mu, sy, hh,
                                qp_view(A, 1), i, A.pos + (A.pos_offset + i) * 4,
                                reinterpret_cast<FT *>(A.fe));
}

// FP32 Tet4 with the block's node records staged in LDS: the 256 elements of
// a block share about 0.7 distinct nodes each, so each record is read from
// global memory once per block instead of once per element corner.
template <int LAW>
__global__ void __launch_bounds__(256) k_tet4_lds(ElemArgs A) {
  extern __shared__ double2 s_xu[]; // [bl_maxu][3]
  const int64_t blk = xcd_block(A.nblocks_padded);
  if (blk * 256 >= A.n) // padding block: no elements, no node list
    return;
  const int64_t i = blk * 256 + threadIdx.x;
  const bool active = i < A.n;
  // the element's own streams are loaded before the staging, so that their
  // round trip overlaps it (loading the last element's for the lanes past
  // the end instead, without the branch, measured 2.5% slower here)
  ushort4 lc = make_ushort4(0, 0, 0, 0);
  int4 pv = make_int4(0, 0, 0, 0);
  float lambda = 0.f, mu = 0.f, sy = 0.f, hh = 0.f;
  if (active) {
    lc = *reinterpret_cast<const ushort4 *>(A.lconn + i * 4);
    pv = *reinterpret_cast<const int4 *>(A.pos + (A.pos_offset + i) * 4);
    element_params(A, i, lambda, mu, sy, hh);
  }
  akx::stage_block_records(A, blk, s_xu);
  __syncthreads();
  if (!active)
    return;
  tet4_one<LAW, float, float, QpViewT<double>, akx::NodesLDS, 3, true>(
      make_int4(lc.x, lc.y, lc.z, lc.w), akx::NodesLDS{reinterpret_cast<const double *>(s_xu)},
      lambda, mu, sy, hh, qp_view(A, 1), i, reinterpret_cast<const int32_t *>(&pv),
      reinterpret_cast<float *>(A.fe));
}

// FP32 Tet4 with block-partial assembly.  As k_tet4_lds, then the block sums
// the forces its elements put on each of its distinct nodes and writes one
// partial per (block, distinct node) instead of one table entry per element
// corner: the corner forces go to LDS slots (the corners of one distinct node
// take consecutive slots in ascending element order), and one thread per
// distinct node adds its slots in that order (in FP64, rounded once) and
// writes the partial.  The gather then adds a node's partials in ascending
// block order.  The table traffic falls from four entries per element to
// one per (block, node) pair: about 0.7 per element on the box meshes.
//
// Bound by a mix: VALU busy 44 % of the time, LDS 50 %, the rest the wait for
// the element's streams, then the node list, then the nodes.  The slots lie
// spread over the banks (slot_pos) and take the place of the records, whose
// differences are in registers by then: 8 instead of 7 workgroups per CU.  1.9 M
// elements 27.8 (dense slots, behind the records) -> 26.5 (spread) -> 25.6 us,
// 4.4 M 52.5 -> 49.7 -> 48.
template <int LAW>
__global__ void __launch_bounds__(256) k_tet4_bpa(ElemArgs A) {
  extern __shared__ double2 s_xu[]; // [bl_maxu][3] records, later the corner slots
  const int64_t blk = xcd_block(A.nblocks_padded);
  if (blk * 256 >= A.n) // padding block: no elements, no node list
    return;
  const int64_t i = blk * 256 + threadIdx.x;
  const bool active = i < A.n;
  ushort4 lc = make_ushort4(0, 0, 0, 0), ls = make_ushort4(0, 0, 0, 0);
  float lambda = 0.f, mu = 0.f, sy = 0.f, hh = 0.f;
  if (active) {
    lc = *reinterpret_cast<const ushort4 *>(A.lconn + i * 4);
    ls = *reinterpret_cast<const ushort4 *>(A.lslot + i * 4);
    element_params(A, i, lambda, mu, sy, hh);
  }
  // this lane's first distinct node of the summing phase, read ahead so
  // that its loads overlap the staging instead of following the barrier
  const uint16_t *soff = A.bl_soff + blk * (A.bl_maxu + 1);
  const int32_t *dst = A.bl_pos + blk * A.bl_maxu;
  int32_t d_first = -1;
  int s0_first = 0, s1_first = 0;
  if ((int)threadIdx.x < A.bl_maxu) {
    d_first = dst[threadIdx.x];
    s0_first = soff[threadIdx.x];
    s1_first = soff[threadIdx.x + 1];
  }
  akx::stage_block_records(A, blk, s_xu);
  __syncthreads();
  float J[3][3], H[3][3];
  tet4_JH<float, akx::NodesLDS, false>(
      make_int4(lc.x, lc.y, lc.z, lc.w),
      akx::NodesLDS{reinterpret_cast<const double *>(s_xu)}, J, H);
  __syncthreads(); // the records are dead: the LDS now takes the slots
  float *s_f = reinterpret_cast<float *>(s_xu);
  if (active) {
    float Q[3][3];
    tet4_Q<LAW, float>(J, H, lambda, mu, sy, hh, qp_view(A, 1), i, Q);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      s_f[3 * slot_pos(ls.x) + c] = -(Q[c][0] + Q[c][1] + Q[c][2]);
      s_f[3 * slot_pos(ls.y) + c] = Q[c][1];
      s_f[3 * slot_pos(ls.z) + c] = Q[c][2];
      s_f[3 * slot_pos(ls.w) + c] = Q[c][0];
    }
  }
  __syncthreads();
  float *fe = reinterpret_cast<float *>(A.fe);
  for (int k = threadIdx.x; k < A.bl_maxu; k += blockDim.x) {
    const bool first = k == (int)threadIdx.x;
    const int32_t d = first ? d_first : dst[k];
    if (d < 0)
      continue;
    const int s0 = first ? s0_first : soff[k], s1 = first ? s1_first : soff[k + 1];
    sum_slots<true>(s_f, s0, s1, fe, (int64_t)d);
  }
}

// One step of a small FP32 Tet4 model (akx_step.hpp): one lane per element of
// the workgroup's list, the corners of its own nodes to LDS slots.
template <int LAW> __global__ void __launch_bounds__(256) k_tet4_step_f32(StepArgs S) {
  extern __shared__ double2 s_rec[]; // records, then slots, then the runs' ends
  const int64_t b = xcd_block(S.nblocks_padded);
  if (b >= S.nblocks) // padding block
    return;
  const int t = threadIdx.x;
  float *s_slot = reinterpret_cast<float *>(s_rec + 3 * S.max_nodes);
  uint8_t *s_run = reinterpret_cast<uint8_t *>(s_slot + 3 * (S.max_slots + 1));
  // lanes past the list do its last element again, to the slot nothing reads
  const bool active = t < S.max_elems;
  const int64_t i = b * S.max_elems + (active ? t : S.max_elems - 1);
  const ushort4 lc = *reinterpret_cast<const ushort4 *>(S.lc + i * 4);
  const ushort4 ls = *reinterpret_cast<const ushort4 *>(S.ls + i * 4);
  float lambda = (float)S.lambda, mu = (float)S.mu;
  if (S.lm_f) {
    const float2 lm = S.lm_f[S.lelem[i] & ~akx::STEP_GUEST];
    lambda = lm.x;
    mu = lm.y;
  }
  StepDof<true> dof;
  dof.load(S, b);
  for (int k = t; k < S.max_slots; k += blockDim.x)
    s_run[k] = S.run[b * S.max_slots + k];
  step_stage<true>(S, b, s_rec);
  __syncthreads();
  if (active) {
    float J[3][3], H[3][3], Q[3][3];
    tet4_JH<float, akx::NodesLDS, false>(
        make_int4(lc.x, lc.y, lc.z, lc.w),
        akx::NodesLDS{reinterpret_cast<const double *>(s_rec)}, J, H);
    tet4_Q<LAW, float>(J, H, lambda, mu, 0.f, 0.f, QpViewT<double>{}, 0, Q);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      s_slot[3 * ls.x + c] = -(Q[c][0] + Q[c][1] + Q[c][2]);
      s_slot[3 * ls.y + c] = Q[c][1];
      s_slot[3 * ls.z + c] = Q[c][2];
      s_slot[3 * ls.w + c] = Q[c][0];
    }
  }
  __syncthreads();
  dof.update<true>(S, s_slot, s_run);
}

// The same for FP32 Hex8: four lanes per element (hex8_quad) of the up to 64
// around a workgroup's run of nodes.  Up to some 4,000 nodes the host's queueing
// and the load chain (lists, records, state) bound it, above the element code,
// done 3.5 to 4.3 times.  us a step of neo-Hookean boxes against
// two launches: 1,331 nodes 9.1 -> 5.6, 8,192 9.6 -> 6.8, 11,200 9.2 -> 8.0.
template <int LAW> __global__ void __launch_bounds__(256) k_hex8_step_f32(StepArgs S) {
  extern __shared__ double2 s_rec[]; // records, then slots, then the runs' ends
  const int64_t b = xcd_block(S.nblocks_padded);
  if (b >= S.nblocks) // padding block
    return;
  const int t = threadIdx.x, q = t & 3;
  float *s_slot = reinterpret_cast<float *>(s_rec + 3 * S.max_nodes);
  uint8_t *s_run = reinterpret_cast<uint8_t *>(s_slot + 3 * (S.max_slots + 1));
  const bool active = (t >> 2) < S.max_elems;
  const int64_t i = b * S.max_elems + (active ? t >> 2 : S.max_elems - 1);
  const uint32_t lc = reinterpret_cast<const uint32_t *>(S.lc + i * 8)[q];
  const uint32_t ls = reinterpret_cast<const uint32_t *>(S.ls + i * 8)[q];
  double lambda = S.lambda, mu = S.mu;
  if (S.lm_f) {
    const float2 lm = S.lm_f[S.lelem[i] & ~akx::STEP_GUEST];
    lambda = lm.x;
    mu = lm.y;
  }
  StepDof<true> dof;
  dof.load(S, b);
  for (int k = t; k < S.max_slots; k += blockDim.x)
    s_run[k] = S.run[b * S.max_slots + k];
  step_stage<true>(S, b, s_rec);
  __syncthreads();
  if (active)
    hex8_quad<LAW>(q, lc, ls, akx::NodesLDS{reinterpret_cast<const double *>(s_rec)},
                   lame_quad(lambda, mu, q), float(lambda), float(mu), QpViewT<double>{}, 0,
                   s_slot);
  __syncthreads();
  dof.update<true>(S, s_slot, s_run);
}

// ---------------------------------------------------------------------------
// Batched FP32 form (block-partial assembly): one tile, which is one block, of
// one instance per workgroup; per-instance parameters, compact FP32 plastic
// state (ping-pong by step parity).
// ---------------------------------------------------------------------------
// the {X, u} records of a tile's distinct nodes, built in LDS from the X and
// u arrays (FP32 instances keep u in the [3][ncap] array, BInst::urec = 0)
__device__ __forceinline__ void stage_tile_records(const BatchElemArgs &A, const BBlk &B,
                                                   double2 *s) {
  for (int k = threadIdx.x; k < B.count; k += blockDim.x) {
    const int64_t nd = A.bnode[B.off + k];
    s[3 * k] = make_double2(A.X[nd], A.X[A.ncap + nd]);
    s[3 * k + 1] = make_double2(A.X[2 * A.ncap + nd], A.u[nd]);
    s[3 * k + 2] = make_double2(A.u[A.ncap + nd], A.u[2 * A.ncap + nd]);
  }
}

// Batched FP32 Tet4 with block-partial assembly: each tile is one block of
// at most 256 consecutive elements of one instance, and each workgroup does
// one tile (a persistent loop over tiles measured 25% slower: a workgroup's
// staging, element and summing phases then ran one after another, their
// load latencies exposed).  The block's distinct
// node records are staged in LDS, the elements' corner forces go to LDS
// slots (the corners of one distinct node take consecutive slots in
// ascending element order), and one thread per distinct node adds its slots
// in that order (FP64, rounded once) and writes one table entry per (block,
// node).  The gather adds a node's partials in ascending block order.
template <int LAW>
__device__ __forceinline__ void batch_tet4_block(const BatchElemArgs &A, const BTile &T,
                                                 const BBlk &B, const BInst &P,
                                                 double2 *s_xu) { // [bmaxu][3] records,
                                                                  // later the corner slots
  float *fe = reinterpret_cast<float *>(A.fe);
  const QpCompact V = batch_compact_view(A, (P.parity_base ^ A.parity) & 1);
  // the element's own streams and this lane's first distinct node of the
  // summing phase, read ahead so that their loads overlap the staging (lanes
  // past the end read the last element's)
  const int t = threadIdx.x;
  const bool active = t < T.count;
  const int64_t e = T.first + (active ? t : T.count - 1);
  const ushort4 lc = *reinterpret_cast<const ushort4 *>(A.lc + e * 4);
  const ushort4 ls = *reinterpret_cast<const ushort4 *>(A.ls + e * 4);
  int s0_first = 0, s1_first = 0, pos_first = 0;
  if (t < B.count) {
    s0_first = t > 0 ? (int)A.bsend[B.off + t - 1] : 0;
    s1_first = A.bsend[B.off + t];
    pos_first = A.bpos[B.off + t];
  }
  stage_tile_records(A, B, s_xu);
  __syncthreads();
  float J[3][3], H[3][3];
  tet4_JH<float, akx::NodesLDS, false>(
      make_int4(lc.x, lc.y, lc.z, lc.w),
      akx::NodesLDS{reinterpret_cast<const double *>(s_xu)}, J, H);
  __syncthreads(); // the records are dead: the LDS now takes the slots
  float *s_f = reinterpret_cast<float *>(s_xu);
  if (active) {
    float Q[3][3];
    tet4_Q<LAW, float>(J, H, float(P.lambda), float(P.mu), float(P.sigma_y), float(P.h), V,
                       A.hoff + e, Q);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      s_f[3 * slot_pos(ls.x) + c] = -(Q[c][0] + Q[c][1] + Q[c][2]);
      s_f[3 * slot_pos(ls.y) + c] = Q[c][1];
      s_f[3 * slot_pos(ls.z) + c] = Q[c][2];
      s_f[3 * slot_pos(ls.w) + c] = Q[c][0];
    }
  }
  __syncthreads();
  for (int k = t; k < B.count; k += 256) {
    const bool first = k == t;
    const int s0 = first ? s0_first : (int)A.bsend[B.off + k - 1];
    const int s1 = first ? s1_first : (int)A.bsend[B.off + k];
    const int pos = first ? pos_first : A.bpos[B.off + k];
    sum_slots<true>(s_f, s0, s1, fe, (int64_t)pos);
  }
}

// Batched FP32 Hex8 with block-partial assembly: each tile is one block of at
// most BPA_HEX8 consecutive elements of one instance and each workgroup does
// one tile, as k_hex8_bpa.
template <int LAW>
__device__ __forceinline__ void batch_hex8_block(const BatchElemArgs &A, const BTile &T,
                                                 const BBlk &B, const BInst &P,
                                                 double2 *s_xu) { // [bmaxu][3] records, then
                                                                  // [63 * 8][3] floats
  float *s_f = reinterpret_cast<float *>(s_xu + 3 * A.bmaxu);
  const int t = threadIdx.x;
  const QpCompact V = batch_compact_view(A, (P.parity_base ^ A.parity) & 1);
  const bool active = (t >> 2) < T.count;
  const int64_t e = T.first + (t >> 2);
  uint32_t lc = 0, ls = 0;
  if (LAW != LAW_PLASTIC && active) {
    lc = reinterpret_cast<const uint32_t *>(A.lc + e * 8)[t & 3];
    ls = reinterpret_cast<const uint32_t *>(A.ls + e * 8)[t & 3];
  }
  int s0_first = 0, s1_first = 0, pos_first = 0;
  if (t < B.count) {
    s0_first = t > 0 ? (int)A.bsend[B.off + t - 1] : 0;
    s1_first = A.bsend[B.off + t];
    pos_first = A.bpos[B.off + t];
  }
  stage_tile_records(A, B, s_xu);
  __syncthreads();
  const akx::NodesLDS rec{reinterpret_cast<const double *>(s_xu)};
  if constexpr (LAW == LAW_PLASTIC)
    hex8_plastic_block(T.count, A.lc + T.first * 8, A.ls + T.first * 8, rec, V,
                       A.hoff + T.first * 8,
                       [&](int, float &l, float &m, float &y, float &h) {
                         l = float(P.lambda), m = float(P.mu), y = float(P.sigma_y), h = float(P.h);
                       },
                       s_f);
  else if (active)
    hex8_quad<LAW>(t & 3, lc, ls, rec, lame_quad(P.lambda, P.mu, t & 3), float(P.lambda),
                   float(P.mu), V, A.hoff + e * 8, s_f);
  __syncthreads();
  float *fe = reinterpret_cast<float *>(A.fe);
  for (int k = t; k < B.count; k += 256) {
    const bool first = k == t;
    const int s0 = first ? s0_first : (int)A.bsend[B.off + k - 1];
    const int s1 = first ? s1_first : (int)A.bsend[B.off + k];
    sum_slots<false>(s_f, s0, s1, fe, (int64_t)(first ? pos_first : A.bpos[B.off + k]));
  }
}

// one (element type, law) group
template <int ET, int LAW>
__global__ void __launch_bounds__(256) k_batch_bpa(BatchElemArgs A) {
  extern __shared__ double2 s_xu[];
  const int64_t tt = blockIdx.x;
  if (tt >= A.ntiles)
    return;
  const BTile T = A.tiles[tt];
  const BBlk B = A.blks[tt];
  const BInst P = A.inst[T.inst];
  if constexpr (ET == 0)
    batch_tet4_block<LAW>(A, T, B, P, s_xu);
  else
    batch_hex8_block<LAW>(A, T, B, P, s_xu);
}

// all groups of a batch: the Hex8 tiles H, then the Tet4 tiles A
__global__ void __launch_bounds__(256) k_batch_bpa_all(BatchElemArgs A, BatchElemArgs H) {
  extern __shared__ double2 s_xu[];
  const int64_t tt = blockIdx.x;
  if (tt >= H.ntiles + A.ntiles)
    return;
  if (tt < H.ntiles) {
    const BTile T = H.tiles[tt];
    const BBlk B = H.blks[tt];
    const BInst P = H.inst[T.inst];
    switch (P.law) {
    case LAW_ELASTIC: batch_hex8_block<LAW_ELASTIC>(H, T, B, P, s_xu); break;
    case LAW_ELASTIC_FD: batch_hex8_block<LAW_ELASTIC_FD>(H, T, B, P, s_xu); break;
    case LAW_NEOHOOKEAN: batch_hex8_block<LAW_NEOHOOKEAN>(H, T, B, P, s_xu); break;
    default: batch_hex8_block<LAW_PLASTIC>(H, T, B, P, s_xu); break;
    }
  } else {
    const BTile T = A.tiles[tt - H.ntiles];
    const BBlk B = A.blks[tt - H.ntiles];
    const BInst P = A.inst[T.inst];
    switch (P.law) {
    case LAW_ELASTIC: batch_tet4_block<LAW_ELASTIC>(A, T, B, P, s_xu); break;
    case LAW_ELASTIC_FD: batch_tet4_block<LAW_ELASTIC_FD>(A, T, B, P, s_xu); break;
    case LAW_NEOHOOKEAN: batch_tet4_block<LAW_NEOHOOKEAN>(A, T, B, P, s_xu); break;
    default: batch_tet4_block<LAW_PLASTIC>(A, T, B, P, s_xu); break;
    }
  }
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
hipError_t upload_hex8_dnds(const double *dnds) {
  return hipMemcpyToSymbol(HIP_SYMBOL(c_dnds), dnds, sizeof(double) * 192);
}

int64_t elements_per_block(int etype, bool bpa) {
  return etype == 1 ? (bpa ? akx::BPA_HEX8 : HEX_EPB) : 256;
}

// LDS of the FP32 Tet4 block passes: the records, later 1024 corner slots
static size_t tet4_bpa_lds(int32_t maxu) {
  return std::max((size_t)maxu * 48, (size_t)slot_pos(1024) * 12);
}

template <int L, class CT, class FT>
static void launch_one(int etype, const ElemArgs &A, hipStream_t s) {
  dim3 grid((unsigned)A.nblocks_padded), block(256);
  if (etype != 1) {
    if constexpr (sizeof(CT) == 4)
      if (A.lconn) {
        if (A.lslot) // block-partial assembly
          hipLaunchKernelGGL((k_tet4_bpa<L>), grid, block,
                             tet4_bpa_lds(A.bl_maxu), s, A);
        else
          hipLaunchKernelGGL((k_tet4_lds<L>), grid, block, (size_t)A.bl_maxu * 48, s, A);
        return;
      }
    hipLaunchKernelGGL((k_tet4_fast<L, CT, FT>), grid, block, 0, s, A);
  }
  else if constexpr (sizeof(CT) == 4) { // FP32: sum-factorised Hex8
    if (A.lslot) // block-partial assembly
      hipLaunchKernelGGL((A.grad_u ? k_hex8_bpa<L, true> : k_hex8_bpa<L, false>), grid, block,
                         (size_t)A.bl_maxu * 48 + akx::BPA_HEX8 * 8 * 12, s, A);
    else
      hipLaunchKernelGGL((k_hex8_sf<L, FT>), grid, block, 0, s, A);
  }
  else
    hipLaunchKernelGGL((k_hex8_fast<L, CT, FT>), grid, block, 0, s, A);
}

template <class CT, class FT>
static hipError_t launch_t(int etype, int law, ElemArgs A, hipStream_t s) {
  switch (law) {
  case LAW_ELASTIC: launch_one<LAW_ELASTIC, CT, FT>(etype, A, s); break;
  case LAW_ELASTIC_FD: launch_one<LAW_ELASTIC_FD, CT, FT>(etype, A, s); break;
  case LAW_NEOHOOKEAN: launch_one<LAW_NEOHOOKEAN, CT, FT>(etype, A, s); break;
  case LAW_PLASTIC: launch_one<LAW_PLASTIC, CT, FT>(etype, A, s); break;
  default:
    return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_elements(int etype, int law, bool fp32, const ElemArgs &A,
                           hipStream_t stream) {
  return fp32 ? launch_t<float, float>(etype, law, A, stream)
              : launch_t<double, double>(etype, law, A, stream);
}

template <int LAW>
static void launch_step_law(int etype, const akx::StepArgs &S, size_t lds, hipStream_t s) {
  const dim3 grid((unsigned)S.nblocks_padded);
  const int lanes = (etype == 0 ? 1 : 4) * S.max_elems;
  const dim3 block((unsigned)(lanes + 63) / 64 * 64);
  if (etype == 0)
    hipLaunchKernelGGL(k_tet4_step_f32<LAW>, grid, block, lds, s, S);
  else
    hipLaunchKernelGGL(k_hex8_step_f32<LAW>, grid, block, lds, s, S);
}

hipError_t launch_step(int etype, int law, const akx::StepArgs &S, size_t lds, hipStream_t stream) {
  switch (law) {
  case LAW_ELASTIC: launch_step_law<LAW_ELASTIC>(etype, S, lds, stream); break;
  case LAW_ELASTIC_FD: launch_step_law<LAW_ELASTIC_FD>(etype, S, lds, stream); break;
  case LAW_NEOHOOKEAN: launch_step_law<LAW_NEOHOOKEAN>(etype, S, lds, stream); break;
  default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

static size_t hex8_bpa_lds(int32_t maxu) {
  return (size_t)maxu * 48 + akx::BPA_HEX8 * 8 * 12;
}

template <int LAW> static void launch_batch_law(int etype, const BatchElemArgs &A, hipStream_t s) {
  const dim3 grid((unsigned)A.ntiles), block(256);
  if (etype == 0)
    hipLaunchKernelGGL((k_batch_bpa<0, LAW>), grid, block, tet4_bpa_lds(A.bmaxu), s, A);
  else
    hipLaunchKernelGGL((k_batch_bpa<1, LAW>), grid, block, hex8_bpa_lds(A.bmaxu), s, A);
}

hipError_t launch_batch_elements_f32(int etype, int law, const BatchElemArgs &A,
                                     hipStream_t stream) {
  switch (law) {
  case LAW_ELASTIC: launch_batch_law<LAW_ELASTIC>(etype, A, stream); break;
  case LAW_ELASTIC_FD: launch_batch_law<LAW_ELASTIC_FD>(etype, A, stream); break;
  case LAW_NEOHOOKEAN: launch_batch_law<LAW_NEOHOOKEAN>(etype, A, stream); break;
  case LAW_PLASTIC: launch_batch_law<LAW_PLASTIC>(etype, A, stream); break;
  default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_batch_all_f32(const BatchElemArgs &tets, const BatchElemArgs &hexes,
                                hipStream_t stream) {
  const size_t lds = std::max(tets.ntiles > 0 ? tet4_bpa_lds(tets.bmaxu) : 0,
                              hexes.ntiles > 0 ? hex8_bpa_lds(hexes.bmaxu) : 0);
  hipLaunchKernelGGL(k_batch_bpa_all, dim3((unsigned)(tets.ntiles + hexes.ntiles)), dim3(256), lds,
                     stream, tets, hexes);
  return hipGetLastError();
}

} // namespace akxf
