// akx_model.hip -- host runtime and C ABI of the MI355X explicit internal
// force path (declared in include/akantu_mi355x.h).
//
// One akx_model = one SolidMechanicsModel on one device and one stream
// (default priority).  The per-step work is two launches:
//   element pass (one kernel per material)  ->  nodal gather + update
// with the predictor of step k+1 fused into the gather of step k when
// several steps are queued together; small models take one launch per step
// (plan_small_steps).
#include "../../include/akantu_mi355x.h"
#include "akx_download.hpp"
#include "akx_fast.hpp"
#include "akx_host.hpp"
#include "akx_kernels.hpp"
#include "akx_step.hpp"

#include <hip/hip_runtime.h>
#include <hip/hiprtc.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <memory>
#include <mutex>
#include <stdexcept>
#include <string>
#include <vector>

namespace akx {

__constant__ Hex8Tables c_hex8;

thread_local std::string g_last_error;

// ---------------------------------------------------------------------------
// One step of a small FP64 model (akx_step.hpp).
// ---------------------------------------------------------------------------

// A view whose previous history of one Gauss point is in registers, read ahead
// of the staging (step of 4,032 nodes 10.6 -> 10.3 us; the two-launch pass keeps
// reading it inside the law: its 330,000-element pass went from 34.7 to 37.7)
struct QpHeld : QpView {
  double pg[3][3], ps[3][3], pe[3][3], iso, work;
  __device__ __forceinline__ void read(int64_t iq) {
    QpView::history(iq, pg, ps, pe, iso);
    work = p_pe ? p_pe[iq] : 0.;
  }
  __device__ __forceinline__ double energy(int64_t) const { return work; }
  __device__ __forceinline__ void history(int64_t, double (&g)[3][3], double (&s)[3][3],
                                          double (&e)[3][3], double &k) const {
#pragma unroll
    for (int ii = 0; ii < 3; ++ii)
#pragma unroll
      for (int jj = 0; jj < 3; ++jj) {
        g[ii][jj] = pg[ii][jj];
        s[ii][jj] = ps[ii][jj];
        e[ii][jj] = pe[ii][jj];
      }
    k = iso;
  }
};

template <int LAW> struct QpAhead {
  using type = QpView;
};
template <> struct QpAhead<LAW_PLASTIC> {
  using type = QpHeld;
};

// Tet4: one lane per element of the workgroup's list
template <int LAW>
__global__ void __launch_bounds__(256) k_tet4_step(StepArgs S) {
  extern __shared__ double2 s_rec[]; // records, then slots
  const int64_t b = xcd_block(S.nblocks_padded);
  if (b >= S.nblocks) // padding block
    return;
  const int t = threadIdx.x;
  double *s_slot = reinterpret_cast<double *>(s_rec + 3 * S.max_nodes);
  const bool active = t < S.max_elems;
  const int64_t i = b * S.max_elems + (active ? t : S.max_elems - 1);
  const ushort4 lc = *reinterpret_cast<const ushort4 *>(S.lc + i * 4);
  const ushort4 ls = *reinterpret_cast<const ushort4 *>(S.ls + i * 4);
  const int32_t le = S.lelem[i], e = le & ~STEP_GUEST;
  double lambda = S.lambda, mu = S.mu, sy = S.sigma_y, hh = S.h;
  if (S.lam_el) {
    lambda = S.lam_el[e];
    mu = S.mu_el[e];
  }
  typename QpAhead<LAW>::type V{};
  if constexpr (LAW == LAW_PLASTIC) {
    static_cast<QpView &>(V) = S.hist;
    V.keep = le >= 0;
    V.read(e);
    if (S.sy_el)
      sy = S.sy_el[e];
    if (S.h_el)
      hh = S.h_el[e];
  }
  StepDof<false> dof;
  dof.load(S, b);
  step_stage<false>(S, b, s_rec);
  __syncthreads();
  if (active) {
    const int4 nd = make_int4(lc.x, lc.y, lc.z, lc.w);
    const int4 slots = make_int4(-1 - ls.x, -1 - ls.y, -1 - ls.z, -1 - ls.w);
    element_forces_one<ET_TET4, LAW, double, double, double, NodesLDS, 3, false, true>(
        reinterpret_cast<const int32_t *>(&nd),
        NodesLDS{reinterpret_cast<const double *>(s_rec)}, lambda, mu, sy, hh, V, e,
        reinterpret_cast<const int32_t *>(&slots), s_slot, s_slot);
  }
  __syncthreads();
  dof.update<false>(S, s_slot, nullptr);
}

// hex8_strict_group's results to the slots of the element's corners
struct PutSlots {
  const uint16_t *ls; // LDS, the element's 8 corners
  double *s_slot;
  __device__ __forceinline__ void operator()(int n, int c, double s) const {
    s_slot[3 * ls[n] + c] = s;
  }
};

// Hex8: eight lanes per element, STEP_HEX_EPB elements at a time
constexpr int STEP_HEX_EPB = 32;
template <int LAW> __global__ void __launch_bounds__(STEP_HEX_EPB * 8) k_hex8_step(StepArgs S) {
  extern __shared__ double2 s_rec[]; // records, then slots
  __shared__ double sN[STEP_HEX_EPB][8][6];
  __shared__ double sD[8][3][8];
  __shared__ uint16_t s_ls[STEP_HEX_EPB][8];
  const int64_t b = xcd_block(S.nblocks_padded);
  if (b >= S.nblocks) // padding block
    return;
  const int t = threadIdx.x, el = t >> 3, q = t & 7;
  double *s_slot = reinterpret_cast<double *>(s_rec + 3 * S.max_nodes);
  StepDof<false> dof;
  dof.load(S, b);
  for (int base = 0; base < S.max_elems; base += STEP_HEX_EPB) {
    const bool active = base + el < S.max_elems;
    const int64_t i = b * S.max_elems + (active ? base + el : S.max_elems - 1);
    const int32_t e = S.lelem[i] & ~STEP_GUEST;
    const int32_t nd = S.lc[i * 8 + q];
    double lambda = S.lambda, mu = S.mu;
    if (S.lam_el) {
      lambda = S.lam_el[e];
      mu = S.mu_el[e];
    }
    s_ls[el][q] = S.ls[i * 8 + q];
    HexJac pre;
    pre.load<false>(S.jw + (int64_t)e * 8 + q, S.nel * 8);
    if (base == 0) {
      step_stage<false>(S, b, s_rec);
      for (int k = t; k < 192; k += STEP_HEX_EPB * 8)
        (&sD[0][0][0])[k] = (&c_hex8.dnds[0][0][0])[k];
      __syncthreads();
    }
    hex8_strict_group<LAW, STEP_HEX_EPB, double, NodesLDS, true>(
        sN, sD, c_hex8.w[q], el, q, active, nd,
        NodesLDS{reinterpret_cast<const double *>(s_rec)}, lambda, mu, 0., 0., QpView{}, 0,
        PutSlots{s_ls[el], s_slot}, pre);
  }
  dof.update<false>(S, s_slot, nullptr); // the group's last barrier is behind
}

// The lists of StepArgs, one workgroup per workgroup of the step, from what
// group_nodes found: owner, slot0 and rank give a node's workgroup, its first
// slot and a corner's place among its node's; ends the partial sums' ends in
// the order of `first`.
struct StepListArgs {
  int32_t *lnode, *onode, *lelem;
  uint16_t *lc, *ls, *send;
  uint8_t *run; // FP32 form, else null
  const int32_t *ooff, *onodes, *eoff, *elems, *noff, *nodes, *owner, *slot0, *first;
  const uint16_t *lcs;
  const uint8_t *rank, *ends;
  const int32_t *conn;
  int32_t nnpe;
};

__global__ void __launch_bounds__(256) k_step_lists(StepArgs S, StepListArgs L) {
  const int64_t b = blockIdx.x;
  const int e0 = L.eoff[b], ne = L.eoff[b + 1] - e0;
  for (int k = threadIdx.x; k < S.max_elems; k += blockDim.x) {
    // padding: the list's first element again (an empty list: element 0 of the
    // mesh on the records of no node), to the slot nothing reads
    const int src = e0 + (k < ne ? k : 0);
    const int32_t e = ne > 0 ? L.elems[src] : 0;
    const int32_t *c = L.conn + (int64_t)e * L.nnpe;
    const int64_t at = b * S.max_elems + k;
    // an element's history is written where its first node is owned
    L.lelem[at] = k < ne && L.owner[c[0]] == b ? e : e | STEP_GUEST;
    for (int a = 0; a < L.nnpe; ++a) {
      L.lc[at * L.nnpe + a] = ne > 0 ? L.lcs[(int64_t)src * L.nnpe + a] : 0;
      L.ls[at * L.nnpe + a] =
          (uint16_t)(k < ne && L.owner[c[a]] == b
                         ? L.slot0[c[a]] + L.rank[(int64_t)e * L.nnpe + a]
                         : S.max_slots);
    }
  }
  const int n0 = L.noff[b], nb_nodes = L.noff[b + 1] - n0;
  for (int k = threadIdx.x; k < S.max_nodes; k += blockDim.x)
    L.lnode[b * S.max_nodes + k] = k < nb_nodes ? L.nodes[n0 + k] : -1;
  const int o0 = L.ooff[b], nb_own = L.ooff[b + 1] - o0;
  for (int k = threadIdx.x; k < S.own; k += blockDim.x) {
    const int32_t n = k < nb_own ? L.onodes[o0 + k] : -1;
    L.onode[b * S.own + k] = n;
    const int deg = n < 0 ? 0 : L.first[n + 1] - L.first[n];
    L.send[b * S.own + k] = (uint16_t)(n < 0 ? 0 : L.slot0[n] + deg);
    if (L.run)
      for (int d = 0; d < deg; ++d)
        L.run[b * S.max_slots + L.slot0[n] + d] = L.ends[L.first[n] + d];
  }
}

// ---------------------------------------------------------------------------
// Layout kernels (array-of-structures at the API, structure-of-arrays on the
// device)
// ---------------------------------------------------------------------------
template <class T>
__global__ void k_aos_to_soa(const T *aos, T *soa, int64_t n, int comps) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n * comps)
    return;
  int64_t r = i / comps, c = i % comps;
  soa[c * n + r] = aos[i];
}

// rows first .. first + count - 1 of the n
template <class T>
__global__ void k_soa_to_aos(const T *soa, T *aos, int64_t n, int comps, int64_t first,
                             int64_t count) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count * comps)
    return;
  int64_t r = i / comps, c = i % comps;
  aos[i] = soa[c * n + first + r];
}

__global__ void k_bits_from_bool3(const uint8_t *b3, uint8_t *bits, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n)
    return;
  bits[i] = (b3[3 * i] ? 1 : 0) | (b3[3 * i + 1] ? 2 : 0) | (b3[3 * i + 2] ? 4 : 0);
}

__global__ void k_bool3_from_bits(const uint8_t *bits, uint8_t *b3, int64_t first,
                                  int64_t count) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count)
    return;
  uint8_t b = bits[first + i];
  b3[3 * i] = b & 1;
  b3[3 * i + 1] = (b >> 1) & 1;
  b3[3 * i + 2] = (b >> 2) & 1;
}

__global__ void k_mass_to3(const double *m, double *m3, int64_t first, int64_t count) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count)
    return;
  const double v = m[first + i];
  m3[3 * i] = v;
  m3[3 * i + 1] = v;
  m3[3 * i + 2] = v;
}

// streaming copy used to calibrate the HBM byte counters and to report the
// measured copy bandwidth next to the 8 TB/s peak
// (two 32-byte items per thread, both loads issued before the stores: the
// fastest plain copy shape measured on MI355X)
__global__ void __launch_bounds__(256) k_copy_calibration(const double4 *src,
                                                          double4 *dst,
                                                          int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 512 + threadIdx.x;
  double4 v0, v1;
  if (i < n)
    v0 = src[i];
  if (i + 256 < n)
    v1 = src[i + 256];
  if (i < n)
    dst[i] = v0;
  if (i + 256 < n)
    dst[i + 256] = v1;
}

__global__ void k_fill_f32(float *p, int64_t n, float v) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n)
    p[i] = v;
}
__global__ void k_fill_f64(double *p, int64_t n, double v) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n)
    p[i] = v;
}

// FP32 copies of the per-element Lame constants (the FP32 form's reads)
__global__ void k_lame_f32(const double *lam, const double *mu, float2 *lm, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n)
    lm[i] = make_float2(float(lam[i]), float(mu[i]));
}

// Lame constants per element from E, nu (material_elastic.cc:53-62)
__global__ void k_lame(const double *E, const double *nu, double E0, double nu0,
                       double *lam, double *mu, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n)
    return;
  double l, m;
  lame(E ? E[i] : E0, nu ? nu[i] : nu0, l, m);
  lam[i] = l;
  mu[i] = m;
}

// ---------------------------------------------------------------------------
// Init kernels: jacobian check, lumped mass, stable time step
// ---------------------------------------------------------------------------
struct InitArgs {
  int64_t n, nel, first, pos_offset, nn;
  const int32_t *filter, *conn;
  const double *X, *u;
  double rho;
  double lambda, mu;
  const double *lam_el, *mu_el;
  const int32_t *pos; // [slot] entry of the node-major table
  double *me;         // [entry] mass contributions
  unsigned long long *min_bits;
  long long *first_bad;
};

template <int ET>
__device__ __forceinline__ void load_element_X(const InitArgs &A, int64_t e,
                                               bool add_u,
                                               double (&X)[Elem<ET>::nnpe][3]) {
#pragma unroll
  for (int n = 0; n < Elem<ET>::nnpe; ++n) {
    int32_t node = A.conn[e * Elem<ET>::nnpe + n];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      double x = A.X[(int64_t)c * A.nn + node];
      X[n][c] = add_u ? x + A.u[(int64_t)c * A.nn + node] : x;
    }
  }
}

// IntegratorGauss::checkJacobians over every element of the mesh
template <int ET> __global__ void k_check_jacobians(InitArgs A) {
  constexpr int NN = Elem<ET>::nnpe, NQ = Elem<ET>::nqp;
  int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= A.nel)
    return;
  double X[NN][3];
  load_element_X<ET>(A, e, false, X);
  for (int q = 0; q < NQ; ++q) {
    double Ji[3][3], detJ;
    Shape<ET, double>::jacobian_at(X, q, Ji, detJ);
    if (detJ < 0.) {
      atomicMin(A.first_bad, (long long)(e * NQ + q));
      return;
    }
  }
}

// J^-1 and w det J of every Hex8 Gauss point of the mesh, one thread per
// Gauss point, in the arithmetic of the element pass (Shape::jacobian_at:
// J = dN/dxi X summed over the nodes in order, the LU inverse, det J * w).
__global__ void __launch_bounds__(256) k_hex8_jacobian_table(const int32_t *conn,
                                                             const double *X, int64_t nn,
                                                             int64_t nel, double2 *jw) {
  const int64_t iq = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t nq = nel * 8;
  if (iq >= nq)
    return;
  const int64_t e = iq >> 3;
  const int q = (int)(iq & 7);
  double Xe[8][3];
#pragma unroll
  for (int n = 0; n < 8; ++n) {
    const int32_t nd = conn[e * 8 + n];
#pragma unroll
    for (int c = 0; c < 3; ++c)
      Xe[n][c] = X[(int64_t)c * nn + nd];
  }
  double Ji[3][3], detJ;
  const double wJ = Shape<ET_HEX8, double>::jacobian_at(Xe, q, Ji, detJ);
  jw[iq] = make_double2(Ji[0][0], Ji[0][1]);
  jw[nq + iq] = make_double2(Ji[0][2], Ji[1][0]);
  jw[2 * nq + iq] = make_double2(Ji[1][1], Ji[1][2]);
  jw[3 * nq + iq] = make_double2(Ji[2][0], Ji[2][1]);
  jw[4 * nq + iq] = make_double2(Ji[2][2], wJ);
}

// {X, u} node records of the Tet4 element pass from the [3][nn] arrays:
// u only (refresh after an upload of u) or X and u (init)
__global__ void __launch_bounds__(256) k_fill_xu(const double *X, const double *u, int64_t nn,
                                                 double *xu, bool with_x) {
  const int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= nn)
    return;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    if (with_x)
      xu[6 * n + c] = X[(int64_t)c * nn + n];
    xu[6 * n + 3 + c] = u[(int64_t)c * nn + n];
  }
}

// Lumped mass contributions m_e(a) = sum_q (rho N_a(q)) wJ_q
// (fe_engine_template_tmpl_field.hh:112-138)
template <int ET> __global__ void k_mass_elements(InitArgs A) {
  constexpr int NN = Elem<ET>::nnpe, NQ = Elem<ET>::nqp;
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= A.n)
    return;
  int64_t e = A.filter ? (int64_t)A.filter[i] : A.first + i;
  double X[NN][3];
  load_element_X<ET>(A, e, false, X);
  double m[NN];
#pragma unroll
  for (int n = 0; n < NN; ++n)
    m[n] = 0.;
  for (int q = 0; q < NQ; ++q) {
    double Ji[3][3], detJ;
    double wJ = Shape<ET, double>::jacobian_at(X, q, Ji, detJ);
#pragma unroll
    for (int n = 0; n < NN; ++n) {
      double N = (ET == ET_TET4) ? .25 : c_hex8.N[q][n];
      m[n] += (A.rho * N) * wJ;
    }
  }
#pragma unroll
  for (int n = 0; n < NN; ++n)
    A.me[A.pos[(A.pos_offset + i) * NN + n]] = m[n];
}

// min_e h_e / c_e over one material (solid_mechanics_model.cc:423-473)
template <int ET> __global__ void __launch_bounds__(256) k_stable_dt(InitArgs A) {
  constexpr int NN = Elem<ET>::nnpe;
  __shared__ double red[256];
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  double dt = 1.7976931348623157e308;
  if (i < A.n) {
    int64_t e = A.filter ? (int64_t)A.filter[i] : A.first + i;
    double X[NN][3];
    load_element_X<ET>(A, e, true, X);
    double lambda = A.lam_el ? A.lam_el[i] : A.lambda;
    double mu = A.mu_el ? A.mu_el[i] : A.mu;
    double h = inradius<ET>(X);
    double c = sqrt((lambda + 2 * mu) / A.rho);
    dt = h / c;
  }
  red[threadIdx.x] = dt;
  __syncthreads();
  for (int s = blockDim.x / 2; s > 0; s >>= 1) {
    if (threadIdx.x < s)
      red[threadIdx.x] = fmin(red[threadIdx.x], red[threadIdx.x + s]);
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    // positive doubles order like their bit patterns
    atomicMin(A.min_bits, (unsigned long long)__double_as_longlong(red[0]));
  }
}

// Lumped mass gather: M = 0 + sum 1 * m_e over the node's entries in order
__global__ void k_gather_mass(int64_t nn, const int64_t *ell_off,
                              const uint8_t *deg, const double *me,
                              double *mass) {
  int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= nn)
    return;
  double m = 0.;
  const double *p = me + ell_off[n >> 8] + (n & 255);
  for (int d = 0; d < deg[n]; ++d)
    m += 1. * p[d * 256];
  mass[n] = m;
}

// ---------------------------------------------------------------------------
// Energies (solid_mechanics_model.cc:476-606, material.cc:604-649,
// material_plastic.cc:47-99).  Per-node or per-element values, then one
// deterministic tree sum (fixed shape, so repeated calls give the same bits).
// ---------------------------------------------------------------------------
template <class R> __device__ __forceinline__ R ddot3(const R (&a)[3][3], const R (&b)[3][3]) {
  R s = a[0][0] * b[0][0]; // cwiseProduct().sum(), column-major order
#pragma unroll
  for (int j = 0; j < 3; ++j)
#pragma unroll
    for (int i = 0; i < 3; ++i)
      if (i + j > 0)
        s += a[i][j] * b[i][j];
  return s;
}

// Potential energy density of one Gauss point:
//   elastic          .5 sigma : grad u  (material_elastic_inline_impl.hh:113-116)
//   elastic finite   .5 S : E(grad u)   (material_elastic.cc:138-160)
//   neo-Hookean      lambda (ln J)^2 + mu (-ln J + (tr C - 3) / 2) / 2, as the
//                    reference writes it (material_neohookean_inline_impl.hh
//                    :119-126)
//   plastic          .5 sigma : (grad u - eps_p)  (material_plastic.cc:71-83)
template <int LAW>
__device__ __forceinline__ double epot_density(double lambda, double mu,
                                               const double (&g)[3][3],
                                               const double (&S)[3][3],
                                               const double (&ep)[3][3]) {
  if constexpr (LAW == LAW_ELASTIC) {
    return .5 * ddot3(S, g);
  } else if constexpr (LAW == LAW_ELASTIC_FD) {
    double E[3][3];
    green_strain(g, E);
    return .5 * ddot3(S, E);
  } else if constexpr (LAW == LAW_NEOHOOKEAN) {
    double F[3][3], C[3][3];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int j = 0; j < 3; ++j)
        F[i][j] = (i == j) ? 1. + g[i][j] : g[i][j];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        double c = F[0][i] * F[0][j];
        c += F[1][i] * F[1][j];
        c += F[2][i] * F[2][j];
        C[i][j] = c;
      }
    const double lj = log(det3(F));
    const double trC = C[0][0] + C[1][1] + C[2][2];
    return lambda * (lj * lj) + mu * (-lj + (trC - 3) / 2.) / 2.;
  } else {
    double el[3][3];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int j = 0; j < 3; ++j)
        el[i][j] = g[i][j] - ep[i][j];
    return .5 * ddot3(S, el);
  }
}

struct EnergyArgs {
  int64_t n, first, nn, nq_all;
  const int32_t *filter, *conn;
  const double *X;
  double lambda, mu;
  const double *lam_el, *mu_el;
  const double *g, *s, *eps; // [9][nq_all] current grad u, stress, plastic strain
  const double *pe;          // [nq_all] accumulated plastic energy, or null
  double *out;               // [n] integral over each element
};

// FEEngine::integrate of the density: sum_q f_q wJ_q of the i-th element of
// the material (integrator_gauss_inline_impl.hh:401-441), wJ as at init
template <int ET, int LAW>
__device__ __forceinline__ double element_energy(const EnergyArgs &A, int64_t i) {
  constexpr int NN = Elem<ET>::nnpe, NQ = Elem<ET>::nqp;
  const int64_t e = A.filter ? (int64_t)A.filter[i] : A.first + i;
  double X[NN][3];
#pragma unroll
  for (int n = 0; n < NN; ++n) {
    const int32_t node = A.conn[e * NN + n];
#pragma unroll
    for (int c = 0; c < 3; ++c)
      X[n][c] = A.X[(int64_t)c * A.nn + node];
  }
  const double lambda = A.lam_el ? A.lam_el[i] : A.lambda;
  const double mu = A.mu_el ? A.mu_el[i] : A.mu;
  double sum = 0.;
  for (int q = 0; q < NQ; ++q) {
    double Ji[3][3], detJ;
    const double wJ = Shape<ET, double>::jacobian_at(X, q, Ji, detJ);
    const int64_t iq = i * NQ + q;
    double f;
    if (A.pe) {
      f = A.pe[iq];
    } else {
      double g[3][3], S[3][3], ep[3][3];
#pragma unroll
      for (int jj = 0; jj < 3; ++jj)
#pragma unroll
        for (int ii = 0; ii < 3; ++ii) {
          const int64_t o = (int64_t)(ii + 3 * jj) * A.nq_all + iq;
          g[ii][jj] = A.g[o];
          S[ii][jj] = A.s[o];
          ep[ii][jj] = A.eps ? A.eps[o] : 0.;
        }
      f = epot_density<LAW>(lambda, mu, g, S, ep);
    }
    sum = (q == 0) ? f * wJ : sum + f * wJ;
  }
  return sum;
}

template <int ET, int LAW> __global__ void k_energy_elements(EnergyArgs A) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= A.n)
    return;
  A.out[i] = element_energy<ET, LAW>(A, i);
}

// kinetic energy per node: sum_i v_i v_i m (m > epsilon) (solid_mechanics_model
// .cc:476-522); external work per node: blocked ? -f_int v : f_ext v
// (solid_mechanics_model.cc:545-583)
struct NodeEnergyArgs {
  int64_t nn;
  int kind; // 0 kinetic, 1 external work
  const double *v, *mass, *fint, *fext;
  const uint8_t *blocked;
};

__device__ __forceinline__ double node_energy(const NodeEnergyArgs &A, int64_t n) {
  double w = 0.;
  for (int c = 0; c < 3; ++c) {
    const int64_t o = (int64_t)c * A.nn + n;
    if (A.kind == 0) {
      const double m = A.mass[n];
      if (m > 2.220446049250313e-16)
        w += A.v[o] * A.v[o] * m;
    } else if ((A.blocked[n] >> c) & 1) {
      w -= A.fint[o] * A.v[o];
    } else {
      w += (A.fext ? A.fext[o] : 0.) * A.v[o];
    }
  }
  return w;
}

__global__ void k_node_energy(NodeEnergyArgs A, double *out) {
  const int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= A.nn)
    return;
  out[n] = node_energy(A, n);
}

// One level of the tree sum: block b sums the values of items b*2048 ..
// b*2048+2047, thread t first adding items t, t+256, .., t+1792 in that order
// from 0, then the 256 thread sums pairwise in shared memory.  value(i) reads
// a stored value or computes it in place; both give the same bits.
template <class F>
__device__ __forceinline__ void block_tree_sum(int64_t n, double *out, F &&value) {
  __shared__ double red[256];
  const int64_t base = (int64_t)blockIdx.x * 2048;
  double s = 0.;
  for (int k = 0; k < 8; ++k) {
    const int64_t i = base + threadIdx.x + 256 * k;
    if (i < n)
      s += value(i);
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w)
      red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0)
    out[blockIdx.x] = red[0];
}

__global__ void __launch_bounds__(256) k_tree_sum(const double *in, int64_t n, double *out) {
  block_tree_sum(n, out, [&](int64_t i) { return in[i]; });
}

// First tree level fused with the per-node / per-element values (the
// no-allocation energy): the same sums as k_node_energy / k_energy_elements
// followed by k_tree_sum, without the [n] array of values.
__global__ void __launch_bounds__(256) k_node_energy_sum(NodeEnergyArgs A, double *out) {
  block_tree_sum(A.nn, out, [&](int64_t n) { return node_energy(A, n); });
}

template <int ET, int LAW>
__global__ void __launch_bounds__(256) k_energy_elements_sum(EnergyArgs A, double *out) {
  block_tree_sum(A.n, out, [&](int64_t i) { return element_energy<ET, LAW>(A, i); });
}

} // namespace akx

using namespace akx;

// ---------------------------------------------------------------------------
// Model
// ---------------------------------------------------------------------------
// A user law compiled at run time into the material's element pass
// (akx_model_set_device_stress): the pass without and with the eigen-gradient
// terms
struct DeviceLaw {
  hipModule_t module = nullptr;
  hipFunction_t kernel[2] = {nullptr, nullptr};
  DeviceLaw() = default;
  DeviceLaw(const DeviceLaw &) = delete;
  DeviceLaw &operator=(const DeviceLaw &) = delete;
  ~DeviceLaw() {
    if (module)
      (void)hipModuleUnload(module);
  }
};

struct Material {
  int law = 0;
  double rho = 0, E = 0, nu = 0, sigma_y = 0, h = 0;
  double lambda = 0, mu = 0;
  int64_t n = 0;          // elements in the filter
  bool contiguous = true; // filter == first..first+n-1
  int64_t first = 0;
  int64_t pos_offset = 0; // assembly position of its first element
  std::vector<int32_t> filter_host;
  DevBuf<int32_t> filter;
  DevBuf<double> lam_el, mu_el, sy_el, h_el;
  DevBuf<float2> lm_f; // FP32 form: (float(lambda), float(mu)) per element
  // FP32 Tet4: distinct nodes of each 256-element block and local corners
  DevBuf<int32_t> bl_nodes;
  DevBuf<uint16_t> lconn;
  int32_t bl_maxu = 0;
  std::vector<int32_t> bl_nodes_host; // [blocks][bl_maxu], -1 padded
  // block-partial assembly (FP32 Tet4): LDS slot of every corner, slot
  // offsets of every distinct node, table entry of every (block, node) partial
  DevBuf<uint16_t> lslot, bl_soff;
  DevBuf<int32_t> bl_pos;
  // partial-sum assembly of the FP64 Tet4 pass: per-corner codes, per-block
  // summed runs (slot ends, table entries)
  DevBuf<int32_t> pcode, poff, ppos;
  DevBuf<uint16_t> pend;
  int64_t t_nblk = 0;
  int32_t t_slots = 0;
  bool per_element = false;
  // materialised internals and plastic history [2][9][n*nqp] / [2][n*nqp]
  DevBuf<double> grad, stress; // materialised by compute_all_stresses
  DevBuf<double> hgrad[2], hsig[2], heps[2], hiso[2];
  DevBuf<double> hpe[2]; // accumulated plastic energy [n*nqp]
  int cur = 0; // index of the current plastic state
  // Material::eigengradu [9][n*nqp] (null: zero); MaterialThermal's sigma_th
  // [n*nqp] (null: -0) and, for the plastic law, its history [2][n*nqp]
  DevBuf<double> eig, sth_now, hsth[2];
  std::vector<double> E_el_host, nu_el_host; // per-element E, nu as given
  bool ext() const { return eig.p != nullptr || sth_now.p != nullptr; }
  // a law computed by the caller (the computeStress plugin)
  bool user() const { return law == AKX_LAW_USER || law == AKX_LAW_USER_FD; }
  // the caller's law compiled for the device, or null (host callback)
  std::unique_ptr<DeviceLaw> dlaw;
};

// meshes of up to this many nodes hold u, v and a twice
constexpr int64_t STEP_NODES_MAX = 12288;
// doubles or floats from one [3][nn] array of the state to the next
inline int64_t state_stride(int64_t nn) { return (3 * nn + 31) / 32 * 32; }

struct akx_model {
  int device = 0;
  hipStream_t stream = nullptr;
  int etype = -1, nnpe = 0, nqp = 0;
  int64_t nn = 0, nel = 0;
  int precision = AKX_PRECISION_FP64;
  bool initialized = false;
  bool has_fext = false;
  double dt = 0.;
  std::vector<int32_t> conn_host; // AoS copy for filters and the gather table
  DevBuf<double> X, fint, fext, mass;
  // u, v, a and the FP32 form's compensation terms, each [3][nn], with the
  // second ones of meshes small enough for single-launch steps
  template <class T> struct Part {
    T *p = nullptr;
  };
  DevBuf<double> state;
  DevBuf<float> comp;
  Part<double> u, v, a, u2, v2, a2;
  Part<float> cu, cv, cu2, cv2;
  DevBuf<uint8_t> blocked;
  DevBuf<int32_t> conn, pos;
  DevBuf<double2> jw;      // Hex8 plain FP64: J^-1, w det J [5][nel * 8]
  DevBuf<double> xu;       // Tet4: [nn][6] {X, u} node records of the element pass
  // the records' u is kept current (by the predictor and the gathers) only
  // while a pass that reads the records runs: the per-element Tet4 passes
  // (filtered materials, user laws, the FP64 fast form, the pipelined
  // schedule's partial launches); the staged passes read X and u
  bool xu_static = false;
  bool records_live() const { return xu_static || (pipe_parts > 1 && pipe_ok); }
  DevBuf<int64_t> ell_off; // [nn/256 + 1]
  DevBuf<uint8_t> deg;     // [nn]
  int64_t ell_total = 0;   // entries of the node-major table
  DevBuf<unsigned char> fe; // [entries][3] of double or float
  // FP32 Tet4 block-partial assembly: the table holds one entry per (block,
  // distinct node of the block) instead of one per element corner
  bool bpa = false;
  DevBuf<int64_t> bp_off;
  DevBuf<uint8_t> bp_deg;
  int64_t bp_total = 0;
  int64_t bp_entries = 0; // without the slices' padding
  // FP64 Tet4 partial-sum assembly: prefix partials (same bits, fewer
  // entries: each node's first-block sum, then one entry per later corner)
  // or, opted into, block partials (one entry per (block, node))
  bool ppa = false;
  int assembly = AKX_ASSEMBLY_DEFAULT; // akx_model_set_block_assembly
  DevBuf<int64_t> pp_off;
  DevBuf<uint8_t> pp_deg;
  int64_t pp_total = 0;
  int64_t pp_entries = 0, pp_runs = 0; // table entries, summed runs
  // one launch per step (plan_small_steps; step.nblocks 0: not planned): the
  // lists and the dynamic LDS
  StepArgs step{};
  DevBuf<unsigned char> step_lists;
  size_t step_lds = 0;
  // more than STREAM_BYTES a step; the Hex8 jacobian table (STREAM_JAC_PLASTIC)
  bool stream_loads = true, stream_jac = true;
  DevBuf<unsigned char> staging;
  Downloader download;
  DevBuf<unsigned long long> scratch_u64;
  DevBuf<long long> scratch_i64;
  std::vector<std::unique_ptr<Material>> mats;
  // computeStress of the user materials, and host copies of their internals
  akx_compute_stress_fn stress_fn = nullptr;
  void *stress_user = nullptr;
  std::vector<double> user_grad, user_stress;
  bool has_user() const {
    for (auto &mp : mats)
      if (mp->user())
        return true;
    return false;
  }
  // pipelined schedule (akx_model_set_pipeline): element parts and the node
  // groups whose gather they complete, a second stream and the events
  int pipe_parts = 0;
  bool pipe_planned = false, pipe_ok = false;
  std::vector<int64_t> pipe_el;   // [P + 1] element ranges of the parts
  std::vector<int64_t> pipe_node; // [P + 1] node ranges of the gather groups
  std::vector<int> pipe_need;     // [P] last group part p's nodes belong to
  hipStream_t stream2 = nullptr;
  std::vector<hipEvent_t> ev_elem, ev_gather[2];
  // kernel timing
  bool timing = false;
  double t_ms[3] = {0, 0, 0};
  int64_t t_n[3] = {0, 0, 0};
  std::vector<std::pair<hipEvent_t, hipEvent_t>> pending[3];
  std::vector<hipEvent_t> event_pool;

  ~akx_model() {
    drain_timing();
    for (auto e : event_pool)
      (void)hipEventDestroy(e);
    for (auto e : ev_elem)
      (void)hipEventDestroy(e);
    for (auto &v : ev_gather)
      for (auto e : v)
        (void)hipEventDestroy(e);
    if (stream2)
      (void)hipStreamDestroy(stream2);
    if (stream)
      (void)hipStreamDestroy(stream);
  }

  void set_device() { HIPCHECK(hipSetDevice(device)); }

  hipEvent_t get_event() {
    if (!event_pool.empty()) {
      hipEvent_t e = event_pool.back();
      event_pool.pop_back();
      return e;
    }
    hipEvent_t e;
    HIPCHECK(hipEventCreate(&e));
    return e;
  }

  void drain_timing() {
    for (int k = 0; k < 3; ++k) {
      for (auto &pr : pending[k]) {
        if (hipEventSynchronize(pr.second) == hipSuccess) {
          float ms = 0.f;
          if (hipEventElapsedTime(&ms, pr.first, pr.second) == hipSuccess) {
            t_ms[k] += ms;
            t_n[k] += 1;
          }
        }
        event_pool.push_back(pr.first);
        event_pool.push_back(pr.second);
      }
      pending[k].clear();
    }
  }

  template <class F> void timed(int cls, F &&launch) {
    if (!timing) {
      launch();
      return;
    }
    hipEvent_t e0 = get_event(), e1 = get_event();
    HIPCHECK(hipEventRecord(e0, stream));
    launch();
    HIPCHECK(hipEventRecord(e1, stream));
    pending[cls].push_back({e0, e1});
    if (pending[cls].size() > 4096)
      drain_timing();
  }

  size_t fe_elem_size() const {
    return precision == AKX_PRECISION_FP32 ? sizeof(float) : sizeof(double);
  }
};

namespace {

constexpr int TPB = 256;

// device address of the no-allocation energy's scratch array (set up once
// per device)
double *device_scratch(int device);

inline unsigned grid_for(int64_t n) { return (unsigned)((n + TPB - 1) / TPB); }
inline int64_t padded_blocks(int64_t n) {
  int64_t nb = (n + TPB - 1) / TPB;
  return (nb + 7) / 8 * 8;
}

void upload_hex8_tables() {
  static bool done_device[64] = {false};
  int dev = 0;
  HIPCHECK(hipGetDevice(&dev));
  if (dev < 64 && done_device[dev])
    return;
  Hex8Tables t;
  fill_hex8_tables(t);
  HIPCHECK(hipMemcpyToSymbol(HIP_SYMBOL(c_hex8), &t, sizeof(t)));
  HIPCHECK(akxf::upload_hex8_dnds(&t.dnds[0][0][0]));
  if (dev < 64)
    done_device[dev] = true;
}

template <class T>
void upload_soa(akx_model *m, const T *host_aos, T *dev_soa, int64_t n, int comps) {
  size_t bytes = (size_t)n * comps * sizeof(T);
  m->staging.alloc(std::max(m->staging.n, bytes));
  HIPCHECK(hipMemcpyAsync(m->staging.p, host_aos, bytes, hipMemcpyHostToDevice,
                          m->stream));
  hipLaunchKernelGGL(k_aos_to_soa<T>, dim3(grid_for(n * comps)), dim3(TPB), 0,
                     m->stream, (const T *)m->staging.p, dev_soa, n, comps);
  HIPCHECK(hipGetLastError());
  HIPCHECK(hipStreamSynchronize(m->stream));
}

template <class T>
Downloader::Field soa_field(akx_model *m, const T *dev_soa, T *host_aos, T *copy, int64_t n,
                            int comps) {
  return {n, comps * sizeof(T), host_aos, copy, [=](void *p, int64_t first, int64_t count) {
            hipLaunchKernelGGL(k_soa_to_aos<T>, dim3(grid_for(count * comps)), dim3(TPB), 0,
                               m->stream, dev_soa, (T *)p, n, comps, first, count);
            HIPCHECK(hipGetLastError());
          }};
}

template <class T>
void download_soa(akx_model *m, const T *dev_soa, T *host_aos, int64_t n, int comps) {
  std::vector<Downloader::Field> f{soa_field<T>(m, dev_soa, host_aos, nullptr, n, comps)};
  m->download.get(m->device, m->stream, f);
}

// Tet4 node records: X and u (init) or u alone (after an upload of u)
void refresh_xu(akx_model *m, bool with_x) {
  if (!m->xu.p || m->nn == 0)
    return;
  hipLaunchKernelGGL(k_fill_xu, dim3(grid_for(m->nn)), dim3(TPB), 0, m->stream,
                     (const double *)m->X.p, (const double *)m->u.p, m->nn, m->xu.p, with_x);
  HIPCHECK(hipGetLastError());
}

// Element passes with block lists: for each block of bs consecutive
// elements of a contiguous material, its distinct nodes in ascending order
// (the staging loads coalesce; every block's list padded with -1 to the longest) and each element's
// corners as indices into them (the Tet4 passes stage these nodes' records
// in LDS).  In FP32 also, for block-partial assembly, the LDS slot of every
// corner: the corners of distinct node k of a block take consecutive slots
// in ascending element (then corner) order.
void build_block_nodes(akx_model *m, Material &mat, int64_t bs = 256) {
  const int nnpe = m->nnpe;
  const int64_t n = mat.n, nb = (n + bs - 1) / bs;
  std::vector<int32_t> off(nb + 1, 0), nodes;
  std::vector<uint16_t> lc(n * nnpe);
  std::vector<int32_t> local(m->nn, 0);
  DistinctNodes distinct(m->nn);
  const int32_t *conn = m->conn_host.data() + mat.first * nnpe;
  nodes.reserve(n);
  int32_t maxu = 0;
  for (int64_t b = 0; b < nb; ++b) {
    const int64_t start = (int64_t)nodes.size();
    const int64_t c0 = b * bs * nnpe, c1 = std::min<int64_t>(n, b * bs + bs) * nnpe;
    distinct.append(conn + c0, c1 - c0, nodes);
    for (int64_t k = start; k < (int64_t)nodes.size(); ++k)
      local[nodes[k]] = (int32_t)(k - start);
    for (int64_t i = c0; i < c1; ++i)
      lc[i] = (uint16_t)local[conn[i]];
    require((int64_t)nodes.size() < (int64_t)INT32_MAX, "block node lists too large");
    off[b + 1] = (int32_t)nodes.size();
    maxu = std::max<int32_t>(maxu, off[b + 1] - off[b]);
  }
  std::vector<int32_t> padded((size_t)nb * maxu, -1);
  for (int64_t b = 0; b < nb; ++b)
    std::copy(nodes.begin() + off[b], nodes.begin() + off[b + 1],
              padded.begin() + b * maxu);
  mat.bl_nodes.alloc(padded.size());
  mat.lconn.alloc(n * nnpe);
  HIPCHECK(hipMemcpy(mat.bl_nodes.p, padded.data(), padded.size() * sizeof(int32_t),
                     hipMemcpyHostToDevice));
  HIPCHECK(hipMemcpy(mat.lconn.p, lc.data(), lc.size() * sizeof(uint16_t),
                     hipMemcpyHostToDevice));
  mat.bl_maxu = maxu;
  mat.bl_nodes_host = std::move(padded);
  if (m->precision != AKX_PRECISION_FP32)
    return;
  std::vector<uint16_t> soff((size_t)nb * (maxu + 1), 0), slot(n * nnpe);
  std::vector<uint16_t> cnt(maxu + 1);
  for (int64_t b = 0; b < nb; ++b) {
    const int64_t e0 = b * bs, e1 = std::min<int64_t>(n, b * bs + bs);
    std::fill(cnt.begin(), cnt.end(), 0);
    for (int64_t i = e0 * nnpe; i < e1 * nnpe; ++i)
      cnt[lc[i]]++;
    uint16_t *o = &soff[b * (maxu + 1)];
    o[0] = 0;
    for (int k = 0; k < maxu; ++k)
      o[k + 1] = (uint16_t)(o[k] + cnt[k]);
    std::fill(cnt.begin(), cnt.end(), 0);
    for (int64_t i = e0 * nnpe; i < e1 * nnpe; ++i)
      slot[i] = (uint16_t)(o[lc[i]] + cnt[lc[i]]++);
  }
  mat.lslot.alloc(slot.size());
  mat.bl_soff.alloc(soff.size());
  HIPCHECK(hipMemcpy(mat.lslot.p, slot.data(), slot.size() * sizeof(uint16_t),
                     hipMemcpyHostToDevice));
  HIPCHECK(hipMemcpy(mat.bl_soff.p, soff.data(), soff.size() * sizeof(uint16_t),
                     hipMemcpyHostToDevice));
}

// Gather table of the block-partial assembly: node n's entries are the
// partials of the (material, block) pairs whose elements touch it, ranked
// in material order, then ascending block -- a fixed order, so repeated
// runs give the same bits.  Same node-major sliced-ELL layout as the
// per-element table.
void build_bpa_table(akx_model *m) {
  std::vector<int32_t> deg(m->nn, 0);
  for (auto &mp : m->mats)
    for (int32_t node : mp->bl_nodes_host)
      if (node >= 0)
        deg[node]++;
  const int64_t nslices = (m->nn + 255) / 256;
  std::vector<int64_t> off(nslices + 1, 0);
  for (int64_t sl = 0; sl < nslices; ++sl) {
    int w = 0;
    for (int64_t nd = sl * 256; nd < std::min<int64_t>(m->nn, sl * 256 + 256); ++nd)
      w = std::max(w, deg[nd]);
    require(w <= 255, "a node belongs to more than 255 element blocks");
    off[sl + 1] = off[sl] + (int64_t)w * 256;
  }
  m->bp_total = off[nslices];
  require(m->bp_total < (int64_t)INT32_MAX, "block-partial table too large for int32");
  std::vector<int32_t> fill(m->nn, 0);
  for (auto &mp : m->mats) {
    std::vector<int32_t> pos(mp->bl_nodes_host.size(), -1);
    for (size_t k = 0; k < pos.size(); ++k) {
      const int32_t node = mp->bl_nodes_host[k];
      if (node < 0)
        continue;
      const int32_t d = fill[node]++;
      pos[k] = (int32_t)(off[node >> 8] + (int64_t)d * 256 + (node & 255));
    }
    mp->bl_pos.alloc(pos.size());
    HIPCHECK(hipMemcpy(mp->bl_pos.p, pos.data(), pos.size() * sizeof(int32_t),
                       hipMemcpyHostToDevice));
  }
  std::vector<uint8_t> deg8(m->nn);
  m->bp_entries = 0;
  for (int64_t nd = 0; nd < m->nn; ++nd) {
    deg8[nd] = (uint8_t)deg[nd];
    m->bp_entries += deg[nd];
  }
  m->bp_off.alloc(off.size());
  m->bp_deg.alloc(std::max<int64_t>(m->nn, 1));
  HIPCHECK(hipMemcpy(m->bp_off.p, off.data(), off.size() * sizeof(int64_t),
                     hipMemcpyHostToDevice));
  HIPCHECK(hipMemcpy(m->bp_deg.p, deg8.data(), deg8.size(), hipMemcpyHostToDevice));
}

// Prefix- or block-partial assembly of the FP64 Tet4 path (k_tet4_ppa) on
// the 256-element blocks of the staged node records (build_block_nodes).
// Node n's corners, in assembly order (materials in order, elements
// ascending), come in runs: the corners in one block of one material.
// full = false: the node's first run is summed in LDS in that order (the
// gather then adds the same values in the same order: same bits) and every
// later corner keeps an entry of its own.  full = true: every run is summed,
// one entry per (block, node), added by the gather in block order (other
// rounding).  The table keeps the node-major sliced-ELL layout.  Requires
// every material contiguous and its block lists built.
void build_ppa(akx_model *m, bool full) {
  const int64_t TB = PPA_TB;
  const size_t nm = m->mats.size();
  std::vector<int32_t> nent(m->nn, 0), seen(m->nn, 0), base(m->nn, 0), cnt(m->nn, 0);
  std::vector<int64_t> stamp(m->nn, -1), entry0(m->nn, 0);
  std::vector<uint8_t> summed(m->nn, 0);
  std::vector<int64_t> off;
  std::vector<int32_t> nodes;
  int32_t maxslots = 0;
  // one traversal in assembly order; the second also writes the tables
  auto traverse = [&](bool write, std::vector<std::vector<int32_t>> *code,
                      std::vector<std::vector<int32_t>> *poff,
                      std::vector<std::vector<uint16_t>> *pend,
                      std::vector<std::vector<int32_t>> *ppos) {
    std::fill(nent.begin(), nent.end(), 0);
    std::fill(stamp.begin(), stamp.end(), -1);
    int64_t gb = 0;
    for (size_t k = 0; k < nm; ++k) {
      const Material &mat = *m->mats[k];
      const int64_t nb = (mat.n + TB - 1) / TB;
      if (write) {
        (*code)[k].assign(mat.n * 4, 0);
        (*poff)[k].assign(nb + 1, 0);
        (*pend)[k].clear();
        (*ppos)[k].clear();
      }
      for (int64_t b = 0; b < nb; ++b, ++gb) {
        const int64_t e0 = b * TB, e1 = std::min<int64_t>(mat.n, e0 + TB);
        nodes.clear();
        for (int64_t i = e0; i < e1; ++i)
          for (int a = 0; a < 4; ++a) {
            const int32_t node = m->conn_host[(mat.first + i) * 4 + a];
            if (stamp[node] != gb) {
              stamp[node] = gb;
              cnt[node] = 0;
              nodes.push_back(node);
            }
            cnt[node]++;
          }
        int32_t slots = 0;
        for (int32_t node : nodes) {
          summed[node] = full || nent[node] == 0;
          seen[node] = 0;
          entry0[node] = nent[node];
          if (summed[node]) {
            base[node] = slots;
            slots += cnt[node];
            if (write) {
              (*pend)[k].push_back((uint16_t)slots);
              (*ppos)[k].push_back(
                  (int32_t)(off[node >> 8] + (int64_t)nent[node] * 256 + (node & 255)));
            }
            nent[node] += 1;
          } else {
            nent[node] += cnt[node];
          }
        }
        maxslots = std::max(maxslots, slots);
        if (!write)
          continue;
        (*poff)[k][b + 1] = (int32_t)(*pend)[k].size();
        for (int64_t i = e0; i < e1; ++i)
          for (int a = 0; a < 4; ++a) {
            const int32_t node = m->conn_host[(mat.first + i) * 4 + a];
            const int32_t j = seen[node]++;
            (*code)[k][i * 4 + a] =
                summed[node] ? -1 - (base[node] + j)
                             : (int32_t)(off[node >> 8] + (entry0[node] + j) * 256 + (node & 255));
          }
      }
    }
  };
  traverse(false, nullptr, nullptr, nullptr, nullptr);
  const int64_t nslices = (m->nn + 255) / 256;
  off.assign(nslices + 1, 0);
  std::vector<uint8_t> deg8(m->nn, 0);
  for (int64_t sl = 0; sl < nslices; ++sl) {
    int w = 0;
    for (int64_t nd = sl * 256; nd < std::min<int64_t>(m->nn, sl * 256 + 256); ++nd) {
      require(nent[nd] <= 255, "a node has more than 255 table entries");
      deg8[nd] = (uint8_t)nent[nd];
      w = std::max<int>(w, nent[nd]);
    }
    off[sl + 1] = off[sl] + (int64_t)w * 256;
  }
  require(off[nslices] < (int64_t)INT32_MAX, "partial-sum table too large for int32");
  std::vector<std::vector<int32_t>> code(nm), poff(nm), ppos(nm);
  std::vector<std::vector<uint16_t>> pend(nm);
  traverse(true, &code, &poff, &pend, &ppos);
  for (size_t k = 0; k < nm; ++k) {
    Material &mat = *m->mats[k];
    mat.t_nblk = (mat.n + TB - 1) / TB;
    mat.t_slots = maxslots;
    const size_t np = pend[k].size();
    mat.pcode.alloc(mat.n * 4);
    mat.poff.alloc(poff[k].size());
    mat.pend.alloc(std::max<size_t>(np, 1));
    mat.ppos.alloc(std::max<size_t>(np, 1));
    HIPCHECK(hipMemcpy(mat.pcode.p, code[k].data(), mat.n * 4 * sizeof(int32_t),
                       hipMemcpyHostToDevice));
    HIPCHECK(hipMemcpy(mat.poff.p, poff[k].data(), poff[k].size() * sizeof(int32_t),
                       hipMemcpyHostToDevice));
    if (np > 0) {
      HIPCHECK(hipMemcpy(mat.pend.p, pend[k].data(), np * sizeof(uint16_t),
                         hipMemcpyHostToDevice));
      HIPCHECK(hipMemcpy(mat.ppos.p, ppos[k].data(), np * sizeof(int32_t),
                         hipMemcpyHostToDevice));
    }
  }
  m->pp_total = off[nslices];
  m->pp_entries = 0;
  for (int64_t nd = 0; nd < m->nn; ++nd)
    m->pp_entries += nent[nd];
  m->pp_runs = 0;
  for (size_t k = 0; k < nm; ++k)
    m->pp_runs += (int64_t)pend[k].size();
  m->pp_off.alloc(off.size());
  m->pp_deg.alloc(std::max<int64_t>(m->nn, 1));
  HIPCHECK(hipMemcpy(m->pp_off.p, off.data(), off.size() * sizeof(int64_t),
                     hipMemcpyHostToDevice));
  HIPCHECK(hipMemcpy(m->pp_deg.p, deg8.data(), deg8.size(), hipMemcpyHostToDevice));
}

// FP32 form: (float(lambda), float(mu)) pairs of a material with per-element
// constants, the values its element pass rounds the FP64 pair to
void fill_lame_f32(akx_model *m, Material &mat) {
  mat.lm_f.alloc(mat.n);
  hipLaunchKernelGGL(k_lame_f32, dim3(grid_for(mat.n)), dim3(TPB), 0, m->stream,
                     (const double *)mat.lam_el.p, (const double *)mat.mu_el.p,
                     mat.lm_f.p, mat.n);
  HIPCHECK(hipGetLastError());
}

void zero_async(akx_model *m, double *p, int64_t n) {
  if (n <= 0)
    return;
  hipLaunchKernelGGL(k_fill_f64, dim3(grid_for(n)), dim3(TPB), 0, m->stream, p, n, 0.);
  HIPCHECK(hipGetLastError());
}

// ------------------------------------------------------------- launches ----
ElemArgs elem_args(akx_model *m, Material &mat, bool materialize) {
  ElemArgs A{};
  A.n = mat.n;
  A.nel = m->nel;
  A.filter = mat.contiguous ? nullptr : mat.filter.p;
  A.first = mat.first;
  A.pos_offset = mat.pos_offset;
  A.conn = m->conn.p;
  A.X = m->X.p;
  A.u = m->u.p;
  A.nn = m->nn;
  A.lambda = mat.lambda;
  A.mu = mat.mu;
  A.sigma_y = mat.sigma_y;
  A.h = mat.h;
  A.lam_el = mat.per_element ? mat.lam_el.p : nullptr;
  A.mu_el = mat.per_element ? mat.mu_el.p : nullptr;
  A.lm_f = mat.per_element ? mat.lm_f.p : nullptr;
  A.bl_nodes = mat.bl_nodes.p;
  A.lconn = mat.lconn.p;
  A.bl_maxu = mat.bl_maxu;
  if (m->bpa) {
    A.lslot = mat.lslot.p;
    A.bl_soff = mat.bl_soff.p;
    A.bl_pos = mat.bl_pos.p;
  }
  if (m->ppa) {
    A.pcode = mat.pcode.p;
    A.poff = mat.poff.p;
    A.pend = mat.pend.p;
    A.ppos = mat.ppos.p;
    A.t_nblk = mat.t_nblk;
    A.t_slots = mat.t_slots;
  }
  A.sy_el = mat.sy_el.p;
  A.h_el = mat.h_el.p;
  A.pos = m->pos.p;
  A.fe = m->fe.p;
  A.jw = m->jw.p;
  A.xu = m->xu.p;
  if (mat.user()) {
    A.stress = mat.stress.p; // read by the force pass
  } else if (materialize && mat.law != AKX_LAW_PLASTIC_LIH) {
    A.grad_u = mat.grad.p;
    A.stress = mat.stress.p;
  }
  if (mat.law == AKX_LAW_PLASTIC_LIH) {
    int p = mat.cur, c = 1 - mat.cur;
    A.p_grad = mat.hgrad[p].p;
    A.p_sig = mat.hsig[p].p;
    A.p_eps = mat.heps[p].p;
    A.p_iso = mat.hiso[p].p;
    A.c_grad = mat.hgrad[c].p;
    A.c_sig = mat.hsig[c].p;
    A.c_eps = mat.heps[c].p;
    A.c_iso = mat.hiso[c].p;
    A.p_pe = mat.hpe[p].p;
    A.c_pe = mat.hpe[c].p;
    if (mat.sth_now.p) {
      A.sth_p = mat.hsth[p].p;
      A.sth_c = mat.hsth[c].p;
    }
  }
  A.eig = mat.eig.p;
  A.sth_now = mat.sth_now.p;
  A.nblocks_padded = padded_blocks(mat.n);
  return A;
}

// Host-side checks that every buffer a kernel variant dereferences exists
// (a kernel must never be launched with a null pointer it will use).
void check_gather_args(const GatherArgs &G, bool update, bool comp) {
  require(G.ell_off && G.deg && G.fe, "gather launched without its table");
  require(G.fint || update, "a gather without update must store f_int");
  if (update)
    require(G.mass && G.blocked && G.u && G.v && G.a,
            "nodal update launched without nodal state");
  if (comp)
    require(G.cu && G.cv, "compensated update launched without compensation terms");
}

void check_elem_args(const ElemArgs &A, int law) {
  require(A.conn && A.X && A.u && A.fe && A.pos,
          "element pass launched without mesh or state");
  require(A.n <= 0 || A.nblocks_padded > 0, "element pass launched with an empty grid");
  if (law == AKX_LAW_PLASTIC_LIH)
    require(A.p_grad && A.p_sig && A.p_eps && A.p_iso && A.c_grad && A.c_sig &&
                A.c_eps && A.c_iso,
            "plastic element pass launched without history buffers");
  if (A.lam_el || A.mu_el)
    require(A.lam_el && A.mu_el, "per-element parameters incomplete");
  if (law == AKX_LAW_USER || law == AKX_LAW_USER_FD)
    require(A.stress != nullptr, "user material without its stress array");
  else if (A.grad_u || A.stress)
    require(A.grad_u && A.stress, "materialised internals incomplete");
}

template <int ET, class CT, class FT, bool EXT>
void launch_elem_law_x(akx_model *m, Material &mat, const ElemArgs &A) {
  dim3 grid((unsigned)A.nblocks_padded), block(TPB);
  if constexpr (ET == ET_TET4) {
    if (A.lconn && TPB == 256) { // block node lists of a whole contiguous material
      const size_t lds = (size_t)A.bl_maxu * 48;
      switch (mat.law) {
      case AKX_LAW_ELASTIC:
        hipLaunchKernelGGL((k_tet4_strict_lds<LAW_ELASTIC, CT, FT, EXT>), grid, block, lds,
                           m->stream, A);
        HIPCHECK(hipGetLastError());
        return;
      case AKX_LAW_ELASTIC_FD:
        hipLaunchKernelGGL((k_tet4_strict_lds<LAW_ELASTIC_FD, CT, FT, EXT>), grid, block, lds,
                           m->stream, A);
        HIPCHECK(hipGetLastError());
        return;
      case AKX_LAW_NEOHOOKEAN:
        hipLaunchKernelGGL((k_tet4_strict_lds<LAW_NEOHOOKEAN, CT, FT, EXT>), grid, block, lds,
                           m->stream, A);
        HIPCHECK(hipGetLastError());
        return;
      case AKX_LAW_PLASTIC_LIH:
        hipLaunchKernelGGL((k_tet4_strict_lds<LAW_PLASTIC, CT, FT, EXT>), grid, block, lds,
                           m->stream, A);
        HIPCHECK(hipGetLastError());
        return;
      default: // user laws: the per-element pass
        break;
      }
    }
  }
  switch (mat.law) {
  case AKX_LAW_ELASTIC:
    hipLaunchKernelGGL((k_element_forces<ET, LAW_ELASTIC, CT, FT, EXT>), grid, block,
                       0, m->stream, A);
    break;
  case AKX_LAW_ELASTIC_FD:
    hipLaunchKernelGGL((k_element_forces<ET, LAW_ELASTIC_FD, CT, FT, EXT>), grid,
                       block, 0, m->stream, A);
    break;
  case AKX_LAW_NEOHOOKEAN:
    hipLaunchKernelGGL((k_element_forces<ET, LAW_NEOHOOKEAN, CT, FT, EXT>), grid,
                       block, 0, m->stream, A);
    break;
  case AKX_LAW_PLASTIC_LIH:
    hipLaunchKernelGGL((k_element_forces<ET, LAW_PLASTIC, CT, FT, EXT>), grid, block,
                       0, m->stream, A);
    break;
  case AKX_LAW_USER:
    hipLaunchKernelGGL((k_element_forces<ET, LAW_USER, CT, FT, EXT>), grid, block, 0,
                       m->stream, A);
    break;
  case AKX_LAW_USER_FD:
    hipLaunchKernelGGL((k_element_forces<ET, LAW_USER_FD, CT, FT, EXT>), grid, block, 0,
                       m->stream, A);
    break;
  default:
    throw Error(AKX_ERR_UNSUPPORTED, "unknown law");
  }
  HIPCHECK(hipGetLastError());
}

template <int ET, class CT, class FT>
void launch_elem_law(akx_model *m, Material &mat, const ElemArgs &A) {
  if (mat.ext())
    launch_elem_law_x<ET, CT, FT, true>(m, mat, A);
  else
    launch_elem_law_x<ET, CT, FT, false>(m, mat, A);
}

template <int LAW> void launch_hex8_strict_law(akx_model *m, Material &mat, const ElemArgs &A) {
  const dim3 grid((unsigned)A.nblocks_padded), block(64);
  if (mat.ext())
    hipLaunchKernelGGL((k_hex8_strict<LAW, true>), grid, block, 0, m->stream, A);
  else if (m->stream_jac)
    hipLaunchKernelGGL((k_hex8_strict<LAW, false, true>), grid, block, 0, m->stream, A);
  else
    hipLaunchKernelGGL((k_hex8_strict<LAW, false, false>), grid, block, 0, m->stream, A);
}

void launch_hex8_strict(akx_model *m, Material &mat, const ElemArgs &A) {
  require(A.jw != nullptr, "Hex8 element pass without its jacobian table");
  switch (mat.law) {
  case AKX_LAW_ELASTIC: launch_hex8_strict_law<LAW_ELASTIC>(m, mat, A); break;
  case AKX_LAW_ELASTIC_FD: launch_hex8_strict_law<LAW_ELASTIC_FD>(m, mat, A); break;
  case AKX_LAW_NEOHOOKEAN: launch_hex8_strict_law<LAW_NEOHOOKEAN>(m, mat, A); break;
  case AKX_LAW_PLASTIC_LIH: launch_hex8_strict_law<LAW_PLASTIC>(m, mat, A); break;
  case AKX_LAW_USER: launch_hex8_strict_law<LAW_USER>(m, mat, A); break;
  case AKX_LAW_USER_FD: launch_hex8_strict_law<LAW_USER_FD>(m, mat, A); break;
  default:
    throw Error(AKX_ERR_UNSUPPORTED, "unknown law");
  }
  HIPCHECK(hipGetLastError());
}

template <int LAW> void launch_tet4_ppa_law(akx_model *m, Material &mat, const ElemArgs &A) {
  const dim3 grid((unsigned)A.nblocks_padded), block(PPA_TB);
  const size_t lds = std::max((size_t)A.bl_maxu * 48, (size_t)A.t_slots * 24);
  if (mat.ext())
    hipLaunchKernelGGL((k_tet4_ppa<LAW, true, true>), grid, block, lds, m->stream, A);
  else if (LAW == LAW_PLASTIC || A.grad_u)
    hipLaunchKernelGGL((k_tet4_ppa<LAW, false, true>), grid, block, lds, m->stream, A);
  else
    hipLaunchKernelGGL((k_tet4_ppa<LAW, false, LAW == LAW_PLASTIC>), grid, block, lds, m->stream,
                       A);
}

void launch_tet4_ppa(akx_model *m, Material &mat, const ElemArgs &A) {
  switch (mat.law) {
  case AKX_LAW_ELASTIC: launch_tet4_ppa_law<LAW_ELASTIC>(m, mat, A); break;
  case AKX_LAW_ELASTIC_FD: launch_tet4_ppa_law<LAW_ELASTIC_FD>(m, mat, A); break;
  case AKX_LAW_NEOHOOKEAN: launch_tet4_ppa_law<LAW_NEOHOOKEAN>(m, mat, A); break;
  case AKX_LAW_PLASTIC_LIH: launch_tet4_ppa_law<LAW_PLASTIC>(m, mat, A); break;
  default: // user laws never take this path
    throw Error(AKX_ERR_UNSUPPORTED, "prefix-partial pass for a user law");
  }
  HIPCHECK(hipGetLastError());
}

void launch_device_law(akx_model *m, Material &mat, ElemArgs A, bool materialize);

void launch_element_pass(akx_model *m, bool materialize) {
  const bool strict = m->precision == AKX_PRECISION_FP64;
  for (auto &mp : m->mats) {
    Material &mat = *mp;
    if (mat.n == 0)
      continue;
    ElemArgs A = elem_args(m, mat, materialize);
    check_elem_args(A, mat.law);
    require(!mat.ext() || strict,
            "eigen_grad_u and thermal stresses run on the plain FP64 path");
    require(!(mat.sth_now.p && mat.law == AKX_LAW_PLASTIC_LIH) || (A.sth_p && A.sth_c),
            "plastic thermal stress without its history");
    require(m->etype != AKX_TET4 || A.xu != nullptr, "Tet4 element pass without its node records");
    require(m->fe.n >= (size_t)(m->ell_total * 3 * m->fe_elem_size()) &&
                m->fe.n >= (size_t)(m->bp_total * 3 * m->fe_elem_size()) &&
                m->pos.n >= (size_t)((mat.pos_offset + mat.n) * m->nnpe),
            "element force table too small for this material");
    if (m->bpa)
      require(A.lslot && A.bl_soff && A.bl_pos && A.bl_nodes && A.lconn,
              "block-partial pass launched without its block tables");
    if (strict && m->etype == AKX_HEX8) {
      int64_t nb = (mat.n + HEX_STRICT_EPB - 1) / HEX_STRICT_EPB;
      A.nblocks_padded = (nb + 7) / 8 * 8;
    } else if (!strict) {
      int64_t epb = akxf::elements_per_block(m->etype, m->bpa);
      int64_t nb = (mat.n + epb - 1) / epb;
      A.nblocks_padded = (nb + 7) / 8 * 8;
    }
    if (strict && m->ppa) {
      require(A.pcode && A.poff && A.pend && A.ppos && A.bl_nodes && A.lconn &&
                  A.t_nblk == (mat.n + PPA_TB - 1) / PPA_TB,
              "prefix-partial pass launched without its block tables");
      A.nblocks_padded = (A.t_nblk + 7) / 8 * 8;
    }
    m->timed(0, [&] {
      if (mat.dlaw) {
        require(strict, "device laws run on the plain FP64 path");
        launch_device_law(m, mat, A, materialize);
      } else if (strict && m->ppa) {
        launch_tet4_ppa(m, mat, A);
      } else if (strict) {
        if (m->etype == AKX_TET4)
          launch_elem_law<ET_TET4, double, double>(m, mat, A);
        else
          launch_hex8_strict(m, mat, A);
      } else {
        HIPCHECK(akxf::launch_elements(m->etype, mat.law,
                                       m->precision == AKX_PRECISION_FP32, A,
                                       m->stream));
      }
    });
  }
}

// The computeStress plugin of the user materials (Material::computeStress,
// material.cc:128-154): grad u at every Gauss point of the material (the
// reference order, as the other laws form it), handed to the caller, whose
// stress goes back to the device for the force pass.
void user_stress_phase(akx_model *m) {
  if (!m->has_user())
    return;
  for (int k = 0; k < (int)m->mats.size(); ++k) {
    Material &mat = *m->mats[k];
    if (!mat.user() || mat.n == 0)
      continue;
    if (mat.dlaw) // the law runs inside the element pass
      continue;
    require(m->stress_fn != nullptr,
            "a user material needs a computeStress callback (akx_model_set_stress_callback) "
            "or a device law (akx_model_set_device_stress)");
    const int64_t nq = mat.n * m->nqp;
    ElemArgs A = elem_args(m, mat, false);
    A.grad_u = mat.grad.p;
    A.stress = nullptr;
    require(A.grad_u && A.conn && A.X && A.u, "user material gradient pass without buffers");
    require(m->etype != AKX_TET4 || A.xu != nullptr, "Tet4 gradient pass without its node records");
    if (m->etype == AKX_HEX8) {
      require(A.jw != nullptr, "Hex8 gradient pass without its jacobian table");
      const int64_t nb = (mat.n + HEX_STRICT_EPB - 1) / HEX_STRICT_EPB;
      A.nblocks_padded = (nb + 7) / 8 * 8;
      if (mat.ext())
        hipLaunchKernelGGL((k_hex8_strict<LAW_USER_GRAD, true>),
                           dim3((unsigned)A.nblocks_padded), dim3(64), 0, m->stream, A);
      else
        hipLaunchKernelGGL((k_hex8_strict<LAW_USER_GRAD, false>),
                           dim3((unsigned)A.nblocks_padded), dim3(64), 0, m->stream, A);
    } else {
      if (mat.ext())
        hipLaunchKernelGGL((k_element_forces<ET_TET4, LAW_USER_GRAD, double, double, true>),
                           dim3((unsigned)A.nblocks_padded), dim3(TPB), 0, m->stream, A);
      else
        hipLaunchKernelGGL((k_element_forces<ET_TET4, LAW_USER_GRAD, double, double, false>),
                           dim3((unsigned)A.nblocks_padded), dim3(TPB), 0, m->stream, A);
    }
    HIPCHECK(hipGetLastError());
    m->user_grad.resize(9 * nq);
    m->user_stress.assign(9 * nq, 0.);
    download_soa(m, mat.grad.p, m->user_grad.data(), nq, 9);
    const int rc = m->stress_fn(m->stress_user, k, nq, m->user_grad.data(),
                                m->user_stress.data());
    if (rc != 0)
      throw Error(AKX_ERR_INVALID,
                  "computeStress of material " + std::to_string(k) + " failed");
    upload_soa(m, m->user_stress.data(), mat.stress.p, nq, 9);
  }
}

#include "akx_rtc_sources.inc"

// Compiles the caller's law into the material's element pass with hiprtc for
// the model's GPU -- the library's own kernel headers, the plain path's
// floating-point rules (-O3, no contraction: every multiply and add rounds on
// its own) -- for the pass without and with the eigen-gradient terms, and
// loads it.  The parameters become constants of the program (hexadecimal
// literals: exact).
std::unique_ptr<DeviceLaw> compile_device_law(akx_model *m, const Material &mat,
                                              const char *source, const double *params,
                                              int nparams) {
  hipDeviceProp_t prop;
  HIPCHECK(hipGetDeviceProperties(&prop, m->device));
  std::string arch(prop.gcnArchName);
  arch = "--offload-arch=" + arch.substr(0, arch.find(':'));
  const int law = mat.law == AKX_LAW_USER_FD ? LAW_DEVICE_FD : LAW_DEVICE;
  std::string src =
      "typedef __hip_internal::int8_t int8_t;\n"
      "typedef __hip_internal::uint8_t uint8_t;\n"
      "typedef __hip_internal::int16_t int16_t;\n"
      "typedef __hip_internal::uint16_t uint16_t;\n"
      "typedef __hip_internal::int32_t int32_t;\n"
      "typedef __hip_internal::uint32_t uint32_t;\n"
      "typedef __hip_internal::int64_t int64_t;\n"
      "typedef __hip_internal::uint64_t uint64_t;\n"
      "#define AKX_DEVICE_LAW 1\n";
  src += "#line 1 \"device law\"\n";
  src += source;
  src += "\n#line 1 \"akx device law program\"\n";
  src += "__constant__ double akx_law_params[" + std::to_string(std::max(nparams, 1)) + "] = {";
  for (int k = 0; k < std::max(nparams, 1); ++k) {
    char buf[64];
    std::snprintf(buf, sizeof buf, "%a", nparams > 0 ? params[k] : 0.);
    src += (k ? ", " : "") + std::string(buf);
  }
  src += "};\n#include \"akx_kernels.hpp\"\nnamespace akx {\n__constant__ Hex8Tables c_hex8;\n}\n";
  std::string names[2];
  for (int ext = 0; ext < 2; ++ext)
    names[ext] = m->etype == AKX_HEX8
                     ? "akx::k_hex8_strict<" + std::to_string(law) + ", " +
                           (ext ? "true" : "false") + ">"
                     : "akx::k_element_forces<0, " + std::to_string(law) + ", double, double, " +
                           (ext ? "true" : "false") + ">";
  const std::string table = "&akx::c_hex8";
  hiprtcProgram prog;
  if (hiprtcCreateProgram(&prog, src.c_str(), "akx_device_law.hip", 3, k_rtc_headers,
                          k_rtc_header_names) != HIPRTC_SUCCESS)
    throw Error(AKX_ERR_HIP, "hiprtcCreateProgram failed");
  for (auto &nm : names)
    (void)hiprtcAddNameExpression(prog, nm.c_str());
  (void)hiprtcAddNameExpression(prog, table.c_str());
  const char *opts[] = {arch.c_str(), "-O3", "-std=c++17", "-ffp-contract=off",
                        "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"};
  const hiprtcResult rc = hiprtcCompileProgram(prog, 8, opts);
  if (rc != HIPRTC_SUCCESS) {
    size_t n = 0;
    std::string log;
    if (hiprtcGetProgramLogSize(prog, &n) == HIPRTC_SUCCESS && n > 0) {
      log.resize(n);
      (void)hiprtcGetProgramLog(prog, &log[0]);
    }
    (void)hiprtcDestroyProgram(&prog);
    throw Error(AKX_ERR_INVALID, std::string("the device law did not compile (") +
                                     hiprtcGetErrorString(rc) + "):\n" + log);
  }
  std::string lowered[3];
  for (int k = 0; k < 3; ++k) {
    const char *low = nullptr;
    if (hiprtcGetLoweredName(prog, k < 2 ? names[k].c_str() : table.c_str(), &low) !=
            HIPRTC_SUCCESS ||
        !low) {
      (void)hiprtcDestroyProgram(&prog);
      throw Error(AKX_ERR_HIP, "the device law program lost an instantiation");
    }
    lowered[k] = low;
  }
  size_t size = 0;
  std::vector<char> code;
  if (hiprtcGetCodeSize(prog, &size) == HIPRTC_SUCCESS && size > 0) {
    code.resize(size);
    if (hiprtcGetCode(prog, code.data()) != HIPRTC_SUCCESS)
      code.clear();
  }
  (void)hiprtcDestroyProgram(&prog);
  require(!code.empty(), "the device law compiled to no code");
  auto dl = std::make_unique<DeviceLaw>();
  HIPCHECK(hipModuleLoadData(&dl->module, code.data()));
  for (int ext = 0; ext < 2; ++ext)
    HIPCHECK(hipModuleGetFunction(&dl->kernel[ext], dl->module, lowered[ext].c_str()));
  hipDeviceptr_t tab = nullptr;
  size_t tab_bytes = 0;
  HIPCHECK(hipModuleGetGlobal(&tab, &tab_bytes, dl->module, lowered[2].c_str()));
  Hex8Tables t;
  fill_hex8_tables(t);
  require(tab_bytes == sizeof(t), "the device law program's Hex8 table has another size");
  HIPCHECK(hipMemcpy((void *)tab, &t, sizeof(t), hipMemcpyHostToDevice));
  return dl;
}

// The element pass of a material whose law was compiled in
void launch_device_law(akx_model *m, Material &mat, ElemArgs A, bool materialize) {
  A.grad_u = materialize ? mat.grad.p : nullptr; // grad u and the stress, when asked
  A.stress = mat.stress.p;
  void *args[] = {&A};
  const unsigned grid = (unsigned)A.nblocks_padded;
  const unsigned block = m->etype == AKX_HEX8 ? 64 : TPB;
  HIPCHECK(hipModuleLaunchKernel(mat.dlaw->kernel[mat.ext() ? 1 : 0], grid, 1, 1, block, 1, 1,
                                 0, m->stream, args, nullptr));
}

void flip_plastic_state(akx_model *m) {
  for (auto &mp : m->mats)
    if (mp->law == AKX_LAW_PLASTIC_LIH)
      mp->cur = 1 - mp->cur;
}

// per_corner: the per-corner table whatever the model's assembly (the
// pipelined schedule's partial launches write it)
GatherArgs gather_args(akx_model *m, bool per_corner = false) {
  GatherArgs G{};
  G.nn = m->nn;
  G.node0 = 0;
  G.node_end = m->nn;
  G.ell_off = m->ell_off.p;
  G.deg = m->deg.p;
  if (m->bpa && !per_corner) {
    G.ell_off = m->bp_off.p;
    G.deg = m->bp_deg.p;
  } else if (m->ppa && !per_corner) {
    G.ell_off = m->pp_off.p;
    G.deg = m->pp_deg.p;
  }
  G.fe = m->fe.p;
  G.fint = m->fint.p;
  G.fext = m->has_fext ? m->fext.p : nullptr;
  G.mass = m->mass.p;
  G.blocked = m->blocked.p;
  G.u = m->u.p;
  G.xu = m->records_live() ? m->xu.p : nullptr;
  G.v = m->v.p;
  G.a = m->a.p;
  G.cu = m->cu.p;
  G.cv = m->cv.p;
  G.dt = m->dt;
  G.nblocks_padded = padded_blocks(m->nn);
  G.stream = m->stream_loads;
  return G;
}

template <class FT, bool COMP, bool FEW>
void launch_gather_form(const GatherArgs &G, bool update, bool predict, hipStream_t s) {
  const dim3 grid((unsigned)G.nblocks_padded), block(TPB);
  if (!update)
    hipLaunchKernelGGL((k_gather_update<FT, false, false, false, FEW>), grid, block, 0, s, G);
  else if (predict)
    hipLaunchKernelGGL((k_gather_update<FT, true, true, COMP, FEW>), grid, block, 0, s, G);
  else
    hipLaunchKernelGGL((k_gather_update<FT, true, false, COMP, FEW>), grid, block, 0, s, G);
}

void launch_gather_kernel(const GatherArgs &G, bool f64, bool update, bool predict,
                          hipStream_t s) {
  const bool few = G.node_end - G.node0 <= GATHER_FEW_NODES;
  if (f64 && few)
    launch_gather_form<double, false, true>(G, update, predict, s);
  else if (f64)
    launch_gather_form<double, false, false>(G, update, predict, s);
  else if (few)
    launch_gather_form<float, true, true>(G, update, predict, s);
  else
    launch_gather_form<float, true, false>(G, update, predict, s);
}

// f_int is stored by the last step of a solve_step call (and by the gathers
// without update): the steps in between use it only inside the gather, and
// nothing reads the stored array before the call returns.
void launch_gather(akx_model *m, bool update, bool predict) {
  GatherArgs G = gather_args(m);
  if (update && predict)
    G.fint = nullptr;
  const bool f64 = m->precision != AKX_PRECISION_FP32;
  check_gather_args(G, update, update && !f64);
  m->timed(1, [&] { launch_gather_kernel(G, f64, update, predict, m->stream); });
  HIPCHECK(hipGetLastError());
}

void launch_predictor(akx_model *m) {
  GatherArgs G = gather_args(m);
  dim3 grid((unsigned)G.nblocks_padded), block(TPB);
  check_gather_args(G, true, m->precision == AKX_PRECISION_FP32);
  m->timed(2, [&] {
    if (m->precision != AKX_PRECISION_FP32)
      hipLaunchKernelGGL((k_predictor<false>), grid, block, 0, m->stream, G);
    else
      hipLaunchKernelGGL((k_predictor<true>), grid, block, 0, m->stream, G);
  });
  HIPCHECK(hipGetLastError());
}

// ---------------------------------------------------------------------------
// One launch per step for small models (akx_step.hpp): one contiguous material
// of a built-in law over the whole mesh; Tet4 in FP64 (with plasticity) and
// FP32, Hex8 in FP64 and FP32 (block partials).
//
// A step of two launches takes 8 to 16 us however small the mesh; in one
// launch it takes 5 (plastic 7.5), what the host needs to queue it.  An
// element's arithmetic is repeated in every workgroup that owns one of its
// nodes, so the gain ends where that fills the chip.
//
// A workgroup owns a run of 8 nodes (Tet4; along a row of a box they have 150
// elements, one a lane), 6 (FP64 Hex8; 28 elements of eight lanes) or up to 16
// (FP32 Hex8; 64 elements of four lanes).  In runs a Tet4 is computed 3.1
// times, a Hex8 4.6 (FP32 4.1) times.  Groups of up to 16 neighbours (group_nodes)
// take that to 2.3 for Tet4, with a longer sum per lane: they pay in FP64 where
// the runs need more than two workgroups per CU.  (Hex8 in groups of 8: 4.1; no
// faster in FP64 up to 2,560 nodes, 1 us slower in FP32.)  The lists cost
// initFull 0.1 ms at 1,000 nodes, 1.5 ms at 7,000 (FP32 Hex8 1.1 at 11,000).
// us a step of boxes, two launches / runs / groups:
//   Tet4 FP64 elastic   525 nodes 12.0/5.1/-, 4,032 12.5/5.9/6.7, 10,416
//                       13.6/9.3/8.1
//   Tet4 FP64 neo-H.    4,032 13.6/7.5/8.2, 6,630 14.1/9.4/8.5, 10,416
//                       14.4/12.7/10.5
//   Tet4 FP64 plastic   525 14.8/7.4/-, 4,032 16/10.3/13.2, 6,975
//                       16.2/16.2/13.9, 10,416 18.3/-/21.6; in groups of 16 / 20
//                       6,630 13.7/14.1, 7,168 13.9/-, 8,192 18.7/14.6 (two
//                       launches 15.4): two of its workgroups fill a CU, and
//                       groups of 16 become more than that
//   Tet4 FP32 elastic   1,152 7.9/5.2/-, 4,032 8.1/5.7/6.7, 10,416 8.4/6.9/7.9,
//                       26,691 9.5/12.0/12.1
//   Hex8 FP64 neo-H.    1,331 9.5/7.8/-, 1,540 9.6/9.9/-, 2,520 9.7/10.0/10.4,
//                       4,032 10.8/12.5/10.8 (and with the stress at finite
//                       strain 1,540 9.4/9.4, 2,560 9.2/9.5): a second workgroup
//                       on a CU, above 256 of them, takes what the launch saved
//   Hex8 FP32 neo-H.    runs of 8 / 12 / 16 nodes: 343 8.7/5.7/-/-, 1,331
//                       9.1/5.8/5.6/5.6, 4,096 9.1/6.6/6.7/5.6, 8,192
//                       9.6/8.1/8.0/6.8, 11,200 9.2/-/8.9/8.0, 15,972
//                       9.3/-/11.3/9.1 (a numbering without locality makes more
//                       and fuller workgroups: the limit of 1,024)
//   Hex8 FP32 elastic   4,352 8.8/-/6.3/6.1, 14,801 9.5/-/8.7/8.1
//   Hex8 FP64 elastic   1,536 9.1/6.4/-, 2,520 9.2/7.7/8.0, 4,032 9.3/9.3/8.3
// ---------------------------------------------------------------------------
constexpr int STEP_RUN_TET4 = 8, STEP_GROUP_TET4 = 16, STEP_RUN_HEX8 = 6, STEP_RUN_HEX8_F32 = 16;
constexpr int STEP_GROUP_PLASTIC = 20;
constexpr int64_t STEP_RUNS_TET4 = 4096; // most nodes in runs (FP64)
constexpr int64_t STEP_GROUPS_PLASTIC = 7168; // most in groups of 16 (plastic)
constexpr int64_t STEP_NODES_TET4 = 10240, STEP_NODES_PLASTIC = 8192;
constexpr int64_t STEP_NODES_HEX8 = 1536, STEP_NODES_HEX8_ELASTIC = 2560;
constexpr int64_t STEP_NODES_HEX8_F32 = 12288, STEP_GROUPS_HEX8_F32 = 1024;
static_assert(STEP_NODES_TET4 <= STEP_NODES_MAX && STEP_NODES_PLASTIC <= STEP_NODES_MAX &&
                  STEP_NODES_HEX8 <= STEP_NODES_MAX && STEP_NODES_HEX8_ELASTIC <= STEP_NODES_MAX &&
                  STEP_NODES_HEX8_F32 <= STEP_NODES_MAX,
              "larger meshes have no second state arrays");
constexpr size_t STEP_LDS = 48 * 1024;

// Who owns which nodes: workgroup b the nodes onodes[ooff[b]] .., around them
// the elements elems[eoff[b]] .. whose corners lcs index its nodes noff[b] ..,
// all numbered as they are met.
struct StepGroups {
  std::vector<int32_t> ooff{0}, onodes, eoff{0}, elems, noff{0}, nodes;
  std::vector<uint16_t> lcs;
};

// Groups of up to `own` nodes with up to max_elems elements around them (one
// node may have more).  grow: a group starts at the lowest node left and takes
// the node of its elements that adds the fewest; else the groups are runs.
// first, around: the elements around every node.
void group_nodes(const akx_model *m, const std::vector<int32_t> &first,
                 const std::vector<int32_t> &around, int own, int max_elems, bool grow,
                 StepGroups &G) {
  const int nnpe = m->nnpe;
  const int32_t *conn = m->conn_host.data();
  const int32_t nn = (int32_t)m->nn;
  constexpr int16_t TAKEN = INT16_MAX / 2; // no node has that many elements
  std::vector<int32_t> elem_in(m->nel, -1);
  struct Met {
    int32_t in, no; // a node's latest group and its number there
  };
  std::vector<Met> met_in(nn, Met{-1, 0});
  std::vector<int16_t> more(256); // elements that each of the group's nodes would add
  std::vector<uint8_t> taken(nn, 0);
  G.onodes.reserve(nn);
  G.elems.reserve(4 * m->nel);
  G.lcs.reserve(4 * m->nel * nnpe);
  G.nodes.reserve(8 * nn);
  for (int32_t start = 0, b = 0; start < nn; ++start) {
    if (taken[start])
      continue;
    const int32_t n0 = G.noff[b];
    int32_t met = 0; // nodes of the group's elements
    for (int32_t n = start;;) {
      taken[n] = 1;
      G.onodes.push_back(n);
      if (met_in[n].in == b)
        more[met_in[n].no] = TAKEN;
      const size_t most = G.lcs.size() + (size_t)(first[n + 1] - first[n]) * nnpe;
      if (most > G.lcs.capacity())
        G.lcs.reserve(2 * most);
      if (more.size() < (size_t)met + (most - G.lcs.size()))
        more.resize(2 * (met + (most - G.lcs.size())));
      for (int32_t d = first[n]; d < first[n + 1]; ++d) {
        const int32_t e = around[d];
        if (elem_in[e] == b)
          continue;
        elem_in[e] = b;
        G.elems.push_back(e);
        uint16_t lc[8];
        for (int a = 0; a < nnpe; ++a) {
          const int32_t c = conn[(int64_t)e * nnpe + a];
          Met &at = met_in[c];
          if (at.in != b) {
            at = Met{b, met};
            G.nodes.push_back(c);
            if (grow)
              more[met] = taken[c] ? TAKEN : (int16_t)(first[c + 1] - first[c]);
            ++met;
          }
          if (grow)
            more[at.no]--;
          lc[a] = (uint16_t)at.no;
        }
        G.lcs.insert(G.lcs.end(), lc, lc + nnpe);
      }
      if ((int)G.onodes.size() - G.ooff[b] == own)
        break;
      const int32_t left = max_elems - ((int32_t)G.elems.size() - G.eoff[b]);
      if (!grow) {
        if (++n == nn || std::count_if(around.begin() + first[n], around.begin() + first[n + 1],
                                       [&](int32_t e) { return elem_in[e] != b; }) > left)
          break;
        continue;
      }
      int16_t fewest = TAKEN / 2;
      for (int32_t k = 0; k < met; ++k)
        fewest = std::min(fewest, more[k]);
      if (fewest == TAKEN / 2 || fewest > left)
        break;
      n = G.nodes[n0 + (std::find(more.begin(), more.end(), fewest) - more.begin())];
    }
    G.ooff.push_back((int32_t)G.onodes.size());
    G.eoff.push_back((int32_t)G.elems.size());
    G.noff.push_back((int32_t)G.nodes.size());
    ++b;
  }
}

void plan_small_steps(akx_model *m) {
  const bool hex = m->etype == AKX_HEX8;
  if (m->mats.size() != 1 || m->nn == 0 || m->precision == AKX_PRECISION_FP64_FAST)
    return;
  const Material &mat = *m->mats[0];
  const bool f32 = m->precision == AKX_PRECISION_FP32, plastic = mat.law == AKX_LAW_PLASTIC_LIH;
  const int64_t most_hex = f32                          ? STEP_NODES_HEX8_F32
                           : mat.law == AKX_LAW_ELASTIC ? STEP_NODES_HEX8_ELASTIC
                                                        : STEP_NODES_HEX8;
  const int64_t most = hex ? most_hex : plastic ? STEP_NODES_PLASTIC : STEP_NODES_TET4;
  if (m->nn > most)
    return;
  if (!mat.contiguous || mat.first != 0 || mat.n != m->nel || mat.n == 0 || mat.user() ||
      (plastic && (hex || f32)) || (hex && f32 && !m->bpa))
    return;
  if (!f32 && m->ppa && m->assembly == AKX_ASSEMBLY_BLOCK_PARTIALS)
    return; // sums runs in FP64 without rounding them as the FP32 form does
  const int nnpe = m->nnpe;
  const int32_t *conn = m->conn_host.data();
  const int64_t nn = m->nn, nel = m->nel;
  // elements around every node, in ascending order
  std::vector<int32_t> first(nn + 1, 0), around(nel * nnpe);
  for (int64_t i = 0; i < nel * nnpe; ++i)
    first[conn[i] + 1]++;
  for (int64_t n = 0; n < nn; ++n)
    first[n + 1] += first[n];
  std::vector<uint8_t> rank(nel * nnpe); // of a corner among its node's
  {
    std::vector<uint8_t> at(nn, 0);
    for (int32_t e = 0; e < (int32_t)nel; ++e)
      for (int a = 0; a < nnpe; ++a) {
        const int32_t n = conn[(int64_t)e * nnpe + a];
        rank[(int64_t)e * nnpe + a] = at[n];
        around[first[n] + at[n]++] = e;
      }
  }
  // who owns which nodes
  const int lanes = !hex ? 256 : f32 ? 64 : STEP_HEX_EPB; // elements at a time
  const bool grouped = !hex && !f32 && nn > STEP_RUNS_TET4;
  const int own = hex                                   ? f32 ? STEP_RUN_HEX8_F32 : STEP_RUN_HEX8
                  : !grouped                            ? STEP_RUN_TET4
                  : plastic && nn > STEP_GROUPS_PLASTIC ? STEP_GROUP_PLASTIC
                                                        : STEP_GROUP_TET4;
  StepGroups G;
  group_nodes(m, first, around, own, hex && !f32 ? 2 * lanes : lanes, grouped, G);
  const auto &[ooff, onodes, eoff, elems, noff, nodes, lcs] = G;
  const int64_t nb = (int64_t)ooff.size() - 1;
  if (hex && f32 && nb > STEP_GROUPS_HEX8_F32)
    return;
  std::vector<int32_t> owner(nn), slot0(nn);
  int32_t max_elems = 1, max_nodes = 1, max_slots = 1;
  for (int64_t b = 0; b < nb; ++b) {
    int32_t slots = 0;
    for (int32_t k = ooff[b]; k < ooff[b + 1]; ++k) {
      owner[onodes[k]] = (int32_t)b;
      slot0[onodes[k]] = slots;
      slots += first[onodes[k] + 1] - first[onodes[k]];
    }
    max_elems = std::max(max_elems, eoff[b + 1] - eoff[b]);
    max_nodes = std::max(max_nodes, noff[b + 1] - noff[b]);
    max_slots = std::max(max_slots, slots);
  }
  const size_t lds = (size_t)max_nodes * 48 +
                     (size_t)(max_slots + 1) * 3 * (f32 ? sizeof(float) : sizeof(double)) +
                     (f32 ? max_slots : 0);
  // one lane per Tet4; at most two rounds of Hex8 (a numbering without
  // locality makes long lists)
  if (max_elems > (hex && !f32 ? 2 : 1) * lanes || lds > STEP_LDS)
    return;
  // FP32 partial sums end where the element pass's block of elements does
  // (every corner is one without block assembly)
  const int32_t block = (int32_t)akxf::elements_per_block(m->etype, true);
  std::vector<uint8_t> ends(f32 ? around.size() : 0, 1);
  if (f32 && m->bpa)
    for (int64_t n = 0; n < nn; ++n)
      for (int32_t d = first[n]; d + 1 < first[n + 1]; ++d)
        ends[d] = around[d] / block != around[d + 1] / block;
  // the lists, by k_step_lists from what was found here; the upload sits in the
  // force table, which nothing uses yet
  StepArgs S{};
  S.own = own;
  S.max_nodes = max_nodes;
  S.max_elems = max_elems;
  S.max_slots = max_slots;
  S.nn = nn;
  S.nel = nel;
  S.nblocks_padded = (int32_t)((nb + 7) / 8 * 8);
  S.nblocks = (int32_t)nb;
  struct Part {
    const void *host;
    size_t bytes, at;
  };
  size_t total = 0;
  auto part = [&](const auto &v) {
    const Part p{v.data(), v.size() * sizeof(v[0]), total};
    total += (p.bytes + 15) / 16 * 16;
    return p;
  };
  const Part parts[] = {part(ooff), part(onodes), part(eoff),  part(elems), part(noff), part(nodes),
                        part(lcs),  part(owner),  part(slot0), part(rank),  part(first), part(ends)};
  std::unique_ptr<unsigned char[]> up(new unsigned char[total]);
  for (const Part &p : parts)
    std::memcpy(up.get() + p.at, p.host, p.bytes);
  DevBuf<unsigned char> more;
  unsigned char *dev = m->fe.p;
  if (m->fe.n < total) {
    more.alloc(total);
    dev = more.p;
  }
  HIPCHECK(hipMemcpy(dev, up.get(), total, hipMemcpyHostToDevice));
  const size_t n32 = nb * (max_nodes + own + max_elems), n16 = nb * (2 * max_elems * nnpe + own);
  m->step_lists.alloc((4 * n32 + 7) / 8 * 8 + 2 * n16 + (f32 ? nb * max_slots : 0));
  StepListArgs L{};
  L.lnode = reinterpret_cast<int32_t *>(m->step_lists.p);
  L.onode = L.lnode + nb * max_nodes;
  L.lelem = L.onode + nb * own;
  L.lc = reinterpret_cast<uint16_t *>(m->step_lists.p + (4 * n32 + 7) / 8 * 8);
  L.ls = L.lc + nb * max_elems * nnpe;
  L.send = L.ls + nb * max_elems * nnpe;
  L.run = f32 ? reinterpret_cast<uint8_t *>(L.send + nb * own) : nullptr;
  auto at = [&](int k) { return reinterpret_cast<const int32_t *>(dev + parts[k].at); };
  L.ooff = at(0);
  L.onodes = at(1);
  L.eoff = at(2);
  L.elems = at(3);
  L.noff = at(4);
  L.nodes = at(5);
  L.lcs = reinterpret_cast<const uint16_t *>(at(6));
  L.owner = at(7);
  L.slot0 = at(8);
  L.rank = reinterpret_cast<const uint8_t *>(at(9));
  L.first = at(10);
  L.ends = reinterpret_cast<const uint8_t *>(at(11));
  L.conn = m->conn.p;
  L.nnpe = nnpe;
  hipLaunchKernelGGL(k_step_lists, dim3((unsigned)nb), dim3(TPB), 0, m->stream, S, L);
  HIPCHECK(hipGetLastError());
  if (more.p)
    HIPCHECK(hipStreamSynchronize(m->stream));
  S.lnode = L.lnode;
  S.onode = L.onode;
  S.lelem = L.lelem;
  S.lc = L.lc;
  S.ls = L.ls;
  S.send = L.send;
  S.run = L.run;
  m->step = S;
  m->step_lds = lds;
}

// whether the next call's steps are single launches: what plan_small_steps
// could not know
bool small_steps(const akx_model *m) {
  return m->step.nblocks > 0 && !m->timing && !m->mats[0]->ext() && !m->records_live();
}

template <int LAW> void launch_step_law(akx_model *m, const StepArgs &S) {
  const dim3 grid((unsigned)S.nblocks_padded);
  if (m->etype == AKX_TET4)
    hipLaunchKernelGGL(k_tet4_step<LAW>, grid, dim3((unsigned)(S.max_elems + 63) / 64 * 64),
                       m->step_lds, m->stream, S);
  else
    hipLaunchKernelGGL(k_hex8_step<LAW>, grid, dim3(STEP_HEX_EPB * 8), m->step_lds, m->stream,
                       S);
}

void launch_small_step(akx_model *m, bool first, bool last) {
  Material &mat = *m->mats[0];
  const bool f32 = m->precision == AKX_PRECISION_FP32;
  StepArgs S = m->step;
  S.first = first;
  S.last = last;
  S.X = m->X.p;
  S.u = m->u.p;
  S.v = m->v.p;
  S.a = m->a.p;
  S.cu = m->cu.p;
  S.cv = m->cv.p;
  const bool new_u = first || !last; // the last step has no predictor to follow
  S.u2 = new_u ? m->u2.p : nullptr;
  S.v2 = first ? m->v2.p : m->v.p;
  S.a2 = first ? m->a2.p : m->a.p;
  S.cu2 = first ? m->cu2.p : m->cu.p;
  S.cv2 = first ? m->cv2.p : m->cv.p;
  S.mass = m->mass.p;
  S.fext = m->has_fext ? m->fext.p : nullptr;
  S.blocked = m->blocked.p;
  S.fint = last ? m->fint.p : nullptr;
  S.dt = m->dt;
  S.lambda = mat.lambda;
  S.mu = mat.mu;
  S.lam_el = mat.per_element ? mat.lam_el.p : nullptr;
  S.mu_el = mat.per_element ? mat.mu_el.p : nullptr;
  S.lm_f = mat.per_element ? mat.lm_f.p : nullptr;
  if (mat.law == AKX_LAW_PLASTIC_LIH) {
    const ElemArgs A = elem_args(m, mat, false);
    check_elem_args(A, mat.law);
    S.sigma_y = A.sigma_y;
    S.h = A.h;
    S.sy_el = A.sy_el;
    S.h_el = A.h_el;
    S.hist = qp_view(A, 1);
  }
  S.jw = m->jw.p;
  require(S.lnode && S.onode && S.lc && S.X && S.mass && S.blocked && S.u && m->u2.p && S.v2 && S.a2,
          "small-model step launched without its lists or state");
  require(!f32 || (S.run && S.cu && S.cv && m->cu2.p && m->cv2.p),
          "small-model step launched without compensation terms");
  require(!S.lam_el == !S.mu_el && (!f32 || !S.lam_el == !S.lm_f),
          "per-element parameters incomplete");
  require(m->etype != AKX_HEX8 || f32 || S.jw, "Hex8 step launched without its jacobian table");
  if (f32)
    HIPCHECK(akxf::launch_step(m->etype, mat.law, S, m->step_lds, m->stream));
  else if (mat.law == AKX_LAW_ELASTIC)
    launch_step_law<LAW_ELASTIC>(m, S);
  else if (mat.law == AKX_LAW_ELASTIC_FD)
    launch_step_law<LAW_ELASTIC_FD>(m, S);
  else if (mat.law == AKX_LAW_NEOHOOKEAN)
    launch_step_law<LAW_NEOHOOKEAN>(m, S);
  else {
    require(m->etype == AKX_TET4, "plastic Hex8 steps take two launches");
    hipLaunchKernelGGL(k_tet4_step<LAW_PLASTIC>, dim3((unsigned)S.nblocks_padded),
                       dim3((unsigned)(S.max_elems + 63) / 64 * 64), m->step_lds, m->stream, S);
  }
  HIPCHECK(hipGetLastError());
  flip_plastic_state(m);
  if (new_u)
    std::swap(m->u, m->u2);
  if (first) {
    std::swap(m->v, m->v2);
    std::swap(m->a, m->a2);
    std::swap(m->cu, m->cu2);
    std::swap(m->cv, m->cv2);
  }
}

// ---------------------------------------------------------------------------
// Pipelined step (opt-in): the elements are cut in P consecutive parts and the
// nodes in P groups, group q = the 256-node slices whose last element (in
// assembly order) lies in part q.  Then
//   gather of group q (step k)        needs the element pass of parts <= q
//   element part p (step k + 1)       needs the gather of the groups its nodes
//                                     belong to (the last is pipe_need[p])
// so the memory-bound gather of group q runs on a second stream while the
// compute-bound element pass of part q + 1 runs.  Values and summation
// orders are those of the plain schedule: it reorders launches, not
// arithmetic.  Planned only for one contiguous non-plastic material whose
// slice groups are monotone (otherwise the plain schedule is used).
// ---------------------------------------------------------------------------
// a change of the materials' inputs re-decides whether the pipelined
// schedule applies
void refresh_pipeline_plan(akx_model *m) { m->pipe_planned = false; }

void plan_pipeline(akx_model *m) {
  m->pipe_planned = true;
  m->pipe_ok = false;
  const int P = m->pipe_parts;
  if (P < 2 || m->mats.size() != 1 || m->bpa || m->mats[0]->ext() || m->mats[0]->dlaw)
    return;
  Material &mat = *m->mats[0];
  if (!mat.contiguous || mat.law == AKX_LAW_PLASTIC_LIH || mat.first != 0 ||
      mat.n != m->nel || mat.pos_offset != 0 || m->nel < P)
    return;
  const int64_t nel = m->nel, nn = m->nn, nnpe = m->nnpe;
  auto part_of = [&](int64_t e) { return (int)(e * P / nel); };
  std::vector<int64_t> maxel(nn, -1);
  for (int64_t e = 0; e < nel; ++e)
    for (int a = 0; a < nnpe; ++a) {
      const int32_t nd = m->conn_host[e * nnpe + a];
      maxel[nd] = std::max<int64_t>(maxel[nd], e);
    }
  const int64_t nsl = (nn + 255) / 256;
  std::vector<int> lp(nsl, 0);
  int last = 0;
  for (int64_t s = 0; s < nsl; ++s) {
    int v = -1;
    for (int64_t n = s * 256; n < std::min<int64_t>(nn, s * 256 + 256); ++n)
      if (maxel[n] >= 0)
        v = std::max(v, part_of(maxel[n]));
    if (v < 0)
      v = last;
    if (v < last)
      return; // groups would not be contiguous node ranges
    lp[s] = last = v;
  }
  m->pipe_el.assign(P + 1, 0);
  m->pipe_node.assign(P + 1, nn);
  for (int p = 0; p <= P; ++p)
    m->pipe_el[p] = (int64_t)p * nel / P;
  // part boundaries must agree with part_of
  for (int p = 0; p < P; ++p)
    if (m->pipe_el[p] < m->pipe_el[p + 1] && part_of(m->pipe_el[p]) != p)
      return;
  m->pipe_node[0] = 0;
  for (int p = 1; p < P; ++p) {
    int64_t s = 0;
    while (s < nsl && lp[s] < p)
      ++s;
    m->pipe_node[p] = std::min<int64_t>(nn, s * 256);
  }
  m->pipe_node[P] = nn;
  m->pipe_need.assign(P, 0);
  for (int p = 0; p < P; ++p) {
    int64_t smax = 0;
    for (int64_t e = m->pipe_el[p]; e < m->pipe_el[p + 1]; ++e)
      for (int a = 0; a < nnpe; ++a)
        smax = std::max<int64_t>(smax, m->conn_host[e * nnpe + a] / 256);
    m->pipe_need[p] = lp[smax];
  }
  if (!m->stream2)
    HIPCHECK(hipStreamCreateWithFlags(&m->stream2, hipStreamNonBlocking));
  auto make = [&](std::vector<hipEvent_t> &v) {
    while ((int)v.size() < P) {
      hipEvent_t e;
      HIPCHECK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
      v.push_back(e);
    }
  };
  make(m->ev_elem);
  make(m->ev_gather[0]);
  make(m->ev_gather[1]);
  m->pipe_ok = true;
  if (!m->xu_static) // the partial launches read the records: bring u in
    refresh_xu(m, false);
}

void launch_element_part(akx_model *m, int p) {
  Material &mat = *m->mats[0];
  const int64_t e0 = m->pipe_el[p], cnt = m->pipe_el[p + 1] - e0;
  if (cnt <= 0)
    return;
  const bool strict = m->precision == AKX_PRECISION_FP64;
  ElemArgs A = elem_args(m, mat, false);
  A.n = cnt;
  A.first = mat.first + e0;
  A.pos_offset = mat.pos_offset + e0;
  if (A.lm_f)
    A.lm_f += e0;
  A.lconn = nullptr; // the block node lists follow the whole range's blocks
  if (A.lam_el) {
    A.lam_el += e0;
    A.mu_el += e0;
  }
  if (A.sy_el)
    A.sy_el += e0;
  if (A.h_el)
    A.h_el += e0;
  int64_t epb = strict ? (m->etype == AKX_HEX8 ? HEX_STRICT_EPB : TPB)
                       : akxf::elements_per_block(m->etype);
  A.nblocks_padded = ((cnt + epb - 1) / epb + 7) / 8 * 8;
  check_elem_args(A, mat.law);
  require(m->etype != AKX_TET4 || A.xu != nullptr, "Tet4 element pass without its node records");
  if (strict) {
    if (m->etype == AKX_TET4)
      launch_elem_law<ET_TET4, double, double>(m, mat, A);
    else
      launch_hex8_strict(m, mat, A);
  } else {
    HIPCHECK(akxf::launch_elements(m->etype, mat.law, m->precision == AKX_PRECISION_FP32,
                                   A, m->stream));
  }
}

void launch_gather_group(akx_model *m, int p, bool predict) {
  GatherArgs G = gather_args(m, true);
  if (predict)
    G.fint = nullptr; // stored by the last step only (launch_gather)
  G.node0 = m->pipe_node[p];
  G.node_end = m->pipe_node[p + 1];
  if (G.node_end <= G.node0)
    return;
  G.nblocks_padded = padded_blocks(G.node_end - G.node0);
  const bool f64 = m->precision != AKX_PRECISION_FP32;
  check_gather_args(G, true, !f64);
  launch_gather_kernel(G, f64, true, predict, m->stream2);
  HIPCHECK(hipGetLastError());
}

void solve_pipelined(akx_model *m, int64_t nb_steps) {
  const int P = m->pipe_parts;
  launch_predictor(m);
  for (int64_t s = 0; s < nb_steps; ++s) {
    const int cur = (int)(s & 1), prev = cur ^ 1;
    for (int p = 0; p < P; ++p) {
      if (s > 0) // the gather of the previous step on this part's nodes
        HIPCHECK(hipStreamWaitEvent(m->stream, m->ev_gather[prev][m->pipe_need[p]], 0));
      launch_element_part(m, p);
      HIPCHECK(hipEventRecord(m->ev_elem[p], m->stream));
      HIPCHECK(hipStreamWaitEvent(m->stream2, m->ev_elem[p], 0));
      launch_gather_group(m, p, s + 1 < nb_steps);
      HIPCHECK(hipEventRecord(m->ev_gather[cur][p], m->stream2));
    }
  }
  // join: the model's stream ends after the last gather
  HIPCHECK(hipStreamWaitEvent(m->stream, m->ev_gather[(nb_steps - 1) & 1][P - 1], 0));
}

// Bytes one launch of a kernel class cannot do without
double kernel_bytes(const akx_model *m, int kernel_class) {
  const double s_node = 8.0; // FP64 nodal state
  const double s_f = (double)m->fe_elem_size();
  int64_t nel_all = 0;
  double extra = 0.;
  for (auto &mp : m->mats) {
    nel_all += mp->n;
    if (mp->per_element) // lambda, mu per element: FP64, or the FP32 pair
      extra += mp->n * (mp->lm_f.p ? 2.0 * 4.0 : 2.0 * 8.0);
    if (mp->lconn.p) // staged records: 2-byte local
      // corners instead of 4-byte node ids, plus the blocks' node lists
      extra += -2.0 * m->nnpe * mp->n + 4.0 * (double)mp->bl_nodes.n;
    if (mp->law == AKX_LAW_PLASTIC_LIH)
      extra += (double)mp->n * m->nqp * (2 * (9 + 9 + 9 + 1) * 8.0); // read + write history
    if (!mp->contiguous)
      extra += mp->n * 4.0;
  }
  // table entries the element pass writes and the gather reads: one per
  // element corner, or one per (block, distinct node) partial
  double entries = (double)nel_all * m->nnpe;
  if (m->bpa) {
    const double partials = (double)m->bp_entries;
    // corner slots (2 B) instead of table positions (4 B); per partial its
    // slot offset (2 B) and table position (4 B)
    extra += -2.0 * m->nnpe * nel_all + 6.0 * partials;
    entries = partials;
  } else if (m->ppa) {
    // corner codes (4 B, as the positions); per summed run its slot end
    // (2 B) and table position (4 B)
    extra += 6.0 * (double)m->pp_runs;
    entries = (double)m->pp_entries;
  }
  switch (kernel_class) {
  case 0: // element pass: connectivity + table entries, X and u once per
          // node, r_e write; with the Hex8 jacobian table, the table (80 B
          // per Gauss point) instead of X
    if (m->jw.p)
      return nel_all * (8.0 * m->nnpe + 80.0 * m->nqp) + entries * 3.0 * s_f +
             m->nn * 3.0 * s_node + extra;
    return nel_all * 8.0 * m->nnpe + entries * 3.0 * s_f +
           m->nn * (3.0 * s_node + 3.0 * s_node) + extra;
  case 1: { // gather + update of a step followed by another: degree, r_e
            // read, mass, blocked, a/v read+write, u read+write (fused
            // predictor); the last step of a call also writes f_int.  The
            // FP32 form reads and writes no a between the steps of a call
            // (its velocity array holds the half-step velocity), and its
            // compensation terms
    const bool f32 = m->precision == AKX_PRECISION_FP32;
    double per_node = 4.0 + s_node /*M*/ + 1.0 + (m->records_live() ? 3 * s_node : 0.) /*u records*/ +
                      (f32 ? 0. : 2 * 3 * s_node) /*a*/ + 2 * 3 * s_node /*v*/ +
                      2 * 3 * s_node /*u*/ + (m->has_fext ? 3 * s_node : 0.);
    if (f32)
      per_node += 2 * 2 * 3 * 4.0; // compensation terms read + write
    return entries * (3.0 * s_f) + m->nn * (per_node - 3.0);
  }
  case 2:
    return m->nn * (1.0 + 3 * s_node + 2 * 2 * 3 * s_node);
  default:
    throw Error(AKX_ERR_INVALID, "bad kernel class");
  }
}

InitArgs init_args(akx_model *m, Material *mat) {
  InitArgs A{};
  A.nel = m->nel;
  A.nn = m->nn;
  A.conn = m->conn.p;
  A.X = m->X.p;
  A.u = m->u.p;
  if (mat) {
    A.n = mat->n;
    A.first = mat->first;
    A.pos_offset = mat->pos_offset;
    A.filter = mat->contiguous ? nullptr : mat->filter.p;
    A.rho = mat->rho;
    A.lambda = mat->lambda;
    A.mu = mat->mu;
    A.lam_el = mat->per_element ? mat->lam_el.p : nullptr;
    A.mu_el = mat->per_element ? mat->mu_el.p : nullptr;
  }
  return A;
}

void check_ready(akx_model *m) {
  require(m != nullptr, "null model");
  require(m->initialized, "initFull has not been called");
}

// Gather table.  Every (element position p, local node a) gets an entry of a
// node-major sliced-ELL table: nodes are cut in slices of 256, slice s has
// width w_s = its largest node degree and starts at ell_off[s]; the entry of
// the d-th element of node n is ell_off[s] + d*256 + n%256.  Elements are
// ranked per node in ascending assembly order -- materials in creation
// order, each material's filter in order -- which is the order of the
// reference's sequential scatter (dof_manager.cc:92-114, called per material
// by material.cc:98-120).  MeshUtils::buildNode2Elements
// (mesh_utils.cc:37-82) builds the same node -> element lists.
void build_gather_table(akx_model *m) {
  int64_t nslots = 0;
  for (auto &mp : m->mats)
    nslots += mp->n * m->nnpe;
  require(nslots < (int64_t)INT32_MAX, "too many element slots for int32 indices");
  std::vector<int32_t> deg(m->nn, 0);
  for (auto &mp : m->mats)
    for (int64_t i = 0; i < mp->n; ++i) {
      int64_t e = mp->contiguous ? mp->first + i : mp->filter_host[i];
      for (int a = 0; a < m->nnpe; ++a)
        deg[m->conn_host[e * m->nnpe + a]]++;
    }
  const int64_t nslices = (m->nn + 255) / 256;
  std::vector<int64_t> off(nslices + 1, 0);
  for (int64_t sl = 0; sl < nslices; ++sl) {
    int w = 0;
    for (int64_t n = sl * 256; n < std::min<int64_t>(m->nn, sl * 256 + 256); ++n)
      w = std::max(w, deg[n]);
    require(w <= 255, "a node belongs to more than 255 elements");
    off[sl + 1] = off[sl] + (int64_t)w * 256;
  }
  m->ell_total = off[nslices];
  require(m->ell_total < (int64_t)INT32_MAX, "element force table too large for int32");
  std::vector<int32_t> fill(m->nn, 0), pos(std::max<int64_t>(nslots, 1));
  for (auto &mp : m->mats)
    for (int64_t i = 0; i < mp->n; ++i) {
      int64_t e = mp->contiguous ? mp->first + i : mp->filter_host[i];
      int64_t p = mp->pos_offset + i;
      for (int a = 0; a < m->nnpe; ++a) {
        int32_t node = m->conn_host[e * m->nnpe + a];
        int32_t d = fill[node]++;
        pos[p * m->nnpe + a] = (int32_t)(off[node >> 8] + (int64_t)d * 256 + (node & 255));
      }
    }
  std::vector<uint8_t> deg8(m->nn);
  for (int64_t n = 0; n < m->nn; ++n)
    deg8[n] = (uint8_t)deg[n];
  m->pos.alloc(pos.size());
  m->ell_off.alloc(off.size());
  m->deg.alloc(m->nn);
  HIPCHECK(hipMemcpy(m->pos.p, pos.data(), pos.size() * sizeof(int32_t),
                     hipMemcpyHostToDevice));
  HIPCHECK(hipMemcpy(m->ell_off.p, off.data(), off.size() * sizeof(int64_t),
                     hipMemcpyHostToDevice));
  HIPCHECK(hipMemcpy(m->deg.p, deg8.data(), m->nn, hipMemcpyHostToDevice));
}

void alloc_internals(akx_model *m, Material &mat) {
  int64_t nq = mat.n * m->nqp;
  if (mat.law == AKX_LAW_PLASTIC_LIH) {
    for (int s = 0; s < 2; ++s) {
      mat.hgrad[s].alloc(9 * nq);
      mat.hsig[s].alloc(9 * nq);
      mat.heps[s].alloc(9 * nq);
      mat.hiso[s].alloc(nq);
      mat.hpe[s].alloc(nq);
      zero_async(m, mat.hgrad[s].p, 9 * nq);
      zero_async(m, mat.hsig[s].p, 9 * nq);
      zero_async(m, mat.heps[s].p, 9 * nq);
      zero_async(m, mat.hiso[s].p, nq);
      zero_async(m, mat.hpe[s].p, nq);
    }
    mat.cur = 0;
  }
}

} // namespace

// ---------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------
extern "C" {

const char *akx_last_error(void) { return g_last_error.c_str(); }

int akx_version(void) { return 100; }

int akx_device_count(int *count) {
  return guard([&] {
    require(count != nullptr, "null count");
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess)
      n = 0;
    int good = 0;
    for (int d = 0; d < n; ++d) {
      hipDeviceProp_t p;
      if (hipGetDeviceProperties(&p, d) == hipSuccess &&
          std::strncmp(p.gcnArchName, "gfx950", 6) == 0)
        ++good;
    }
    *count = good;
  });
}

int akx_model_create(int device, akx_model **out) {
  return guard([&] {
    require(out != nullptr, "null output pointer");
    auto m = std::make_unique<akx_model>();
    m->device = device;
    m->set_device();
    hipDeviceProp_t p;
    HIPCHECK(hipGetDeviceProperties(&p, device));
    if (std::strncmp(p.gcnArchName, "gfx950", 6) != 0)
      throw Error(AKX_ERR_UNSUPPORTED,
                  std::string("device is not gfx950: ") + p.gcnArchName);
    HIPCHECK(hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking));
    (void)device_scratch(device); // the no-allocation energy's array on this device
    m->scratch_u64.alloc(4);
    m->scratch_i64.alloc(4);
    *out = m.release();
  });
}

int akx_model_destroy(akx_model *m) {
  return guard([&] {
    if (!m)
      return;
    (void)hipSetDevice(m->device);
    if (m->stream)
      (void)hipStreamSynchronize(m->stream);
    delete m;
  });
}

int akx_model_set_mesh(akx_model *m, int element_type, int64_t nb_nodes,
                       const double *nodes, int64_t nb_elements,
                       const int32_t *connectivity) {
  return guard([&] {
    require(m != nullptr, "null model");
    require(!m->initialized, "mesh already initialised");
    require(element_type == AKX_TET4 || element_type == AKX_HEX8,
            "element type must be _tetrahedron_4 or _hexahedron_8");
    require(nb_nodes > 0 && nb_elements > 0, "empty mesh");
    require(nb_nodes < INT32_MAX, "too many nodes for int32 connectivity");
    require(nodes && connectivity, "null mesh arrays");
    m->set_device();
    m->etype = element_type;
    m->nnpe = element_type == AKX_TET4 ? 4 : 8;
    m->nqp = element_type == AKX_TET4 ? 1 : 8;
    m->nn = nb_nodes;
    m->nel = nb_elements;
    m->conn_host.assign(connectivity, connectivity + nb_elements * m->nnpe);
    for (int32_t c : m->conn_host)
      require(c >= 0 && c < nb_nodes, "connectivity refers to a missing node");
    m->X.alloc(3 * nb_nodes);
    const int64_t per = state_stride(nb_nodes);
    const bool twice = nb_nodes <= STEP_NODES_MAX;
    m->state.alloc((twice ? 6 : 3) * per);
    double *part = m->state.p;
    for (auto *f : {&m->u, &m->v, &m->a, &m->u2, &m->v2, &m->a2}) {
      f->p = part < m->state.p + m->state.n ? part : nullptr;
      part += per;
    }
    m->fint.alloc(3 * nb_nodes);
    m->mass.alloc(nb_nodes);
    m->blocked.alloc(nb_nodes);
    m->conn.alloc(nb_elements * m->nnpe);
    upload_soa(m, nodes, m->X.p, nb_nodes, 3);
    HIPCHECK(hipMemcpy(m->conn.p, connectivity,
                       nb_elements * m->nnpe * sizeof(int32_t),
                       hipMemcpyHostToDevice));
    zero_async(m, m->state.p, (int64_t)m->state.n);
    zero_async(m, m->fint.p, 3 * nb_nodes);
    zero_async(m, m->mass.p, nb_nodes);
    HIPCHECK(hipMemsetAsync(m->blocked.p, 0, nb_nodes, m->stream));
    if (m->etype == AKX_HEX8)
      upload_hex8_tables();
    HIPCHECK(hipStreamSynchronize(m->stream));
  });
}

int akx_material_law_by_name(const char *name, int finite_deformation, int *law) {
  return guard([&] {
    require(name && law, "null argument");
    std::string s(name);
    if (s == "elastic")
      *law = finite_deformation ? AKX_LAW_ELASTIC_FD : AKX_LAW_ELASTIC;
    else if (s == "neohookean")
      *law = AKX_LAW_NEOHOOKEAN;
    else if (s == "plastic_linear_isotropic_hardening") {
      // The reference's finite-deformation branch (material_linear_isotropic
      // _hardening.cc:36-52, _inline_impl.hh:88-186) is not provided: refuse
      // it rather than run the small-strain law in its place.
      if (finite_deformation)
        throw Error(AKX_ERR_UNSUPPORTED,
                    "plastic_linear_isotropic_hardening with finite_deformation = true "
                    "is not provided (small-strain plasticity only)");
      *law = AKX_LAW_PLASTIC_LIH;
    } else
      throw Error(AKX_ERR_UNSUPPORTED, "unknown material law: " + s);
  });
}

int akx_model_add_material(akx_model *m, int law, const double *params,
                           int nparams, const int32_t *filter,
                           int64_t nb_filter, int *material_id) {
  return guard([&] {
    require(m != nullptr && m->etype >= 0, "set the mesh first");
    require(!m->initialized, "materials must be added before initFull");
    require(law >= AKX_LAW_ELASTIC && law <= AKX_LAW_USER_FD, "unknown law");
    require(params && nparams >= 3, "params = {rho, E, nu[, sigma_y, h]}");
    m->set_device();
    auto mat = std::make_unique<Material>();
    mat->law = law;
    mat->rho = params[0];
    mat->E = params[1];
    mat->nu = params[2];
    mat->sigma_y = nparams > 3 ? params[3] : 0.;
    mat->h = nparams > 4 ? params[4] : 0.;
    require(mat->rho > 0, "rho must be positive");
    lame(mat->E, mat->nu, mat->lambda, mat->mu);
    int64_t pos = 0;
    for (auto &o : m->mats)
      pos += o->n;
    mat->pos_offset = pos;
    if (filter == nullptr) {
      mat->n = m->nel;
      mat->first = 0;
      mat->contiguous = true;
    } else {
      require(nb_filter >= 0, "negative filter size");
      mat->n = nb_filter;
      mat->filter_host.assign(filter, filter + nb_filter);
      bool contig = true;
      for (int64_t i = 0; i < nb_filter; ++i) {
        require(filter[i] >= 0 && filter[i] < m->nel, "filter refers to a missing element");
        if (filter[i] != filter[0] + i)
          contig = false;
      }
      mat->contiguous = contig;
      mat->first = nb_filter ? filter[0] : 0;
      if (!contig && nb_filter) {
        mat->filter.alloc(nb_filter);
        HIPCHECK(hipMemcpy(mat->filter.p, filter, nb_filter * sizeof(int32_t),
                           hipMemcpyHostToDevice));
      }
    }
    if (material_id)
      *material_id = (int)m->mats.size();
    m->mats.push_back(std::move(mat));
  });
}

int akx_model_set_element_parameters(akx_model *m, int material_id,
                                     const double *E, const double *nu,
                                     const double *sigma_y, const double *h) {
  return guard([&] {
    require(m != nullptr, "null model");
    require(material_id >= 0 && material_id < (int)m->mats.size(), "bad material id");
    m->set_device();
    Material &mat = *m->mats[material_id];
    int64_t n = mat.n;
    if (n == 0)
      return;
    auto up = [&](DevBuf<double> &b, const double *src) {
      b.alloc(n);
      HIPCHECK(hipMemcpy(b.p, src, n * sizeof(double), hipMemcpyHostToDevice));
    };
    if (E || nu) {
      mat.E_el_host.assign(n, mat.E);
      mat.nu_el_host.assign(n, mat.nu);
      if (E)
        mat.E_el_host.assign(E, E + n);
      if (nu)
        mat.nu_el_host.assign(nu, nu + n);
      DevBuf<double> dE, dnu;
      if (E)
        up(dE, E);
      if (nu)
        up(dnu, nu);
      mat.lam_el.alloc(n);
      mat.mu_el.alloc(n);
      hipLaunchKernelGGL(k_lame, dim3(grid_for(n)), dim3(TPB), 0, m->stream,
                         (const double *)dE.p, (const double *)dnu.p, mat.E,
                         mat.nu, mat.lam_el.p, mat.mu_el.p, n);
      HIPCHECK(hipGetLastError());
      mat.per_element = true;
      if (m->precision == AKX_PRECISION_FP32)
        fill_lame_f32(m, mat);
      HIPCHECK(hipStreamSynchronize(m->stream));
    }
    if (sigma_y)
      up(mat.sy_el, sigma_y);
    if (h)
      up(mat.h_el, h);
  });
}

int akx_model_set_eigen_grad_u(akx_model *m, int material_id, const double *eigen_grad_u) {
  return guard([&] {
    require(m != nullptr && m->etype >= 0, "set the mesh first");
    require(material_id >= 0 && material_id < (int)m->mats.size(), "bad material id");
    if (m->precision != AKX_PRECISION_FP64)
      throw Error(AKX_ERR_UNSUPPORTED, "eigen_grad_u runs on the plain FP64 path");
    m->set_device();
    Material &mat = *m->mats[material_id];
    if (!eigen_grad_u || mat.n == 0) {
      mat.eig.release();
      return;
    }
    const int64_t nq = mat.n * m->nqp;
    mat.eig.alloc(9 * nq);
    upload_soa(m, eigen_grad_u, mat.eig.p, nq, 9);
    refresh_pipeline_plan(m);
  });
}

int akx_model_set_thermal(akx_model *m, int material_id, double alpha, const double *delta_T) {
  return guard([&] {
    require(m != nullptr && m->etype >= 0, "set the mesh first");
    require(material_id >= 0 && material_id < (int)m->mats.size(), "bad material id");
    if (m->precision != AKX_PRECISION_FP64)
      throw Error(AKX_ERR_UNSUPPORTED, "thermal stresses run on the plain FP64 path");
    m->set_device();
    Material &mat = *m->mats[material_id];
    if (!delta_T || mat.n == 0) {
      mat.sth_now.release();
      return;
    }
    require(std::isfinite(alpha), "non-finite alpha");
    const int64_t nq = mat.n * m->nqp;
    // sigma_th = -E / (1 - 2 nu) * alpha * delta_T (material_thermal.hh:91-95)
    std::vector<double> sth(nq);
    for (int64_t i = 0; i < mat.n; ++i) {
      const double E = mat.E_el_host.empty() ? mat.E : mat.E_el_host[i];
      const double nu = mat.nu_el_host.empty() ? mat.nu : mat.nu_el_host[i];
      for (int q = 0; q < m->nqp; ++q)
        sth[i * m->nqp + q] = -E / (1. - 2. * nu) * alpha * delta_T[i * m->nqp + q];
    }
    mat.sth_now.alloc(nq);
    HIPCHECK(hipMemcpy(mat.sth_now.p, sth.data(), nq * sizeof(double), hipMemcpyHostToDevice));
    if (mat.law == AKX_LAW_PLASTIC_LIH && !mat.hsth[0].p) {
      // the history starts at zero (material_thermal.cc:34)
      for (int k = 0; k < 2; ++k) {
        mat.hsth[k].alloc(nq);
        zero_async(m, mat.hsth[k].p, nq);
      }
      HIPCHECK(hipStreamSynchronize(m->stream));
    }
    refresh_pipeline_plan(m);
  });
}

int akx_model_set_precision(akx_model *m, int precision) {
  return guard([&] {
    require(m != nullptr, "null model");
    require(!m->initialized, "precision must be set before initFull");
    for (auto &mp : m->mats)
      require(precision == AKX_PRECISION_FP64 || !mp->ext(),
              "eigen_grad_u and thermal stresses run on the plain FP64 path");
    require(precision == AKX_PRECISION_FP64 || precision == AKX_PRECISION_FP32 ||
                precision == AKX_PRECISION_FP64_FAST,
            "unknown precision");
    m->precision = precision;
  });
}

int akx_model_set_block_assembly(akx_model *m, int enable) {
  return guard([&] {
    require(m != nullptr, "null model");
    require(!m->initialized, "the assembly must be chosen before initFull");
    require(enable >= AKX_ASSEMBLY_PER_CORNER && enable <= AKX_ASSEMBLY_BLOCK_PARTIALS,
            "assembly must be AKX_ASSEMBLY_PER_CORNER, _DEFAULT or _BLOCK_PARTIALS");
    m->assembly = enable;
  });
}

int akx_model_get_block_assembly(akx_model *m, int *active) {
  return guard([&] {
    check_ready(m);
    require(active != nullptr, "null output");
    *active = m->bpa ? AKX_ASSEMBLY_BLOCK_PARTIALS
              : m->ppa ? (m->assembly == AKX_ASSEMBLY_BLOCK_PARTIALS ? AKX_ASSEMBLY_BLOCK_PARTIALS
                                                                     : AKX_ASSEMBLY_PREFIX_PARTIALS)
                       : AKX_ASSEMBLY_PER_CORNER;
  });
}

int akx_model_init_full(akx_model *m) {
  return guard([&] {
    require(m != nullptr && m->etype >= 0, "set the mesh first");
    require(!m->initialized, "initFull called twice");
    require(!m->mats.empty(), "no material");
    require(!m->has_user() || m->precision == AKX_PRECISION_FP64,
            "user materials run on the plain FP64 path");
    m->set_device();
    for (auto &mp : m->mats)
      if (mp->user()) { // the internals the plugin reads and writes
        mp->grad.alloc(9 * mp->n * m->nqp);
        mp->stress.alloc(9 * mp->n * m->nqp);
      }
    // IntegratorGauss::checkJacobians
    {
      InitArgs A = init_args(m, nullptr);
      long long init = INT64_MAX;
      HIPCHECK(hipMemcpy(m->scratch_i64.p, &init, sizeof(init), hipMemcpyHostToDevice));
      A.first_bad = m->scratch_i64.p;
      if (m->etype == AKX_TET4)
        hipLaunchKernelGGL(k_check_jacobians<ET_TET4>, dim3(grid_for(m->nel)),
                           dim3(TPB), 0, m->stream, A);
      else
        hipLaunchKernelGGL(k_check_jacobians<ET_HEX8>, dim3(grid_for(m->nel)),
                           dim3(TPB), 0, m->stream, A);
      HIPCHECK(hipGetLastError());
      long long bad = 0;
      HIPCHECK(hipMemcpyAsync(&bad, m->scratch_i64.p, sizeof(bad),
                              hipMemcpyDeviceToHost, m->stream));
      HIPCHECK(hipStreamSynchronize(m->stream));
      if (bad != INT64_MAX) {
        char msg[256];
        std::snprintf(msg, sizeof msg,
                      "Negative jacobian computed, possible problem in the "
                      "element node ordering (Quadrature Point %lld:%lld)",
                      bad % m->nqp, bad / m->nqp);
        throw Error(AKX_ERR_JACOBIAN, msg);
      }
    }
    // FEEngine precompute of the plain FP64 Hex8 pass: J^-1 and w det J per
    // Gauss point (fe_engine_template_tmpl.hh:98-120)
    if (m->etype == AKX_HEX8 && m->precision == AKX_PRECISION_FP64 && m->nel > 0) {
      const int64_t nq = m->nel * 8;
      m->jw.alloc(5 * nq);
      hipLaunchKernelGGL(k_hex8_jacobian_table, dim3(grid_for(nq)), dim3(TPB), 0,
                         m->stream, (const int32_t *)m->conn.p, (const double *)m->X.p,
                         m->nn, m->nel, m->jw.p);
      HIPCHECK(hipGetLastError());
    }
    if (m->etype == AKX_TET4 && m->nn > 0) {
      m->xu.alloc(6 * m->nn);
      refresh_xu(m, true);
      for (auto &mp : m->mats) // Tet4 passes with staged node records
        if (mp->contiguous && mp->n > 0 && m->precision != AKX_PRECISION_FP64_FAST)
          build_block_nodes(m, *mp);
      m->xu_static = m->precision == AKX_PRECISION_FP64_FAST;
      for (auto &mp : m->mats)
        m->xu_static = m->xu_static || (mp->n > 0 && (!mp->contiguous || mp->user()));
      bool ppa = m->assembly != AKX_ASSEMBLY_PER_CORNER &&
                 m->precision == AKX_PRECISION_FP64 && !m->has_user();
      for (auto &mp : m->mats)
        ppa = ppa && mp->contiguous && mp->n > 0 && mp->lconn.p != nullptr;
      if (ppa)
        build_ppa(m, m->assembly == AKX_ASSEMBLY_BLOCK_PARTIALS);
      m->ppa = ppa;
    }
    if (m->etype == AKX_HEX8 && m->precision == AKX_PRECISION_FP32 && m->nn > 0 &&
        m->assembly != AKX_ASSEMBLY_PER_CORNER)
      for (auto &mp : m->mats) // FP32 Hex8 block partials
        if (mp->contiguous && mp->n > 0)
          build_block_nodes(m, *mp, akxf::elements_per_block(AKX_HEX8, true));
    build_gather_table(m);
    m->bpa = m->assembly != AKX_ASSEMBLY_PER_CORNER && m->precision == AKX_PRECISION_FP32 &&
             m->nn > 0;
    for (auto &mp : m->mats)
      m->bpa = m->bpa && mp->contiguous && mp->n > 0 && mp->lslot.p != nullptr;
    if (m->bpa)
      build_bpa_table(m);
    m->fe.alloc(std::max<int64_t>(std::max(m->ell_total, m->bp_total), 1) * 3 *
                m->fe_elem_size());
    // lumped mass
    {
      DevBuf<double> me;
      me.alloc(std::max<int64_t>(m->ell_total, 1));
      for (auto &mp : m->mats) {
        if (mp->n == 0)
          continue;
        InitArgs A = init_args(m, mp.get());
        A.me = me.p;
        A.pos = m->pos.p;
        if (m->etype == AKX_TET4)
          hipLaunchKernelGGL(k_mass_elements<ET_TET4>, dim3(grid_for(mp->n)),
                             dim3(TPB), 0, m->stream, A);
        else
          hipLaunchKernelGGL(k_mass_elements<ET_HEX8>, dim3(grid_for(mp->n)),
                             dim3(TPB), 0, m->stream, A);
        HIPCHECK(hipGetLastError());
      }
      hipLaunchKernelGGL(k_gather_mass, dim3(grid_for(m->nn)), dim3(TPB), 0,
                         m->stream, m->nn, (const int64_t *)m->ell_off.p,
                         (const uint8_t *)m->deg.p, (const double *)me.p,
                         m->mass.p);
      HIPCHECK(hipGetLastError());
      HIPCHECK(hipStreamSynchronize(m->stream));
    }
    plan_small_steps(m);
    const double step_bytes = kernel_bytes(m, 0) + kernel_bytes(m, 1);
    bool plastic = false;
    for (auto &mp : m->mats)
      plastic = plastic || mp->law == AKX_LAW_PLASTIC_LIH;
    m->stream_loads = step_bytes > STREAM_BYTES;
    m->stream_jac = step_bytes > (plastic ? STREAM_JAC_PLASTIC : STREAM_BYTES);
    for (auto &mp : m->mats)
      alloc_internals(m, *mp);
    if (m->precision == AKX_PRECISION_FP32) {
      for (auto &mp : m->mats)
        if (mp->per_element && mp->n > 0)
          fill_lame_f32(m, *mp);
      const int64_t per = state_stride(m->nn);
      m->comp.alloc((m->step.nblocks > 0 ? 4 : 2) * per);
      float *part = m->comp.p;
      for (auto *f : {&m->cu, &m->cv, &m->cu2, &m->cv2}) {
        f->p = part < m->comp.p + m->comp.n ? part : nullptr;
        part += per;
      }
      hipLaunchKernelGGL(k_fill_f32, dim3(grid_for((int64_t)m->comp.n)), dim3(TPB), 0,
                         m->stream, m->comp.p, (int64_t)m->comp.n, 0.f);
      HIPCHECK(hipGetLastError());
    }
    HIPCHECK(hipStreamSynchronize(m->stream));
    m->initialized = true;
  });
}

int akx_model_get_stable_time_step(akx_model *m, double *dt) {
  return guard([&] {
    check_ready(m);
    require(dt != nullptr, "null output");
    m->set_device();
    unsigned long long init = 0x7FEFFFFFFFFFFFFFull; // DBL_MAX bits
    HIPCHECK(hipMemcpyAsync(m->scratch_u64.p, &init, sizeof(init),
                            hipMemcpyHostToDevice, m->stream));
    for (auto &mp : m->mats) {
      if (mp->n == 0)
        continue;
      InitArgs A = init_args(m, mp.get());
      A.min_bits = m->scratch_u64.p;
      if (m->etype == AKX_TET4)
        hipLaunchKernelGGL(k_stable_dt<ET_TET4>, dim3(grid_for(mp->n)),
                           dim3(TPB), 0, m->stream, A);
      else
        hipLaunchKernelGGL(k_stable_dt<ET_HEX8>, dim3(grid_for(mp->n)),
                           dim3(TPB), 0, m->stream, A);
      HIPCHECK(hipGetLastError());
    }
    unsigned long long bits = 0;
    HIPCHECK(hipMemcpyAsync(&bits, m->scratch_u64.p, sizeof(bits),
                            hipMemcpyDeviceToHost, m->stream));
    HIPCHECK(hipStreamSynchronize(m->stream));
    double r;
    std::memcpy(&r, &bits, sizeof(r));
    *dt = r;
  });
}

int akx_model_set_time_step(akx_model *m, double dt) {
  return guard([&] {
    require(m != nullptr, "null model");
    require(dt > 0 && std::isfinite(dt), "time step must be positive");
    m->dt = dt;
  });
}

int akx_model_solve_steps(akx_model *m, int64_t nb_steps) {
  return guard([&] {
    check_ready(m);
    require(m->dt > 0, "setTimeStep has not been called");
    require(nb_steps >= 0, "negative step count");
    if (nb_steps == 0)
      return;
    m->set_device();
    if (m->has_user()) { // the plugin runs on the host between the passes
      launch_predictor(m);
      for (int64_t s = 0; s < nb_steps; ++s) {
        user_stress_phase(m);
        launch_element_pass(m, false);
        flip_plastic_state(m);
        launch_gather(m, true, s + 1 < nb_steps);
      }
      HIPCHECK(hipStreamSynchronize(m->stream));
      return;
    }
    if (m->pipe_parts > 1 && !m->pipe_planned)
      plan_pipeline(m);
    if (m->pipe_parts > 1 && m->pipe_ok && !m->timing) {
      solve_pipelined(m, nb_steps);
      return;
    }
    if (small_steps(m)) {
      for (int64_t s = 0; s < nb_steps; ++s)
        launch_small_step(m, s == 0, s + 1 == nb_steps);
      return;
    }
    launch_predictor(m);
    for (int64_t s = 0; s < nb_steps; ++s) {
      launch_element_pass(m, false);
      flip_plastic_state(m);
      launch_gather(m, true, s + 1 < nb_steps);
    }
  });
}

// ModelSolver::solveStep(solver_id) (model_solver.cc:267-280): "" names the
// default solver, which initFull(_explicit_lumped_mass) registers as
// "explicit_lumped" (solid_mechanics_model.cc:165-169); any other id is not a
// solver of this model and fails as DOFManager::getTimeStepSolver does
// (dof_manager.cc:585-596).
int akx_model_solve_step(akx_model *m, const char *solver_id) {
  const int st = guard([&] {
    const std::string id = solver_id ? solver_id : "";
    if (!id.empty() && id != "explicit_lumped")
      throw Error(AKX_ERR_INVALID, "The non linear solver dof_manager:tss:" + id +
                                       " does not exists in dof_manager");
  });
  return st != AKX_OK ? st : akx_model_solve_steps(m, 1);
}

int akx_model_set_pipeline(akx_model *m, int parts, int *active) {
  return guard([&] {
    check_ready(m);
    require(parts >= 0 && parts <= 64, "parts must be in [0, 64]");
    m->set_device();
    HIPCHECK(hipStreamSynchronize(m->stream));
    m->pipe_parts = parts;
    m->pipe_planned = false;
    if (parts > 1)
      plan_pipeline(m);
    if (active)
      *active = parts > 1 && m->pipe_ok;
  });
}

int akx_model_assemble_internal_forces(akx_model *m) {
  return guard([&] {
    check_ready(m);
    m->set_device();
    // recompute from the previous plastic state so that calling it twice is
    // idempotent (the reference recomputes from the saved previous state)
    for (auto &mp : m->mats)
      if (mp->law == AKX_LAW_PLASTIC_LIH)
        mp->cur = 1 - mp->cur;
    user_stress_phase(m);
    launch_element_pass(m, false);
    flip_plastic_state(m);
    launch_gather(m, false, false);
    HIPCHECK(hipStreamSynchronize(m->stream));
  });
}

int akx_model_get_nb_nodes(akx_model *m, int64_t *nb_nodes) {
  return guard([&] {
    require(m && nb_nodes, "null argument");
    *nb_nodes = m->nn;
  });
}

int akx_model_get_field(akx_model *m, int field, void *host) {
  return akx_model_get_fields(m, 1, &field, &host, nullptr);
}

int akx_model_get_fields(akx_model *m, int count, const int *fields, void *const *host,
                         void *const *copy) {
  return guard([&] {
    require(m != nullptr && m->etype >= 0, "set the mesh first");
    require(count >= 0 && (count == 0 || (fields && host)), "null argument");
    m->set_device();
    std::vector<Downloader::Field> list;
    const int64_t nn = m->nn;
    hipStream_t st = m->stream;
    for (int k = 0; k < count; ++k) {
      require(host[k] != nullptr, "null host array");
      void *dst = host[k], *dup = copy ? copy[k] : nullptr;
      const double *src = nullptr;
      switch (fields[k]) {
      case AKX_FIELD_DISPLACEMENT: src = m->u.p; break;
      case AKX_FIELD_VELOCITY: src = m->v.p; break;
      case AKX_FIELD_ACCELERATION: src = m->a.p; break;
      case AKX_FIELD_INTERNAL_FORCE: src = m->fint.p; break;
      case AKX_FIELD_NODES: src = m->X.p; break;
      case AKX_FIELD_EXTERNAL_FORCE:
        if (!m->has_fext) {
          std::memset(dst, 0, sizeof(double) * 3 * nn);
          if (dup)
            std::memset(dup, 0, sizeof(double) * 3 * nn);
          continue;
        }
        src = m->fext.p;
        break;
      case AKX_FIELD_MASS: {
        const double *mass = m->mass.p;
        list.push_back({nn, 24, dst, dup, [=](void *p, int64_t first, int64_t n) {
                          hipLaunchKernelGGL(k_mass_to3, dim3(grid_for(n)), dim3(TPB), 0, st,
                                             mass, (double *)p, first, n);
                          HIPCHECK(hipGetLastError());
                        }});
        continue;
      }
      case AKX_FIELD_BLOCKED_DOFS: {
        const uint8_t *bits = m->blocked.p;
        list.push_back({nn, 3, dst, dup, [=](void *p, int64_t first, int64_t n) {
                          hipLaunchKernelGGL(k_bool3_from_bits, dim3(grid_for(n)), dim3(TPB), 0,
                                             st, bits, (uint8_t *)p, first, n);
                          HIPCHECK(hipGetLastError());
                        }});
        continue;
      }
      default:
        throw Error(AKX_ERR_INVALID, "unknown field");
      }
      list.push_back(soa_field<double>(m, src, (double *)dst, (double *)dup, nn, 3));
    }
    if (!list.empty())
      m->download.get(m->device, m->stream, list);
  });
}

int akx_host_differs(const void *a, const void *b, int64_t bytes, int *differs) {
  return guard([&] {
    require(a && b && differs && bytes >= 0, "bad arguments");
    *differs = host_differs(a, b, (size_t)bytes);
  });
}

} // extern "C"

namespace {

// BC::Neumann::FromTraction on facets (boundary_condition_tmpl.hh:100-160,
// boundary_condition_functor_inline_impl.hh:109-113): per facet
// intf(i, a) = sum_q N_a(q) t_i wJ_q, then f_ext += intf in facet order
// (dof_manager.cc:65-120).  Facet classes: _triangle_3 (one Gauss point
// (1/3, 1/3), weight 1/2; element_class_triangle_3_inline_impl.hh:52-90,
// gauss_integration.cc:56-57) and _quadrangle_4 (2 x 2 Gauss points, xi
// fastest; element_class_quadrangle_4_inline_impl.hh:64-110); surface
// jacobian |J_xi x J_eta| (element_class_tmpl.hh:352-371).  Host code: it runs
// once per boundary condition, on the facets only.
void traction_on_facets(int facet_type, int64_t nb_facets, const int32_t *conn,
                        const double *X /* [nn][3] */, int64_t nn, const double *t,
                        double *fext /* [nn][3] */) {
  const int nfn = facet_type == AKX_TRI3 ? 3 : 4, nq = facet_type == AKX_TRI3 ? 1 : 4;
  double xi[4][2], w[4];
  if (facet_type == AKX_TRI3) {
    xi[0][0] = 1. / 3.;
    xi[0][1] = 1. / 3.;
    w[0] = 1. / 2.;
  } else {
    const double g = 1. / std::sqrt(3.), pos[2] = {-g, g};
    for (int q = 0; q < 4; ++q) {
      xi[q][0] = pos[q & 1];
      xi[q][1] = pos[q >> 1];
      w[q] = 1. * 1.;
    }
  }
  for (int64_t f = 0; f < nb_facets; ++f) {
    double Xe[4][3];
    for (int a = 0; a < nfn; ++a) {
      const int32_t nd = conn[f * nfn + a];
      require(nd >= 0 && nd < nn, "facet refers to a missing node");
      for (int c = 0; c < 3; ++c)
        Xe[a][c] = X[3 * (int64_t)nd + c];
    }
    double intf[12];
    for (int q = 0; q < nq; ++q) {
      double N[4], d[2][4];
      const double x = xi[q][0], y = xi[q][1];
      if (facet_type == AKX_TRI3) {
        N[0] = 1 - x - y;
        N[1] = x;
        N[2] = y;
        d[0][0] = -1.; d[0][1] = 1.; d[0][2] = 0.;
        d[1][0] = -1.; d[1][1] = 0.; d[1][2] = 1.;
      } else {
        N[0] = 1. / 4. * (1. - x) * (1. - y);
        N[1] = 1. / 4. * (1. + x) * (1. - y);
        N[2] = 1. / 4. * (1. + x) * (1. + y);
        N[3] = 1. / 4. * (1. - x) * (1. + y);
        d[0][0] = -1. / 4. * (1. - y);
        d[0][1] = 1. / 4. * (1. - y);
        d[0][2] = 1. / 4. * (1. + y);
        d[0][3] = -1. / 4. * (1. + y);
        d[1][0] = -1. / 4. * (1. - x);
        d[1][1] = -1. / 4. * (1. + x);
        d[1][2] = 1. / 4. * (1. + x);
        d[1][3] = 1. / 4. * (1. - x);
      }
      double J[2][3];
      for (int r = 0; r < 2; ++r)
        for (int c = 0; c < 3; ++c) {
          double sum = d[r][0] * Xe[0][c];
          for (int a = 1; a < nfn; ++a)
            sum += d[r][a] * Xe[a][c];
          J[r][c] = sum;
        }
      const double cx = J[0][1] * J[1][2] - J[0][2] * J[1][1];
      const double cy = J[0][2] * J[1][0] - J[0][0] * J[1][2];
      const double cz = J[0][0] * J[1][1] - J[0][1] * J[1][0];
      const double wJ = std::sqrt(cx * cx + cy * cy + cz * cz) * w[q];
      for (int a = 0; a < nfn; ++a)
        for (int i = 0; i < 3; ++i) {
          const double v = N[a] * t[i] * wJ;
          intf[i + 3 * a] = (q == 0) ? v : intf[i + 3 * a] + v;
        }
    }
    for (int a = 0; a < nfn; ++a)
      for (int i = 0; i < 3; ++i)
        fext[3 * (int64_t)conn[f * nfn + a] + i] += 1. * intf[i + 3 * a];
  }
}

} // namespace

extern "C" {

int akx_model_apply_traction(akx_model *m, int facet_type, int64_t nb_facets,
                             const int32_t *facet_conn, const double *traction) {
  return guard([&] {
    require(m != nullptr && m->etype >= 0, "set the mesh first");
    require(facet_type == AKX_TRI3 || facet_type == AKX_QUAD4, "facet type must be "
                                                               "AKX_TRI3 or AKX_QUAD4");
    require(nb_facets >= 0 && (nb_facets == 0 || facet_conn) && traction,
            "null argument");
    for (int i = 0; i < 3; ++i)
      require(std::isfinite(traction[i]), "non-finite traction");
    m->set_device();
    HIPCHECK(hipStreamSynchronize(m->stream));
    std::vector<double> X(3 * m->nn), f(3 * m->nn, 0.);
    download_soa(m, (const double *)m->X.p, X.data(), m->nn, 3);
    if (m->has_fext)
      download_soa(m, (const double *)m->fext.p, f.data(), m->nn, 3);
    traction_on_facets(facet_type, nb_facets, facet_conn, X.data(), m->nn, traction,
                       f.data());
    m->fext.alloc(3 * m->nn);
    m->has_fext = true;
    upload_soa(m, (const double *)f.data(), m->fext.p, m->nn, 3);
  });
}

int akx_model_set_field(akx_model *m, int field, const void *host) {
  return guard([&] {
    require(m != nullptr && m->etype >= 0, "set the mesh first");
    require(host != nullptr, "null host array");
    m->set_device();
    HIPCHECK(hipStreamSynchronize(m->stream));
    double *dst = nullptr;
    switch (field) {
    case AKX_FIELD_DISPLACEMENT: dst = m->u.p; break;
    case AKX_FIELD_VELOCITY: dst = m->v.p; break;
    case AKX_FIELD_ACCELERATION: dst = m->a.p; break;
    case AKX_FIELD_EXTERNAL_FORCE: {
      const double *h = (const double *)host;
      bool any = false;
      for (int64_t i = 0; i < 3 * m->nn && !any; ++i)
        any = h[i] != 0.;
      if (!any && !m->has_fext)
        return;
      m->fext.alloc(3 * m->nn);
      m->has_fext = true;
      dst = m->fext.p;
      break;
    }
    case AKX_FIELD_BLOCKED_DOFS: {
      size_t bytes = 3 * m->nn;
      m->staging.alloc(std::max(m->staging.n, bytes));
      HIPCHECK(hipMemcpyAsync(m->staging.p, host, bytes, hipMemcpyHostToDevice,
                              m->stream));
      hipLaunchKernelGGL(k_bits_from_bool3, dim3(grid_for(m->nn)), dim3(TPB), 0,
                         m->stream, (const uint8_t *)m->staging.p, m->blocked.p,
                         m->nn);
      HIPCHECK(hipGetLastError());
      HIPCHECK(hipStreamSynchronize(m->stream));
      return;
    }
    default:
      throw Error(AKX_ERR_INVALID, "field is read only or unknown");
    }
    upload_soa(m, (const double *)host, dst, m->nn, 3);
    if (field == AKX_FIELD_DISPLACEMENT)
      refresh_xu(m, false);
  });
}

int akx_model_compute_all_stresses(akx_model *m) {
  return guard([&] {
    check_ready(m);
    m->set_device();
    for (auto &mp : m->mats) {
      int64_t nq = mp->n * m->nqp;
      if (mp->user())
        continue; // allocated at initFull, filled by the plugin
      if (mp->law != AKX_LAW_PLASTIC_LIH) {
        mp->grad.alloc(9 * nq);
        mp->stress.alloc(9 * nq);
      } else {
        mp->cur = 1 - mp->cur; // recompute the current state from the previous
      }
    }
    user_stress_phase(m);
    launch_element_pass(m, true);
    flip_plastic_state(m);
    HIPCHECK(hipStreamSynchronize(m->stream));
  });
}

int akx_model_set_device_stress(akx_model *m, int material_id, const char *source,
                                const double *params, int nparams) {
  return guard([&] {
    require(m != nullptr, "null model");
    require(material_id >= 0 && material_id < (int)m->mats.size(), "no such material");
    Material &mat = *m->mats[material_id];
    require(mat.user(), "a device law replaces the computeStress of a user material");
    require(nparams >= 0 && nparams <= 4096 && (nparams == 0 || params != nullptr),
            "device law parameters: 0 to 4096 values");
    m->set_device();
    require(m->etype >= 0, "set the mesh first");
    std::unique_ptr<DeviceLaw> law;
    if (source != nullptr)
      law = compile_device_law(m, mat, source, params, nparams);
    HIPCHECK(hipStreamSynchronize(m->stream)); // the law it replaces may be running
    mat.dlaw = std::move(law);
  });
}

int akx_model_set_stress_callback(akx_model *m, akx_compute_stress_fn fn, void *user) {
  return guard([&] {
    require(m != nullptr, "null model");
    m->stress_fn = fn;
    m->stress_user = user;
  });
}

} // extern "C"

namespace {

// Tree sum of the n values at in[] down to one (the deterministic shape of
// k_tree_sum); in and out are overwritten, out holds >= ceil(n / 2048).
// Returns the pointer to the final value.
const double *tree_reduce(akx_model *m, double *in, double *out, int64_t n) {
  while (n > 1) {
    const int64_t nb = (n + 2047) / 2048;
    hipLaunchKernelGGL(k_tree_sum, dim3((unsigned)nb), dim3(256), 0, m->stream,
                       (const double *)in, n, out);
    HIPCHECK(hipGetLastError());
    std::swap(in, out);
    n = nb;
  }
  return in;
}

double read_back(akx_model *m, const double *p) {
  double r = 0.;
  HIPCHECK(hipMemcpyAsync(&r, p, sizeof(double), hipMemcpyDeviceToHost, m->stream));
  HIPCHECK(hipStreamSynchronize(m->stream));
  return r;
}

// deterministic sum of n device values (buffer a is overwritten)
double device_sum(akx_model *m, DevBuf<double> &a, DevBuf<double> &b, int64_t n) {
  if (n == 0)
    return 0.;
  return read_back(m, tree_reduce(m, a.p, b.p, n));
}

NodeEnergyArgs node_energy_args(akx_model *m, int kind) {
  NodeEnergyArgs A{};
  A.nn = m->nn;
  A.kind = kind;
  A.v = m->v.p;
  A.mass = m->mass.p;
  A.fint = m->fint.p;
  A.fext = m->has_fext ? m->fext.p : nullptr;
  A.blocked = m->blocked.p;
  require(A.v && A.mass && (kind == 0 || (A.fint && A.blocked)), "energy inputs missing");
  return A;
}

template <int ET>
void launch_energy_elements(akx_model *m, int law, const EnergyArgs &A) {
  dim3 grid(grid_for(A.n)), block(TPB);
  switch (law) {
  case AKX_LAW_ELASTIC:
    hipLaunchKernelGGL((k_energy_elements<ET, LAW_ELASTIC>), grid, block, 0, m->stream, A);
    break;
  case AKX_LAW_ELASTIC_FD:
    hipLaunchKernelGGL((k_energy_elements<ET, LAW_ELASTIC_FD>), grid, block, 0, m->stream,
                       A);
    break;
  case AKX_LAW_NEOHOOKEAN:
    hipLaunchKernelGGL((k_energy_elements<ET, LAW_NEOHOOKEAN>), grid, block, 0, m->stream,
                       A);
    break;
  default:
    hipLaunchKernelGGL((k_energy_elements<ET, LAW_PLASTIC>), grid, block, 0, m->stream, A);
  }
  HIPCHECK(hipGetLastError());
}

// the fused first tree level: ceil(n / 2048) partial sums into out
template <int ET>
void launch_energy_elements_sum(akx_model *m, int law, const EnergyArgs &A, double *out) {
  dim3 grid((unsigned)((A.n + 2047) / 2048)), block(256);
  switch (law) {
  case AKX_LAW_ELASTIC:
    hipLaunchKernelGGL((k_energy_elements_sum<ET, LAW_ELASTIC>), grid, block, 0, m->stream,
                       A, out);
    break;
  case AKX_LAW_ELASTIC_FD:
    hipLaunchKernelGGL((k_energy_elements_sum<ET, LAW_ELASTIC_FD>), grid, block, 0,
                       m->stream, A, out);
    break;
  case AKX_LAW_NEOHOOKEAN:
    hipLaunchKernelGGL((k_energy_elements_sum<ET, LAW_NEOHOOKEAN>), grid, block, 0,
                       m->stream, A, out);
    break;
  default:
    hipLaunchKernelGGL((k_energy_elements_sum<ET, LAW_PLASTIC>), grid, block, 0, m->stream,
                       A, out);
  }
  HIPCHECK(hipGetLastError());
}

// inputs of Material::getEnergy("potential" / "plastic") of one material
EnergyArgs energy_args(akx_model *m, Material &mat, bool plastic_energy) {
  const bool plastic = mat.law == AKX_LAW_PLASTIC_LIH;
  EnergyArgs A{};
  A.n = mat.n;
  A.first = mat.first;
  A.nn = m->nn;
  A.nq_all = mat.n * m->nqp;
  A.filter = mat.filter.p;
  A.conn = m->conn.p;
  A.X = m->X.p;
  A.lambda = mat.lambda;
  A.mu = mat.mu;
  A.lam_el = mat.per_element ? mat.lam_el.p : nullptr;
  A.mu_el = mat.per_element ? mat.mu_el.p : nullptr;
  if (plastic) {
    A.g = mat.hgrad[mat.cur].p;
    A.s = mat.hsig[mat.cur].p;
    A.eps = mat.heps[mat.cur].p;
    if (plastic_energy)
      A.pe = mat.hpe[mat.cur].p;
  } else {
    A.g = mat.grad.p;
    A.s = mat.stress.p;
  }
  require(A.conn && A.X && (A.pe || (A.g && A.s)), "energy inputs missing");
  return A;
}

// Material::getEnergy gives 0 for ids it does not know: "plastic" of a
// material that is not plastic
bool material_has_energy(const Material &mat, bool plastic_energy) {
  return mat.n > 0 && (!plastic_energy || mat.law == AKX_LAW_PLASTIC_LIH);
}

// Material::getEnergy("potential" / "plastic") of one material
double material_energy(akx_model *m, Material &mat, bool plastic_energy,
                       DevBuf<double> &a, DevBuf<double> &b) {
  if (!material_has_energy(mat, plastic_energy))
    return 0.;
  EnergyArgs A = energy_args(m, mat, plastic_energy);
  a.reserve(mat.n);
  b.reserve((mat.n + 2047) / 2048 + 1);
  A.out = a.p;
  if (m->etype == AKX_TET4)
    launch_energy_elements<ET_TET4>(m, mat.law, A);
  else
    launch_energy_elements<ET_HEX8>(m, mat.law, A);
  return device_sum(m, a, b, mat.n);
}

void refuse_user_potential(akx_model *m, int material_id) {
  for (int k = 0; k < (int)m->mats.size(); ++k)
    if ((material_id == -1 || material_id == k) && m->mats[k]->user())
      throw Error(AKX_ERR_UNSUPPORTED,
                  "the potential energy of a user material is not computed here");
}

// The potential energy reads the stress of the current displacement: one
// element pass that materialises grad u and sigma of the non-plastic
// materials and recomputes the plastic state from the previous one.
// allocate = false: the internals must exist already (no device allocation).
void evaluate_stresses_for_energy(akx_model *m, bool allocate) {
  bool need = false;
  for (auto &mp : m->mats)
    need = need || mp->law != AKX_LAW_PLASTIC_LIH;
  if (!need)
    return;
  for (auto &mp : m->mats) {
    if (mp->user() || mp->law == AKX_LAW_PLASTIC_LIH)
      continue;
    const size_t nq9 = (size_t)(9 * mp->n * m->nqp);
    if (allocate) {
      mp->grad.alloc(nq9);
      mp->stress.alloc(nq9);
    } else if (nq9 > 0) {
      require(mp->grad.p && mp->stress.p && mp->grad.n == nq9 && mp->stress.n == nq9,
              "the stress arrays of the materials do not exist yet: call "
              "akx_model_get_energy(\"potential\") or akx_model_compute_all_stresses once "
              "before akx_model_get_energy_noalloc(\"potential\")");
    }
  }
  user_stress_phase(m);
  for (auto &mp : m->mats)
    if (mp->law == AKX_LAW_PLASTIC_LIH)
      mp->cur = 1 - mp->cur;
  launch_element_pass(m, true);
  flip_plastic_state(m);
}

// ---------------------------------------------------------------------------
// No-allocation energy (akx_model_get_energy_noalloc): the partial sums live
// in one file-scope device array.  Each device holds its own copy of it; the
// host reaches it only through the address hipGetSymbolAddress gives on that
// device (the array's name is a host-side stand-in, not a device address).
// ---------------------------------------------------------------------------
constexpr int64_t NOALLOC_PARTIALS = AKX_NOALLOC_MAX_ITEMS / 2048; // first level
constexpr int64_t NOALLOC_SCRATCH = NOALLOC_PARTIALS + 256;        // + second level

} // namespace

static __device__ __align__(256) double scratch[NOALLOC_SCRATCH];

namespace {

constexpr int MAX_DEVICES = 64;
std::mutex g_scratch_mutex;
double *g_scratch_ptr[MAX_DEVICES] = {};

// Set up once per device, with that device current (akx_model_create).
double *device_scratch(int device) {
  require(device >= 0 && device < MAX_DEVICES, "device index out of range");
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[device]) {
    int cur = -1;
    HIPCHECK(hipGetDevice(&cur));
    require(cur == device, "scratch set-up needs its device current");
    void *p = nullptr;
    HIPCHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    require(p != nullptr, "no device address for the energy scratch array");
    g_scratch_ptr[device] = static_cast<double *>(p);
  }
  return g_scratch_ptr[device];
}

// partials of the first level at sc[0 ..), the second level at
// sc[NOALLOC_PARTIALS ..); returns the final value
double noalloc_reduce(akx_model *m, double *sc, int64_t first_level_sums) {
  return read_back(m, tree_reduce(m, sc, sc + NOALLOC_PARTIALS, first_level_sums));
}

void require_noalloc_size(int64_t n, const char *what) {
  if (n > AKX_NOALLOC_MAX_ITEMS)
    throw Error(AKX_ERR_INVALID,
                std::string("akx_model_get_energy_noalloc: ") + what + " (" +
                    std::to_string(n) + ") exceed the scratch limit of " +
                    std::to_string((long long)AKX_NOALLOC_MAX_ITEMS));
}

} // namespace

extern "C" {

int akx_model_get_energy(akx_model *m, const char *energy_id, int material_id,
                         double *energy) {
  return guard([&] {
    check_ready(m);
    require(energy_id != nullptr && energy != nullptr, "null argument");
    require(material_id >= -1 && material_id < (int)m->mats.size(), "bad material id");
    m->set_device();
    const std::string id(energy_id);
    DevBuf<double> a, b;
    if (id == "kinetic" || id == "external work") {
      require(material_id == -1, "kinetic energy and external work are model energies");
      const int kind = id == "kinetic" ? 0 : 1;
      a.reserve(m->nn);
      b.reserve((m->nn + 2047) / 2048 + 1);
      hipLaunchKernelGGL(k_node_energy, dim3(grid_for(m->nn)), dim3(TPB), 0, m->stream,
                         node_energy_args(m, kind), a.p);
      HIPCHECK(hipGetLastError());
      const double s = device_sum(m, a, b, m->nn);
      *energy = kind == 0 ? s / 2. : s * m->dt;
      return;
    }
    if (id != "potential" && id != "plastic") {
      *energy = 0.; // the reference's Material::getEnergy returns 0 for other ids
      return;
    }
    const bool plastic_energy = id == "plastic";
    if (!plastic_energy) {
      refuse_user_potential(m, material_id);
      evaluate_stresses_for_energy(m, true);
    }
    double e = 0.;
    for (int k = 0; k < (int)m->mats.size(); ++k)
      if (material_id == -1 || material_id == k)
        e += material_energy(m, *m->mats[k], plastic_energy, a, b);
    *energy = e;
  });
}

int akx_model_get_energy_noalloc(akx_model *m, const char *energy_id, int material_id,
                                 double *energy) {
  return guard([&] {
    check_ready(m);
    require(energy_id != nullptr && energy != nullptr, "null argument");
    require(material_id >= -1 && material_id < (int)m->mats.size(), "bad material id");
    m->set_device();
    double *sc = device_scratch(m->device);
    const std::string id(energy_id);
    if (id == "kinetic" || id == "external work") {
      require(material_id == -1, "kinetic energy and external work are model energies");
      require_noalloc_size(m->nn, "nodes");
      const int kind = id == "kinetic" ? 0 : 1;
      double s = 0.;
      if (m->nn > 0) {
        const int64_t nb = (m->nn + 2047) / 2048;
        hipLaunchKernelGGL(k_node_energy_sum, dim3((unsigned)nb), dim3(256), 0, m->stream,
                           node_energy_args(m, kind), sc);
        HIPCHECK(hipGetLastError());
        s = noalloc_reduce(m, sc, nb);
      }
      *energy = kind == 0 ? s / 2. : s * m->dt;
      return;
    }
    if (id != "potential" && id != "plastic") {
      *energy = 0.;
      return;
    }
    const bool plastic_energy = id == "plastic";
    for (int k = 0; k < (int)m->mats.size(); ++k)
      if (material_id == -1 || material_id == k)
        require_noalloc_size(m->mats[k]->n, "elements of a material");
    if (!plastic_energy) {
      refuse_user_potential(m, material_id);
      if (m->has_user())
        throw Error(AKX_ERR_UNSUPPORTED,
                    "akx_model_get_energy_noalloc(\"potential\") runs no computeStress "
                    "plugin: the model has a user material");
      evaluate_stresses_for_energy(m, false);
    }
    double e = 0.;
    for (int k = 0; k < (int)m->mats.size(); ++k) {
      if (material_id != -1 && material_id != k)
        continue;
      Material &mat = *m->mats[k];
      if (!material_has_energy(mat, plastic_energy))
        continue;
      EnergyArgs A = energy_args(m, mat, plastic_energy);
      if (m->etype == AKX_TET4)
        launch_energy_elements_sum<ET_TET4>(m, mat.law, A, sc);
      else
        launch_energy_elements_sum<ET_HEX8>(m, mat.law, A, sc);
      e += noalloc_reduce(m, sc, (mat.n + 2047) / 2048);
    }
    *energy = e;
  });
}

int akx_model_get_internal(akx_model *m, int material_id, int internal,
                           double *host) {
  return guard([&] {
    check_ready(m);
    require(host != nullptr, "null host array");
    require(material_id >= 0 && material_id < (int)m->mats.size(), "bad material id");
    m->set_device();
    Material &mat = *m->mats[material_id];
    int64_t nq = mat.n * m->nqp;
    const double *src = nullptr;
    int comps = 9;
    bool plastic = mat.law == AKX_LAW_PLASTIC_LIH;
    switch (internal) {
    case AKX_INTERNAL_GRAD_U: src = plastic ? mat.hgrad[mat.cur].p : mat.grad.p; break;
    case AKX_INTERNAL_STRESS: src = plastic ? mat.hsig[mat.cur].p : mat.stress.p; break;
    case AKX_INTERNAL_INELASTIC_STRAIN:
      require(plastic, "inelastic_strain exists only for plastic materials");
      src = mat.heps[mat.cur].p;
      break;
    case AKX_INTERNAL_ISO_HARDENING:
      require(plastic, "iso_hardening exists only for plastic materials");
      src = mat.hiso[mat.cur].p;
      comps = 1;
      break;
    default:
      throw Error(AKX_ERR_INVALID, "unknown internal");
    }
    require(src != nullptr, "call computeAllStresses first");
    if (nq == 0)
      return;
    download_soa(m, src, host, nq, comps);
  });
}

} // extern "C"

namespace {

// ---------------------------------------------------------------------------
// FEEngine / DOFManager calls on arbitrary fields, in the operation order of
// the element passes (the reference's):
//   gradientOnIntegrationPoints  g(k, j) = sum_n u(k, n) B(j, n)
//                                (shape_functions_inline_impl.hh:296-310)
//   computeBtD                   BtD(k, n) = sum_j D(k, j) B(j, n)
//                                (shape_lagrange_inline_impl.hh:373-410)
//   integrate                    I(k) = sum_q f(k, q) wJ_q
//                                (integrator_gauss_inline_impl.hh:401-441)
//   assembleElementalArrayLocalArray
//                                out(conn(e, n), k) += s * r_e(k + d n), the
//                                elements in filter order
//                                (dof_manager.cc:65-120)
// Per-point arrays are [point][comps] with the points of element i at rows
// i * nqp ..; matrices per point are column-major (rows k, columns j).
// ---------------------------------------------------------------------------
struct FeArgs {
  int64_t n;             // elements of the call (filter size)
  const int32_t *filter; // null: element i is i
  const int32_t *conn;
  const double *X; // [3][nn]
  int64_t nn;
  const double *in;
  double *out;
  int d; // rows of the per-point matrix (degrees of freedom)
};

template <int ET>
__device__ __forceinline__ void fe_point(const FeArgs &A, int64_t i, int q, int32_t (&nodes)[Elem<ET>::nnpe],
                                         double (&b)[Elem<ET>::nnpe][3], double &wJ) {
  constexpr int NN = Elem<ET>::nnpe;
  const int64_t e = A.filter ? (int64_t)A.filter[i] : i;
  double X[NN][3];
#pragma unroll
  for (int n = 0; n < NN; ++n) {
    nodes[n] = A.conn[e * NN + n];
#pragma unroll
    for (int c = 0; c < 3; ++c)
      X[n][c] = A.X[(int64_t)c * A.nn + nodes[n]];
  }
  double Ji[3][3], detJ;
  wJ = Shape<ET, double>::jacobian_at(X, q, Ji, detJ);
#pragma unroll
  for (int n = 0; n < NN; ++n)
    Shape<ET, double>::bcol(Ji, q, n, b[n]);
}

// one thread per (element, Gauss point); in = field [nn][d]
template <int ET> __global__ void k_fe_gradient(FeArgs A) {
  constexpr int NN = Elem<ET>::nnpe, NQ = Elem<ET>::nqp;
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= A.n * NQ)
    return;
  int32_t nodes[NN];
  double b[NN][3], wJ;
  fe_point<ET>(A, t / NQ, (int)(t % NQ), nodes, b, wJ);
  double *o = A.out + t * 3 * A.d;
  for (int k = 0; k < A.d; ++k)
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      double s = A.in[(int64_t)nodes[0] * A.d + k] * b[0][j];
#pragma unroll
      for (int n = 1; n < NN; ++n)
        s = s + A.in[(int64_t)nodes[n] * A.d + k] * b[n][j];
      o[k + A.d * j] = s;
    }
}

// one thread per (element, Gauss point); in = D [point][d * 3]
template <int ET> __global__ void k_fe_btd(FeArgs A) {
  constexpr int NN = Elem<ET>::nnpe, NQ = Elem<ET>::nqp;
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= A.n * NQ)
    return;
  int32_t nodes[NN];
  double b[NN][3], wJ;
  fe_point<ET>(A, t / NQ, (int)(t % NQ), nodes, b, wJ);
  const double *D = A.in + t * 3 * A.d;
  double *o = A.out + t * NN * A.d;
  for (int k = 0; k < A.d; ++k)
#pragma unroll
    for (int n = 0; n < NN; ++n) {
      double s = D[k] * b[n][0];
      s += D[k + A.d] * b[n][1];
      s += D[k + 2 * A.d] * b[n][2];
      o[k + A.d * n] = s;
    }
}

// one thread per element; in = f [point][d]
template <int ET> __global__ void k_fe_integrate(FeArgs A) {
  constexpr int NN = Elem<ET>::nnpe, NQ = Elem<ET>::nqp;
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= A.n)
    return;
  double wJ[NQ];
  for (int q = 0; q < NQ; ++q) {
    int32_t nodes[NN];
    double b[NN][3];
    fe_point<ET>(A, i, q, nodes, b, wJ[q]);
  }
  for (int k = 0; k < A.d; ++k) {
    double s = A.in[(i * NQ) * A.d + k] * wJ[0];
    for (int q = 1; q < NQ; ++q)
      s = s + A.in[(i * NQ + q) * A.d + k] * wJ[q];
    A.out[i * A.d + k] = s;
  }
}

// one thread per node: its contributions (offsets into the elemental
// array, in filter order) added in that order
__global__ void k_dof_assemble(int64_t nn, const int64_t *rowptr, const int64_t *entry,
                               const double *elem, int d, double scale, double *out) {
  const int64_t node = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (node >= nn)
    return;
  for (int k = 0; k < d; ++k) {
    double acc = out[node * d + k];
    for (int64_t r = rowptr[node]; r < rowptr[node + 1]; ++r)
      acc += scale * elem[entry[r] + k];
    out[node * d + k] = acc;
  }
}

struct FeCall {
  akx_model *m;
  FeArgs A{};
  DevBuf<int32_t> filter;
  DevBuf<double> in, out;
  FeCall(akx_model *mm, const int32_t *filt, int64_t nb_filter, int d) : m(mm) {
    check_ready(m);
    require(d >= 1 && d <= 64, "nb_degree_of_freedom must be in [1, 64]");
    m->set_device();
    A.n = filt ? nb_filter : m->nel;
    require(A.n >= 0, "negative filter size");
    if (filt && nb_filter > 0) {
      for (int64_t i = 0; i < nb_filter; ++i)
        require(filt[i] >= 0 && filt[i] < m->nel, "filter refers to a missing element");
      filter.alloc(nb_filter);
      HIPCHECK(hipMemcpy(filter.p, filt, nb_filter * 4, hipMemcpyHostToDevice));
    }
    A.filter = filter.p;
    A.conn = m->conn.p;
    A.X = m->X.p;
    A.nn = m->nn;
    A.d = d;
  }
  void put(const double *host, int64_t count) {
    in.alloc(count > 0 ? count : 1);
    if (count > 0)
      HIPCHECK(hipMemcpy(in.p, host, count * 8, hipMemcpyHostToDevice));
    A.in = in.p;
  }
  void make_out(int64_t count) {
    out.alloc(count > 0 ? count : 1);
    A.out = out.p;
  }
  void get(double *host, int64_t count) {
    HIPCHECK(hipStreamSynchronize(m->stream));
    if (count > 0)
      HIPCHECK(hipMemcpy(host, out.p, count * 8, hipMemcpyDeviceToHost));
  }
};

template <template <int> class K> void fe_launch(akx_model *m, const FeArgs &A, int64_t threads) {
  if (threads == 0)
    return;
  const dim3 grid(grid_for(threads)), block(TPB);
  if (m->etype == AKX_HEX8)
    hipLaunchKernelGGL(K<ET_HEX8>::fn, grid, block, 0, m->stream, A);
  else
    hipLaunchKernelGGL(K<ET_TET4>::fn, grid, block, 0, m->stream, A);
  HIPCHECK(hipGetLastError());
}

template <int ET> struct KGrad { static constexpr auto fn = k_fe_gradient<ET>; };
template <int ET> struct KBtd { static constexpr auto fn = k_fe_btd<ET>; };
template <int ET> struct KInt { static constexpr auto fn = k_fe_integrate<ET>; };

} // namespace

extern "C" {

int akx_fe_gradient_on_integration_points(akx_model *m, const double *field, int nb_dof,
                                          const int32_t *filter, int64_t nb_filter,
                                          double *out) {
  return guard([&] {
    require(field && out, "null array");
    FeCall c(m, filter, nb_filter, nb_dof);
    const int64_t npt = c.A.n * m->nqp;
    c.put(field, m->nn * nb_dof);
    c.make_out(npt * 3 * nb_dof);
    fe_launch<KGrad>(m, c.A, npt);
    c.get(out, npt * 3 * nb_dof);
  });
}

int akx_fe_compute_btd(akx_model *m, const double *Ds, int nb_comp, const int32_t *filter,
                       int64_t nb_filter, double *BtDs) {
  return guard([&] {
    require(Ds && BtDs, "null array");
    require(nb_comp % 3 == 0, "D must have 3 columns per point (nb_component = 3 d)");
    FeCall c(m, filter, nb_filter, nb_comp / 3);
    const int64_t npt = c.A.n * m->nqp;
    c.put(Ds, npt * nb_comp);
    c.make_out(npt * m->nnpe * c.A.d);
    fe_launch<KBtd>(m, c.A, npt);
    c.get(BtDs, npt * m->nnpe * c.A.d);
  });
}

int akx_fe_integrate(akx_model *m, const double *f, int nb_dof, const int32_t *filter,
                     int64_t nb_filter, double *intf) {
  return guard([&] {
    require(f && intf, "null array");
    FeCall c(m, filter, nb_filter, nb_dof);
    c.put(f, c.A.n * m->nqp * nb_dof);
    c.make_out(c.A.n * nb_dof);
    fe_launch<KInt>(m, c.A, c.A.n);
    c.get(intf, c.A.n * nb_dof);
  });
}

int akx_dof_assemble_elemental_array(akx_model *m, const double *elementary, int nb_dof,
                                     const int32_t *filter, int64_t nb_filter,
                                     double scale, double *assembled) {
  return guard([&] {
    require(elementary && assembled, "null array");
    FeCall c(m, filter, nb_filter, nb_dof);
    const int nnpe = m->nnpe;
    // node -> contributions, in filter order (a counting sort)
    std::vector<int64_t> rowptr(m->nn + 1, 0), entry(c.A.n * nnpe);
    auto elem_of = [&](int64_t i) { return filter ? (int64_t)filter[i] : i; };
    for (int64_t i = 0; i < c.A.n; ++i)
      for (int a = 0; a < nnpe; ++a)
        rowptr[m->conn_host[elem_of(i) * nnpe + a] + 1]++;
    for (int64_t k = 0; k < m->nn; ++k)
      rowptr[k + 1] += rowptr[k];
    std::vector<int64_t> fill(rowptr.begin(), rowptr.end() - 1);
    for (int64_t i = 0; i < c.A.n; ++i)
      for (int a = 0; a < nnpe; ++a)
        entry[fill[m->conn_host[elem_of(i) * nnpe + a]]++] = (i * nnpe + a) * nb_dof;
    DevBuf<int64_t> drow, dent;
    drow.alloc(rowptr.size());
    dent.alloc(entry.empty() ? 1 : entry.size());
    HIPCHECK(hipMemcpy(drow.p, rowptr.data(), rowptr.size() * 8, hipMemcpyHostToDevice));
    if (!entry.empty())
      HIPCHECK(hipMemcpy(dent.p, entry.data(), entry.size() * 8, hipMemcpyHostToDevice));
    c.put(elementary, c.A.n * nnpe * nb_dof);
    c.make_out(m->nn * nb_dof);
    HIPCHECK(hipMemcpy(c.out.p, assembled, m->nn * nb_dof * 8, hipMemcpyHostToDevice));
    hipLaunchKernelGGL(k_dof_assemble, dim3(grid_for(m->nn)), dim3(TPB), 0, m->stream, m->nn,
                       (const int64_t *)drow.p, (const int64_t *)dent.p, (const double *)c.in.p,
                       nb_dof, scale, c.out.p);
    HIPCHECK(hipGetLastError());
    c.get(assembled, m->nn * nb_dof);
  });
}

int akx_calibration_copy(int device, int64_t bytes, int repeats, double *ms) {
  return guard([&] {
    require(bytes >= 32 && repeats > 0 && ms, "bad calibration arguments");
    HIPCHECK(hipSetDevice(device));
    const int64_t n = bytes / 32;
    DevBuf<double4> a, b;
    a.alloc(n);
    b.alloc(n);
    hipStream_t st;
    HIPCHECK(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
    hipEvent_t e0, e1;
    HIPCHECK(hipEventCreate(&e0));
    HIPCHECK(hipEventCreate(&e1));
    require((n + 511) / 512 < (int64_t)UINT32_MAX, "calibration copy too large");
    const unsigned grid = (unsigned)((n + 511) / 512);
    hipLaunchKernelGGL(k_copy_calibration, dim3(grid), dim3(256), 0, st,
                       (const double4 *)a.p, b.p, n); // warm-up
    HIPCHECK(hipEventRecord(e0, st));
    for (int r = 0; r < repeats; ++r)
      hipLaunchKernelGGL(k_copy_calibration, dim3(grid), dim3(256), 0, st,
                         (const double4 *)a.p, b.p, n);
    HIPCHECK(hipEventRecord(e1, st));
    HIPCHECK(hipEventSynchronize(e1));
    float t = 0.f;
    HIPCHECK(hipEventElapsedTime(&t, e0, e1));
    *ms = (double)t / repeats;
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    (void)hipStreamDestroy(st);
  });
}

int akx_model_synchronize(akx_model *m) {
  return guard([&] {
    require(m != nullptr, "null model");
    m->set_device();
    HIPCHECK(hipStreamSynchronize(m->stream));
  });
}

int akx_model_enable_kernel_timing(akx_model *m, int enable) {
  return guard([&] {
    require(m != nullptr, "null model");
    m->drain_timing();
    m->timing = enable != 0;
    for (int k = 0; k < 3; ++k) {
      m->t_ms[k] = 0;
      m->t_n[k] = 0;
    }
  });
}

int akx_model_get_kernel_timing(akx_model *m, int kernel_class, double *total_ms,
                                int64_t *launches) {
  return guard([&] {
    require(m != nullptr, "null model");
    require(kernel_class >= 0 && kernel_class < 3, "bad kernel class");
    m->set_device();
    m->drain_timing();
    if (total_ms)
      *total_ms = m->t_ms[kernel_class];
    if (launches)
      *launches = m->t_n[kernel_class];
  });
}

int akx_model_get_step_workgroups(akx_model *m, int64_t *workgroups) {
  return guard([&] {
    check_ready(m);
    require(workgroups != nullptr, "null output");
    const bool pipelined = m->pipe_parts > 1 && m->pipe_ok;
    *workgroups = small_steps(m) && !pipelined ? m->step.nblocks : 0;
  });
}

int akx_model_get_kernel_bytes(akx_model *m, int kernel_class, double *bytes) {
  return guard([&] {
    check_ready(m);
    require(bytes != nullptr, "null output");
    *bytes = kernel_bytes(m, kernel_class);
  });
}

} // extern "C"
