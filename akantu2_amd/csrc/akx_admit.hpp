// akx_admit.hpp -- the tables and nodal state of an instance that joins a
// batch, made on the device from its uploaded mesh.
//
// A server steps nothing while a request joins.  With host loops over every
// element corner and some 40 fills and copies that took 1.3 ms for an instance
// of some 40,000 elements (12 requests, 15.8 ms); now 0.3 ms (3.6 ms): the mesh
// goes up once and kernels make
//   blocks   (block-partial assembly) each block's distinct nodes, its corners'
//            indices among them and their LDS slots, by a sort in LDS
//   counts   the entries of every node's row of the force table, and from them
//            the widths of its slices -- the one thing the host waits for, to
//            find the instance's place in the arenas
//   rows     every row's entries, in the order they arrive
//   ranks    each entry's place in its row: the number of smaller ones, so the
//            order is that of the blocks or elements whatever the arrival
//   elements, nodes   the arenas' connectivity and nodal state.
// The tables are those of the host loops, entry by entry.
#pragma once
#include "akx_batch.hpp"
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace akx {

struct AdmitArgs {
  // uploaded: coordinates and velocity [nn][3] (velocity null: zero), blocked
  // flags [nn][3] (null: none), connectivity [nel][nnpe]
  const double *nodes, *velocity;
  const uint8_t *blocked3;
  const int32_t *conn;
  int64_t nn, nn_pad, nel;
  int32_t nnpe, bs, pad; // elements per block; corners per block, padded
  int64_t nblk;          // blocks (0: one table entry per element corner)
  // scratch.  An item is a (block, distinct node) pair, at block * pad + k, or
  // an element corner
  int32_t *deg;    // [nn_pad] items of every node
  int32_t *width;  // [nn_pad / 256]
  int32_t *count;  // [nblk] distinct nodes
  int32_t *item;   // [nblk * pad] node of an item
  uint8_t *arrive; // place of an item in its row as it arrived
  uint16_t *send, *lc, *ls;
  // the host's answer: row starts of the slices and first entry of the blocks,
  // both relative to the instance's
  const int64_t *off, *boff;
  int32_t *row; // the instance's force-table range, as one item per entry
  BBlk *blk;    // [nblk]
  // the instance's place, and the arenas
  int64_t node0, elem0, ell0, bent0, ncap;
  int32_t *a_conn, *a_pos, *a_bnode, *a_bpos;
  uint16_t *a_lc, *a_ls, *a_bsend;
  int64_t *a_ell_off;
  uint8_t *a_deg, *a_blocked;
  double *a_xu, *a_x, *a_u, *a_v, *a_a, *a_fint; // a_x, a_u null in FP64 batches
  float *a_cu, *a_cv;                            // FP32 batches
  unsigned long long *min_bits;
  long long *first_bad;
};

// One workgroup per block; PAD: its corners, rounded up to a power of two.
// Corners sorted by (node, corner): a corner's position is its LDS slot, the
// number of the distinct nodes before it its node's index.
template <int PAD> __global__ void __launch_bounds__(256) k_admit_blocks(AdmitArgs A) {
  __shared__ unsigned long long key[PAD];
  __shared__ int wave_sum[4];
  constexpr int PER = PAD / 256;
  const int64_t b = blockIdx.x, c0 = b * A.bs * A.nnpe;
  const int64_t left = A.nel * A.nnpe - c0;
  const int n = (int)(left < (int64_t)A.bs * A.nnpe ? left : (int64_t)A.bs * A.nnpe);
  for (int i = threadIdx.x; i < PAD; i += 256)
    key[i] = i < n ? (unsigned long long)A.conn[c0 + i] << 10 | i : ~0ull;
  __syncthreads();
  for (int size = 2; size <= PAD; size *= 2)
    for (int step = size / 2; step > 0; step /= 2) {
      for (int i = threadIdx.x; i < PAD / 2; i += 256) {
        const int lo = 2 * i - (i & (step - 1)), hi = lo + step;
        const unsigned long long x = key[lo], y = key[hi];
        if ((x > y) == ((lo & size) == 0)) {
          key[lo] = y;
          key[hi] = x;
        }
      }
      __syncthreads();
    }
  // distinct nodes before this lane's PER positions
  const int i0 = threadIdx.x * PER;
  bool is_new[PER];
  int mine = 0;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int i = i0 + k;
    is_new[k] = i < n && (i == 0 || key[i] >> 10 != key[i - 1] >> 10);
    mine += is_new[k];
  }
  int upto = mine;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int d = 1; d < 64; d *= 2) {
    const int v = __shfl_up(upto, d);
    upto += lane >= d ? v : 0;
  }
  if (lane == 63)
    wave_sum[wave] = upto;
  __syncthreads();
  int idx = upto - mine;
  for (int w = 0; w < wave; ++w)
    idx += wave_sum[w];
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int i = i0 + k;
    if (i >= n)
      break;
    const int32_t node = (int32_t)(key[i] >> 10);
    const int c = (int)(key[i] & 1023);
    if (is_new[k]) {
      const int64_t at = b * A.pad + idx;
      A.item[at] = node;
      if (idx > 0)
        A.send[at - 1] = (uint16_t)i; // the node before ends here
      A.arrive[at] = (uint8_t)atomicAdd(&A.deg[node], 1); // read up to 255 items only
      ++idx;
    }
    A.ls[c0 + c] = (uint16_t)i;
    A.lc[c0 + c] = (uint16_t)(idx - 1);
    if (i == n - 1) {
      A.send[b * A.pad + idx - 1] = (uint16_t)n;
      A.count[b] = idx;
    }
  }
}

// without block tables: the items are the element corners
__global__ void __launch_bounds__(256) k_admit_corners(AdmitArgs A) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < A.nel * A.nnpe)
    A.arrive[i] = (uint8_t)atomicAdd(&A.deg[A.conn[i]], 1);
}

// widest row of every slice; one workgroup per slice
__global__ void __launch_bounds__(256) k_admit_widths(AdmitArgs A) {
  __shared__ int red[4];
  int w = A.deg[(int64_t)blockIdx.x * 256 + threadIdx.x];
#pragma unroll
  for (int d = 32; d > 0; d /= 2)
    w = max(w, __shfl_xor(w, d));
  if ((threadIdx.x & 63) == 0)
    red[threadIdx.x >> 6] = w;
  __syncthreads();
  if (threadIdx.x == 0)
    A.width[blockIdx.x] = max(max(red[0], red[1]), max(red[2], red[3]));
}

// node of item (b, k) or of corner b * 256 + k; false past the last
__device__ __forceinline__ bool admit_item(const AdmitArgs &A, int64_t b, int k, int64_t &at,
                                           int32_t &node) {
  at = A.nblk ? b * A.pad + k : b * 256 + k;
  if (A.nblk ? k >= A.count[b] : at >= A.nel * A.nnpe)
    return false;
  node = A.nblk ? A.item[at] : A.conn[at];
  return true;
}
__device__ __forceinline__ int64_t admit_row(const AdmitArgs &A, int32_t node) {
  return A.off[node >> 8] + (node & 255);
}

// grid: blocks, or 256 corners each
__global__ void __launch_bounds__(256) k_admit_rows(AdmitArgs A) {
  const int64_t b = blockIdx.x;
  const int most = A.nblk ? A.pad : 256;
  for (int k = threadIdx.x; k < most; k += 256) {
    int64_t at;
    int32_t node;
    if (!admit_item(A, b, k, at, node))
      break;
    A.row[admit_row(A, node) + (int64_t)A.arrive[at] * 256] = (int32_t)(A.nblk ? b : at);
  }
}

__global__ void __launch_bounds__(256) k_admit_ranks(AdmitArgs A) {
  const int64_t b = blockIdx.x;
  const int most = A.nblk ? A.pad : 256;
  for (int k = threadIdx.x; k < most; k += 256) {
    int64_t at;
    int32_t node;
    if (!admit_item(A, b, k, at, node))
      break;
    const int64_t row = admit_row(A, node);
    const int32_t me = (int32_t)(A.nblk ? b : at);
    int rank = 0;
    for (int d = 0; d < A.deg[node]; ++d)
      rank += A.row[row + d * 256] < me;
    const int32_t pos = (int32_t)(A.ell0 + row + rank * 256);
    if (A.nblk) {
      const int64_t o = A.bent0 + A.boff[b] + k;
      A.a_bnode[o] = (int32_t)(A.node0 + node);
      A.a_bpos[o] = pos;
      A.a_bsend[o] = A.send[at];
    } else {
      A.a_pos[A.elem0 * A.nnpe + at] = pos;
    }
  }
  if (A.nblk && threadIdx.x == 0)
    A.blk[b] = BBlk{A.bent0 + A.boff[b], A.count[b], 0};
}

__global__ void __launch_bounds__(256) k_admit_elements(AdmitArgs A) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= A.nel * A.nnpe)
    return;
  const int64_t at = A.elem0 * A.nnpe + i;
  A.a_conn[at] = (int32_t)(A.node0 + A.conn[i]);
  if (A.nblk) {
    A.a_lc[at] = A.lc[i];
    A.a_ls[at] = A.ls[i];
  }
}

// nodal state: X and v as given, all else zero, the padding nodes' too; these
// are blocked
__global__ void __launch_bounds__(256) k_admit_nodes(AdmitArgs A) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; // < nn_pad
  const int64_t n = A.node0 + i;
  const bool real = i < A.nn;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const double x = real ? A.nodes[3 * i + c] : 0.;
    const int64_t o = c * A.ncap + n;
    A.a_xu[6 * n + c] = x;
    A.a_xu[6 * n + 3 + c] = 0.;
    if (A.a_x) {
      A.a_x[o] = x;
      A.a_u[o] = 0.;
    }
    A.a_v[o] = real && A.velocity ? A.velocity[3 * i + c] : 0.;
    A.a_a[o] = 0.;
    A.a_fint[o] = 0.;
    if (A.a_cu) {
      A.a_cu[o] = 0.f;
      A.a_cv[o] = 0.f;
    }
  }
  uint8_t bits = 7;
  if (real) {
    bits = 0;
    if (A.blocked3)
#pragma unroll
      for (int c = 0; c < 3; ++c)
        bits |= A.blocked3[3 * i + c] ? 1 << c : 0;
  }
  A.a_blocked[n] = bits;
  A.a_deg[n] = (uint8_t)A.deg[i];
  if (threadIdx.x == 0)
    A.a_ell_off[n >> 8] = A.ell0 + A.off[i >> 8];
  if (i == 0) {
    *A.first_bad = INT64_MAX;
    *A.min_bits = 0x7FEFFFFFFFFFFFFFull; // the largest double
  }
}

// zero Gauss points q0 .. q0 + n - 1 of every component of the plastic history:
// blockIdx.y counts the components of the 8 arrays
struct AdmitHist {
  void *p[8];
  int32_t comps[8];
  int64_t stride, q0, n;
  int32_t bytes; // of a value
};
__global__ void __launch_bounds__(256) k_admit_history(AdmitHist H) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= H.n)
    return;
  int k = 0, c = blockIdx.y;
  while (c >= H.comps[k])
    c -= H.comps[k++];
  const int64_t o = c * H.stride + H.q0 + i;
  if (H.bytes == 4)
    static_cast<float *>(H.p[k])[o] = 0.f;
  else
    static_cast<double *>(H.p[k])[o] = 0.;
}

} // namespace akx
