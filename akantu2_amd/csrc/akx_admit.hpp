// akx_admit.hpp -- the tables and nodal state of an instance that joins a
// batch, made on the device from its uploaded mesh.
//
// A server steps nothing while a request joins.  With host loops over every
// element corner and some 40 fills and copies that took 1.3 ms for an instance
// of some 40,000 elements (12 requests, 15.8 ms); now 0.3 ms (3.6 ms): the mesh
// goes up once and kernels make
//   counts   each block's distinct nodes (block-partial assembly), by a sort in
//            LDS, the entries of every node's row of the force table, and from
//            them the widths of its slices -- the one thing the host waits for,
//            to find the instance's place in the force table
//   blocks   the sort again: the blocks' nodes, the corners' indices among them
//            and their LDS slots
//   rows     every row's entries, in the order they arrive
//   ranks    each entry's place in its row: the number of smaller ones, so the
//            order is that of the blocks or elements whatever the arrival
//   elements, nodes   the arenas' connectivity and nodal state.
// The tables are those of the host loops, entry by entry.
//
// The node and element ranges are taken before anything is uploaded, and what
// the kernels keep between them lies in the instance's own part of the arenas
// (connectivity, mass, force table).  The batch holds a buffer for the rest from
// its creation: ADMIT_NODES nodes' input and the slices' and blocks' counts and
// offsets.  So an admission allocates no device memory; sorting twice costs less
// than reading the first sort's results back (12 requests 3.6 ms either way).
#pragma once
#include "akx_batch.hpp"
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace akx {

constexpr int64_t ADMIT_NODES = 128 * 1024; // uploaded at a time (a multiple of 256)

struct AdmitArgs {
  // uploaded, of the nodes from `first` on: coordinates and velocity [][3]
  // (velocity null: zero), blocked flags [][3] (null: none)
  const double *nodes, *velocity;
  const uint8_t *blocked3;
  int64_t first;
  int64_t nn, nel;
  int32_t nnpe, bs; // elements per block
  int64_t nblk;     // blocks (0: one table entry per element corner)
  // between the kernels.  x: entries of every node's row, y: those that have
  // arrived; in the instance's part of the mass array, which is written last
  int2 *deg;
  int32_t *width; // [slices] longest row
  int32_t *count; // [nblk] distinct nodes
  // the host's answer: row starts of the slices and first entry of the blocks,
  // both relative to the instance's
  const int64_t *off, *boff;
  int32_t *row; // the instance's force-table range, as one item per entry
  BBlk *blk;    // [nblk]
  // the instance's place, and the arenas.  a_conn holds the instance's own node
  // numbers until k_admit_elements
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

// first place of a node's row
__device__ __forceinline__ int64_t admit_row(const AdmitArgs &A, int32_t node) {
  return A.off[node >> 8] + (node & 255);
}

// an item (block or corner) to the next place of its node's row
__device__ __forceinline__ void admit_arrive(const AdmitArgs &A, int32_t node, int32_t item) {
  const int d = atomicAdd(&A.deg[node].y, 1);
  A.row[admit_row(A, node) + (int64_t)d * 256] = item;
}

// the smaller items of a node's row
__device__ __forceinline__ int admit_rank(const AdmitArgs &A, int32_t node, int32_t item) {
  const int64_t row = admit_row(A, node);
  const int deg = A.deg[node].x;
  int rank = 0;
  for (int d = 0; d < deg; ++d)
    rank += A.row[row + (int64_t)d * 256] < item;
  return rank;
}

// One workgroup per block; PAD: its corners, rounded up to a power of two.
// Corners sorted by (node, corner): a corner's position is its LDS slot, the
// number of the distinct nodes before it its node's index.  COUNT: the rows' and
// blocks' numbers of entries only.
template <int PAD, bool COUNT> __global__ void __launch_bounds__(256) k_admit_blocks(AdmitArgs A) {
  __shared__ unsigned long long key[PAD];
  __shared__ int wave_sum[4];
  constexpr int PER = PAD / 256;
  const int64_t b = blockIdx.x, c0 = b * A.bs * A.nnpe, e0 = A.elem0 * A.nnpe + c0;
  const int64_t left = A.nel * A.nnpe - c0;
  const int n = (int)(left < (int64_t)A.bs * A.nnpe ? left : (int64_t)A.bs * A.nnpe);
  for (int i = threadIdx.x; i < PAD; i += 256)
    key[i] = i < n ? (unsigned long long)A.a_conn[e0 + i] << 10 | i : ~0ull;
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
  const int64_t ent = COUNT ? 0 : A.bent0 + A.boff[b];
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int i = i0 + k;
    if (i >= n)
      break;
    const int32_t node = (int32_t)(key[i] >> 10);
    const int c = (int)(key[i] & 1023);
    if (is_new[k]) {
      if constexpr (COUNT) {
        atomicAdd(&A.deg[node].x, 1);
      } else {
        A.a_bnode[ent + idx] = (int32_t)(A.node0 + node);
        if (idx > 0)
          A.a_bsend[ent + idx - 1] = (uint16_t)i; // the node before ends here
        admit_arrive(A, node, (int32_t)b);
      }
      ++idx;
    }
    if constexpr (!COUNT) {
      A.a_ls[e0 + c] = (uint16_t)i;
      A.a_lc[e0 + c] = (uint16_t)(idx - 1);
    }
    if (i == n - 1) {
      if constexpr (COUNT) {
        A.count[b] = idx;
      } else {
        A.a_bsend[ent + idx - 1] = (uint16_t)n;
        A.blk[b] = BBlk{ent, idx, 0};
      }
    }
  }
}

// Without block tables the items are the element corners, each in a row
// of the table; COUNT as above.
template <bool COUNT> __global__ void __launch_bounds__(256) k_admit_corners(AdmitArgs A) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= A.nel * A.nnpe)
    return;
  const int32_t node = A.a_conn[A.elem0 * A.nnpe + i];
  if constexpr (COUNT)
    atomicAdd(&A.deg[node].x, 1);
  else
    admit_arrive(A, node, (int32_t)i);
}

// widest row of every slice; one workgroup per slice
__global__ void __launch_bounds__(256) k_admit_widths(AdmitArgs A) {
  __shared__ int red[4];
  int w = A.deg[(int64_t)blockIdx.x * 256 + threadIdx.x].x;
#pragma unroll
  for (int d = 32; d > 0; d /= 2)
    w = max(w, __shfl_xor(w, d));
  if ((threadIdx.x & 63) == 0)
    red[threadIdx.x >> 6] = w;
  __syncthreads();
  if (threadIdx.x == 0)
    A.width[blockIdx.x] = max(max(red[0], red[1]), max(red[2], red[3]));
}

// grid: blocks, or 256 corners each
__global__ void __launch_bounds__(256) k_admit_ranks(AdmitArgs A) {
  const int64_t b = blockIdx.x;
  if (A.nblk) {
    const int64_t ent = A.bent0 + A.boff[b];
    for (int k = threadIdx.x; k < A.count[b]; k += 256) {
      const int32_t node = (int32_t)(A.a_bnode[ent + k] - A.node0);
      A.a_bpos[ent + k] =
          (int32_t)(A.ell0 + admit_row(A, node) + admit_rank(A, node, (int32_t)b) * 256);
    }
    return;
  }
  const int64_t i = b * 256 + threadIdx.x;
  if (i >= A.nel * A.nnpe)
    return;
  const int64_t at = A.elem0 * A.nnpe + i;
  const int32_t node = A.a_conn[at];
  A.a_pos[at] = (int32_t)(A.ell0 + admit_row(A, node) + admit_rank(A, node, (int32_t)i) * 256);
}

__global__ void __launch_bounds__(256) k_admit_elements(AdmitArgs A) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < A.nel * A.nnpe)
    A.a_conn[A.elem0 * A.nnpe + i] += (int32_t)A.node0;
}

// nodal state of the uploaded nodes' slices: X and v as given, all else zero, the
// padding nodes' too; these are blocked
__global__ void __launch_bounds__(256) k_admit_nodes(AdmitArgs A) {
  const int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x, i = A.first + k; // < nn_pad
  const int64_t n = A.node0 + i;
  const bool real = i < A.nn;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const double x = real ? A.nodes[3 * k + c] : 0.;
    const int64_t o = c * A.ncap + n;
    A.a_xu[6 * n + c] = x;
    A.a_xu[6 * n + 3 + c] = 0.;
    if (A.a_x) {
      A.a_x[o] = x;
      A.a_u[o] = 0.;
    }
    A.a_v[o] = real && A.velocity ? A.velocity[3 * k + c] : 0.;
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
        bits |= A.blocked3[3 * k + c] ? 1 << c : 0;
  }
  A.a_blocked[n] = bits;
  A.a_deg[n] = (uint8_t)A.deg[i].x;
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
