// The FP32 operator of the PCG engine and the AMG levels: one 3x3 block per
// adjacency slot, held as three arrays over the slots
//   A [nadj][4] = entries 0..3,  B [nadj][4] = entries 4..7,  C [nadj] = entry 8
// of the block's [c][d] (entry 3c + d couples row component c to column
// component d), one after the other in 9 nadj floats.  Neighbouring lanes read
// neighbouring 16-byte pieces; as one 36-byte record a block, every load
// straddles and the texture-address unit is what the product waits for (83 %
// busy).  59.5 M blocks (tet10, 2.1 M nodes), one product:
//   36-byte records, 8 lanes a row 576 us (4.1 TB/s), 16 lanes 530;
//   three arrays, 8 lanes 570, 16 lanes 495 (4.8 TB/s), 32 lanes 546.
// (Four-block chunks with the column index inside, rows padded to four: 473 us
// for 16 % more memory; more loads in flight, blocks walking several row
// groups, non-temporal loads: slower.)
#pragma once

#include "common.h"

namespace llfem {
namespace {

typedef float f4v __attribute__((ext_vector_type(4)));

constexpr int kRowLanes = 16;              // lanes per block row
// Threads of a row kernel's block.  AMG solve of 2.1 M nodes with 128, 256, 512,
// 1024: 367, 344, 354, 366 ms; each XCD taking a contiguous run of blocks: 357.
constexpr int kRowThreads = 256;
constexpr int kRowNodes = kRowThreads / kRowLanes;

inline int64_t row_groups(int64_t N) { return N < kRowNodes ? 1 : (N + kRowNodes - 1) / kRowNodes; }

// index of entry e of block g in the 9 nadj floats
__host__ __device__ __forceinline__ int64_t block32_at(int64_t nadj, int64_t g, int e) {
  return e < 8 ? (int64_t)(e >> 2) * 4 * nadj + 4 * g + (e & 3) : 8 * nadj + g;
}

// Row of the operator times x by the row's kRowLanes lanes (l: the lane), blocks
// p0 .. p0 + R - 1: the three components in every lane, by a fixed butterfly.
template <typename VT, typename Adj, typename Val, typename X>
__device__ __forceinline__ void row_product(int64_t nadj, Adj adj, Val val, X x, int64_t p0, int R, int l, VT& a0,
                                            VT& a1, VT& a2) {
  typedef __attribute__((address_space(1))) const f4v* V4;
  const V4 A = (V4)val, B = (V4)(val + 4 * nadj);
  const auto C = val + 8 * nadj;
  a0 = a1 = a2 = 0;
  for (int t = l; t < R; t += kRowLanes) {
    const int64_t p = p0 + t, i = adj[p];
    const f4v a = A[p], b = B[p];
    const float c = C[p];
    const VT x0 = x[3 * i], x1 = x[3 * i + 1], x2 = x[3 * i + 2];
    a0 += (VT)a.x * x0 + (VT)a.y * x1 + (VT)a.z * x2;
    a1 += (VT)a.w * x0 + (VT)b.x * x1 + (VT)b.y * x2;
    a2 += (VT)b.z * x0 + (VT)b.w * x1 + (VT)c * x2;
  }
#pragma unroll
  for (int o = kRowLanes / 2; o > 0; o >>= 1) {
    a0 += __shfl_xor(a0, o, kRowLanes);
    a1 += __shfl_xor(a1, o, kRowLanes);
    a2 += __shfl_xor(a2, o, kRowLanes);
  }
}

// Where the row of this thread's lanes lies: blocks p0 .. p0 + R - 1.
struct RowSpan {
  int64_t p0;
  int R;
};

// Loaded without a branch, so that the load of the system's state can be under
// way with it (0.6 us each on an idle chip).
template <typename AdjPtr>
__device__ __forceinline__ RowSpan row_span(int64_t N, AdjPtr adj_ptr, int64_t lb) {
  const int64_t j = lb * kRowNodes + threadIdx.x / kRowLanes, i = j < N ? j : N - 1;
  const int64_t p0 = adj_ptr[i], p1 = adj_ptr[i + 1];
  return {p0, j < N ? (int)(p1 - p0) : 0};
}

// A wave-uniform value that has to be in its registers here: the fields of a
// table entry are fetched together at the kernel's start instead of one by one
// where they are first used, each a wait of 0.1 us.
template <typename T>
__device__ __forceinline__ T pinned(T v) {
  asm volatile("" : "+s"(v));
  return v;
}

// The rows of one block's kRowNodes nodes: y[3 n + c] = sum_t block(t) x, into
// LDS (48 values).  Ends with a barrier: thread i < 48 may then read sh[i], row
// component 48 lb + i.
template <typename VT, typename Adj, typename Val, typename X>
__device__ __forceinline__ void block_rows(int64_t nadj, RowSpan r, Adj adj, Val val, X x, VT* sh) {
  const int l = threadIdx.x % kRowLanes;
  VT a0, a1, a2;
  row_product<VT>(nadj, adj, val, x, r.p0, r.R, l, a0, a1, a2);
  if (l < 3) sh[3 * (threadIdx.x / kRowLanes) + l] = l == 0 ? a0 : l == 1 ? a1 : a2;
  __syncthreads();
}

// Sum over one wavefront in a fixed order.
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

}  // namespace
}  // namespace llfem
