// Aggregation AMG preconditioner for the elasticity systems of the PCG engine.
//
// Reference: solveDisplacement(K, f; support, iterative=true,
// preconditioner=...) passes its `preconditioner` to cg as Pl
// (src/linear.jl:3711-3743, the call at :3736); the reference's default is
// Identity().  This file provides a multigrid Pl that stays on the device
// across requests on the same mesh and support.
//
// Method (plain aggregation AMG with rigid-body near-null space):
//   * Aggregates: greedy root + strong neighbours (block Frobenius norm
//     >= 0.25 x the row's largest off-diagonal block), then leftovers join
//     the neighbouring aggregate they couple to most.  Coarser levels
//     aggregate the aggregate graph itself.
//   * Tentative prolongator: per aggregate, the six rigid-body modes of its
//     nodes (constrained DoFs zeroed), orthonormalised by modified
//     Gram-Schmidt in FP64; the triangular factor is the next level's
//     near-null space.  Columns that vanish (e.g. aggregates of clamped
//     nodes) are dropped and their coarse DoFs masked.
//   * Coarse operators A_{l+1} = Q^T A_l Q (Galerkin), per request on the
//     device: each coarse 6x6 block sums its fine blocks in a fixed order.
//   * Smoother: Chebyshev (degree 2) on D^-1 A over [0.1, 1.1] x lambda,
//     lambda from 15 power steps; coarse correction scaled by 1.5; dense
//     inverse on the coarsest level (at most 24 aggregates).
//
// Everything a level needs lives in 3-DoF "pseudo-node" block form: a
// coarse aggregate's six DoFs are two pseudo-nodes, so every level uses the
// same block-sparse layout as the fine operator ([slot][c][d] FP32 blocks,
// node-major adjacency, block32.h).  The V-cycle kernels run table-driven over all
// systems of a batch, one launch per kernel and level.
#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cmath>
#include <cstring>
#include <future>
#include <numeric>
#include <thread>
#include <vector>

#include "block32.h"
#include "common.h"

namespace llfem {

namespace {

constexpr int kMB = 256;                 // threads per block
constexpr int kMG = 16;                  // lanes per aggregate in the restriction
constexpr int kMSpN = kMB / kMG;         // aggregates per restriction block
// The row kernels (products, block32.h) take one block per kRowNodes rows; the
// vector and restriction kernels cap their blocks and stride.
constexpr int64_t kMaxVB = 1024, kMaxAB = 1024;
constexpr int kCheb = 2;                 // Chebyshev degree (pre and post)
constexpr double kChebLo = 0.1, kChebHi = 1.1;
constexpr float kOverCorrect = 1.5f;
constexpr double kStrength = 0.25;
constexpr int kPowerSteps = 15;
constexpr int64_t kCoarseAggs = 24;      // coarsest level: at most this many aggregates
constexpr int kMaxLevels = 12;
constexpr int64_t kMaxDense = 1536;      // DoFs of the dense coarsest solve
constexpr int kTB = 1024;                // threads of the tail kernel
constexpr int64_t kTailN = 320;          // pseudo-nodes of a tail's levels together (the coarsest alone: kMaxDense / 3)
constexpr int64_t kTailMax = kTailN > kMaxDense / 3 ? kTailN : kMaxDense / 3;

inline unsigned nblk(int64_t n, int bs = kMB) { return (unsigned)std::max<int64_t>(1, (n + bs - 1) / bs); }
inline int64_t cap(int64_t n, int64_t per, int64_t mx) { return std::max<int64_t>(1, std::min<int64_t>((n + per - 1) / per, mx)); }

__device__ __forceinline__ double msum(double v, double* sh) {
  const int t = threadIdx.x;
  sh[t] = v;
  __syncthreads();
  for (int o = blockDim.x / 2; o > 0; o >>= 1) {
    if (t < o) sh[t] += sh[t + o];
    __syncthreads();
  }
  const double r = sh[0];
  __syncthreads();
  return r;
}

}  // namespace

// One (system, level) entry of a V-cycle launch.
struct MgEnt {
  int64_t N;                 // pseudo-nodes of the level (3 DoFs each)
  const int64_t* adj_ptr;
  const int32_t* adj;
  int64_t nadj;
  const float* val;          // block32.h
  const uint8_t* mask;       // [3N] 1 = no DoF (constrained / dropped)
  const float* dinv;         // [3N] inverse diagonal, 0 on masked DoFs
  float* b;                  // right-hand side of the level
  float* x;                  // iterate of the level; the smoothing steps alternate
  float* y;                  // between x and y, and end in x
  float* d;                  // Chebyshev direction
  const int32_t* agg;        // [N] aggregate of each pseudo-node (-1: none)
  const float* Q;            // [N][3][6] tentative prolongator rows
  const int32_t* mem_ptr;    // [nagg+1] members of each aggregate
  const int32_t* mem;
  int64_t nagg;
  float* bc;                 // next level's b
  const float* xc;           // next level's x
  float *yc, *dc;            // next level's y, d and inverse diagonal (NULL: that level is in the tail)
  const float* dinvc;
  const float* chebc;        // its cheb
  const float* Ainv;         // coarsest: dense inverse [nc][nc]
  int32_t nc;
  const float* cheb;         // 1 / theta, 1 / delta of the smoother's interval
  const double* state;       // system state word: run only while it reads 0 (NULL: always)
  double* rzpart;            // level 0: partial r.z per row block
  int32_t sblk0, nsblk, vblk0, nvblk, ablk0, nablk;
};

// A system's last levels in the tail kernel: entries first .. first + count - 1.
struct MgTail {
  int32_t first, count;
};

namespace {

struct ChebCoef {
  float ca, cbt, cbd;
};
struct ChebSet {
  ChebCoef pre[kCheb - 1], post[kCheb];
};

__device__ __forceinline__ bool mg_skip(const MgEnt& E) { return E.state && *E.state != 0.0; }

// entry of a block; the map is a dependent load that one entry needs none of
__device__ __forceinline__ const MgEnt& mg_ent(const MgEnt* ents, const int32_t* map, int nent) {
  return ents[nent == 1 ? 0 : map[blockIdx.x]];
}


// First Chebyshev step from x = 0: y = d = D^-1 b / theta.  Only where level 0
// starts outside the engine's iteration: there the update kernel does it, and
// k_mg_restrict for the other levels.
__global__ __launch_bounds__(kMB) void k_mg_cheb0(const MgEnt* __restrict__ ents, const int32_t* __restrict__ map,
                                                  int nent) {
  const MgEnt& E = mg_ent(ents, map, nent);
  if (mg_skip(E)) return;
  const int lb = blockIdx.x - E.vblk0;
  const float* __restrict__ dinv = (const float*)gp(E.dinv);
  const float* __restrict__ b = (const float*)gp(E.b);
  float* __restrict__ y = (float*)gp(E.y);
  float* __restrict__ d = (float*)gp(E.d);
  const float it = gp(E.cheb)[0];
  for (int64_t i = (int64_t)lb * kMB + threadIdx.x; i < 3 * E.N; i += (int64_t)E.nvblk * kMB) {
    const float v = it * dinv[i] * b[i];
    y[i] = v;
    d[i] = v;
  }
}

// Chebyshev step: d = ca d + (cbt / theta + cbd / delta) D^-1 (b - A u),
// w = u + d, with u, w = y, x (from_y) or x, y.  D^-1 is 0 on masked DoFs.
// The product's block applies the step to its own rows, so neither A u nor a
// second launch for the vectors is needed: 3 launches a level and a pass over
// the vectors less.  With block32.h's layout, a solve of 2.1 M nodes (92
// iterations) 413 -> 376 ms, eight systems on a server 55.8 -> 51.6 ms.  w is
// another array than u because other blocks still read u.  rz (level 0, last
// step): partial b.w per block.
__global__ __launch_bounds__(kRowThreads) void k_mg_smooth(const MgEnt* __restrict__ ents,
                                                           const int32_t* __restrict__ map, int nent, float ca,
                                                           float cbt, float cbd, int from_y, int rz) {
  __shared__ float sh[3 * kRowNodes];
  const MgEnt& E = mg_ent(ents, map, nent);
  const int lb = blockIdx.x - pinned(E.sblk0);
  const int64_t N = pinned(E.N), nadj = pinned(E.nadj);
  const auto ap = gp(pinned(E.adj_ptr));
  const auto adj = gp(pinned(E.adj));
  const auto val = gp(pinned(E.val));
  const double* const state = pinned(E.state);
  float *const ex = pinned(E.x), *const ey = pinned(E.y), *const ed = pinned(E.d);
  const float *const eb = pinned(E.b), *const edinv = pinned(E.dinv), *const echeb = pinned(E.cheb);
  double* const erz = pinned(E.rzpart);
  const double st = state ? *gp(state) : 0.0;
  const RowSpan rs = row_span(N, ap, lb);
  if (st != 0.0) return;
  const auto* __restrict__ u = gp((const float*)(from_y ? ey : ex));
  const int64_t i = (int64_t)lb * 3 * kRowNodes + threadIdx.x;
  const bool own = threadIdx.x < 3 * kRowNodes && i < 3 * N;
  const float c0 = gp(echeb)[0], c1 = gp(echeb)[1];
  float bi = 0.f, di = 0.f, vi = 0.f, ui = 0.f;
  if (own) {   // loaded now, beside the product's
    bi = gp(eb)[i];
    di = gp(ed)[i];
    vi = gp(edinv)[i];
    ui = u[i];
  }
  block_rows<float>(nadj, rs, adj, val, u, sh);
  if (threadIdx.x >= 64) return;
  double acc = 0.0;
  if (own) {
    const float cb = cbt * c0 + cbd * c1;
    const float dv = ca * di + cb * vi * (bi - sh[threadIdx.x]);
    const float wv = ui + dv;
    gp(ed)[i] = dv;
    gp(from_y ? ex : ey)[i] = wv;
    acc = (double)bi * (double)wv;
  }
  if (rz) {
    acc = wave_sum(acc);
    if (threadIdx.x == 0) gp(erz)[lb] = acc;
  }
}

// residual of the level, w = mask(b - A u): u, w = y, x (from_y) or x, y
__global__ __launch_bounds__(kRowThreads) void k_mg_resid(const MgEnt* __restrict__ ents,
                                                          const int32_t* __restrict__ map, int nent, int from_y) {
  __shared__ float sh[3 * kRowNodes];
  const MgEnt& E = mg_ent(ents, map, nent);
  const int lb = blockIdx.x - pinned(E.sblk0);
  const int64_t N = pinned(E.N), nadj = pinned(E.nadj);
  const auto ap = gp(pinned(E.adj_ptr));
  const auto adj = gp(pinned(E.adj));
  const auto val = gp(pinned(E.val));
  const double* const state = pinned(E.state);
  float *const ex = pinned(E.x), *const ey = pinned(E.y);
  const float* const eb = pinned(E.b);
  const uint8_t* const emask = pinned(E.mask);
  const double st = state ? *gp(state) : 0.0;
  const RowSpan rs = row_span(N, ap, lb);
  if (st != 0.0) return;
  const auto* __restrict__ u = gp((const float*)(from_y ? ey : ex));
  const int64_t i = (int64_t)lb * 3 * kRowNodes + threadIdx.x;
  const bool own = threadIdx.x < 3 * kRowNodes && i < 3 * N;
  float bi = 0.f;
  uint8_t mi = 1;
  if (own) {
    bi = gp(eb)[i];
    mi = gp(emask)[i];
  }
  block_rows<float>(nadj, rs, adj, val, u, sh);
  if (own) gp(from_y ? ex : ey)[i] = mi ? 0.f : bi - sh[threadIdx.x];
}

// bc = Q^T r, r in y (in_y) or x: kMG lanes per aggregate stride over its
// members, then a fixed shuffle tree sums the lanes.
__global__ __launch_bounds__(kMB) void k_mg_restrict(const MgEnt* __restrict__ ents, const int32_t* __restrict__ map,
                                                     int nent, int in_y) {
  const MgEnt& E = mg_ent(ents, map, nent);
  if (mg_skip(E)) return;
  const int lb = blockIdx.x - E.ablk0;
  const int l = threadIdx.x % kMG;
  const int32_t* __restrict__ mem_ptr = (const int32_t*)gp(E.mem_ptr);
  const int32_t* __restrict__ mem = (const int32_t*)gp(E.mem);
  const float* __restrict__ Q = (const float*)gp(E.Q);
  const float* __restrict__ rv = (const float*)gp(in_y ? E.y : E.x);
  float* __restrict__ bc = (float*)gp(E.bc);
  for (int64_t a = (int64_t)lb * kMSpN + threadIdx.x / kMG; a - threadIdx.x / kMG < E.nagg;
       a += (int64_t)E.nablk * kMSpN) {
    float acc[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (a < E.nagg) {
      for (int32_t m = mem_ptr[a] + l; m < mem_ptr[a + 1]; m += kMG) {
        const int64_t j = mem[m];
        const float* Qj = Q + 18 * j;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          const float r = rv[3 * j + c];
#pragma unroll
          for (int u = 0; u < 6; ++u) acc[u] += Qj[6 * c + u] * r;
        }
      }
    }
#pragma unroll
    for (int o = kMG / 2; o > 0; o >>= 1)
#pragma unroll
      for (int u = 0; u < 6; ++u) acc[u] += __shfl_xor(acc[u], o, kMG);
    if (a < E.nagg && l < 6) {
      float v = acc[0];
#pragma unroll
      for (int u = 1; u < 6; ++u) v = l == u ? acc[u] : v;
      const int64_t i = 6 * a + l;
      bc[i] = v;
      if (E.yc) {   // the next level's first Chebyshev step
        const float w = gp(E.chebc)[0] * gp(E.dinvc)[i] * v;
        gp(E.yc)[i] = w;
        gp(E.dc)[i] = w;
      }
    }
  }
}

// u += alpha Q xc, u = y (in_y) or x
__global__ __launch_bounds__(kMB) void k_mg_prolong(const MgEnt* __restrict__ ents, const int32_t* __restrict__ map,
                                                    int nent, float alpha, int in_y) {
  const MgEnt& E = mg_ent(ents, map, nent);
  if (mg_skip(E)) return;
  const int lb = blockIdx.x - E.vblk0;
  const int32_t* __restrict__ agg = (const int32_t*)gp(E.agg);
  const float* __restrict__ Q = (const float*)gp(E.Q);
  const float* __restrict__ xcv = (const float*)gp(E.xc);
  float* __restrict__ x = (float*)gp(in_y ? E.y : E.x);
  for (int64_t j = (int64_t)lb * kMB + threadIdx.x; j < E.N; j += (int64_t)E.nvblk * kMB) {
    const int32_t a = agg[j];
    if (a < 0) continue;
    const float* Qj = Q + 18 * j;
    const float* xc = xcv + 6 * (int64_t)a;
    float v[6];
#pragma unroll
    for (int u = 0; u < 6; ++u) v[u] = xc[u];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      float s = 0.f;
#pragma unroll
      for (int u = 0; u < 6; ++u) s += Qj[6 * c + u] * v[u];
      x[3 * j + c] += alpha * s;
    }
  }
}

// The levels from a system's tail to its coarsest (x = Ainv b there), one block
// per system: their vectors lie in LDS and a barrier stands for the end of a
// launch.  As launches of their own these levels take 4.5 us a kernel, seven a
// level and 8 us for the coarsest, whatever their size; here one CU fetches the
// operator (28 KB a pass of 64 rows) four times over, so a level pays while it
// has few rows: up to 320 23 us instead of 40, up to 1,000 45 us (eight systems
// on a server 44.5 and 47.0 ms under the same load).  Rows kept in registers
// spilled and lost.
__global__ __launch_bounds__(kTB) void k_mg_tail(const MgTail* __restrict__ tails, const MgEnt* __restrict__ ents,
                                                 ChebSet cs, float alpha) {
  __shared__ float sb[3 * kTailMax], sx[3 * kTailMax], sy[3 * kTailMax], sd[3 * kTailMax];
  const MgTail T = tails[blockIdx.x];
  const MgEnt* L = ents + T.first;
  if (mg_skip(L[0])) return;
  const int t = threadIdx.x, l = t % kRowLanes;
  // one Chebyshev step of level E at offset o: u -> w (k_mg_smooth)
  auto smooth = [&](const MgEnt& E, int o, const ChebCoef& c, const float* u, float* w) {
    const float cb = c.cbt * gp(E.cheb)[0] + c.cbd * gp(E.cheb)[1];
    const auto ap = gp(E.adj_ptr);
    const auto dinv = gp(E.dinv);
    for (int j = t / kRowLanes; j < (int)E.N; j += kTB / kRowLanes) {
      const int64_t p0 = ap[j];
      float a0, a1, a2;
      row_product<float>(E.nadj, gp(E.adj), gp(E.val), u + o, p0, (int)(ap[j + 1] - p0), l, a0, a1, a2);
      if (l < 3) {
        const int i = 3 * j + l;
        const float dv = c.ca * sd[o + i] + cb * dinv[i] * (sb[o + i] - (l == 0 ? a0 : l == 1 ? a1 : a2));
        sd[o + i] = dv;
        w[o + i] = u[o + i] + dv;
      }
    }
    __syncthreads();
  };
  int o = 0;
  for (int i = t; i < 3 * (int)L[0].N; i += kTB) sb[i] = gp((const float*)L[0].b)[i];
  __syncthreads();
  for (int k = 0; k + 1 < T.count; ++k) {
    const MgEnt& E = L[k];
    const int n = 3 * (int)E.N;
    for (int i = t; i < n; i += kTB) {
      const float v = gp(E.cheb)[0] * gp(E.dinv)[i] * sb[o + i];
      sy[o + i] = v;
      sd[o + i] = v;
    }
    __syncthreads();
    float *u = sy, *w = sx;
#pragma unroll
    for (int s = 0; s < kCheb - 1; ++s) {
      smooth(E, o, cs.pre[s], u, w);
      float* h = u;
      u = w;
      w = h;
    }
    const auto ap = gp(E.adj_ptr);
    for (int j = t / kRowLanes; j < (int)E.N; j += kTB / kRowLanes) {   // w = mask(b - A u)
      const int64_t p0 = ap[j];
      float a0, a1, a2;
      row_product<float>(E.nadj, gp(E.adj), gp(E.val), u + o, p0, (int)(ap[j + 1] - p0), l, a0, a1, a2);
      if (l < 3) {
        const int i = 3 * j + l;
        w[o + i] = gp(E.mask)[i] ? 0.f : sb[o + i] - (l == 0 ? a0 : l == 1 ? a1 : a2);
      }
    }
    __syncthreads();
    const auto mp = gp(E.mem_ptr);
    const auto mem = gp(E.mem);
    const auto Q = gp(E.Q);
    const int lm = t % kMG;
    for (int a = t / kMG; a < (int)E.nagg; a += kTB / kMG) {   // next b = Q^T w
      float acc[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      for (int32_t m = mp[a] + lm; m < mp[a + 1]; m += kMG) {
        const int j = mem[m];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          const float r = w[o + 3 * j + c];
#pragma unroll
          for (int v = 0; v < 6; ++v) acc[v] += Q[18 * j + 6 * c + v] * r;
        }
      }
#pragma unroll
      for (int q = kMG / 2; q > 0; q >>= 1)
#pragma unroll
        for (int v = 0; v < 6; ++v) acc[v] += __shfl_xor(acc[v], q, kMG);
      if (lm < 6) {
        float r = acc[0];
#pragma unroll
        for (int v = 1; v < 6; ++v) r = lm == v ? acc[v] : r;
        sb[o + n + 6 * a + lm] = r;
      }
    }
    __syncthreads();
    o += n;
  }
  {
    const MgEnt& E = L[T.count - 1];
    const auto Ai = gp(E.Ainv);
    for (int i = t / kRowLanes; i < E.nc; i += kTB / kRowLanes) {
      float s = 0.f;
      for (int k = l; k < E.nc; k += kRowLanes) s += Ai[(int64_t)i * E.nc + k] * sb[o + k];
#pragma unroll
      for (int q = kRowLanes / 2; q > 0; q >>= 1) s += __shfl_xor(s, q, kRowLanes);
      if (l == 0) sx[o + i] = s;
    }
    __syncthreads();
  }
  for (int k = T.count - 2; k >= 0; --k) {
    const MgEnt& E = L[k];
    const int n = 3 * (int)E.N;
    o -= n;
    float* u = kCheb % 2 ? sy : sx;
    float* w = kCheb % 2 ? sx : sy;
    for (int i = t; i < n; i += kTB) {   // u += alpha Q x of the next level
      const int a = gp(E.agg)[i / 3];
      if (a < 0) continue;
      float s = 0.f;
#pragma unroll
      for (int v = 0; v < 6; ++v) s += gp(E.Q)[6 * i + v] * sx[o + n + 6 * a + v];
      u[o + i] += alpha * s;
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < kCheb; ++s) {
      smooth(E, o, cs.post[s], u, w);
      float* h = u;
      u = w;
      w = h;
    }
  }
  for (int i = t; i < 3 * (int)L[0].N; i += kTB) gp(L[0].x)[i] = sx[i];
  if (L[0].rzpart && t < (int)L[0].nsblk) {   // a whole system in the tail
    const int i0 = 3 * kRowNodes * t, i1 = min(3 * (int)L[0].N, i0 + 3 * kRowNodes);
    double acc = 0.0;
    for (int i = i0; i < i1; ++i) acc += (double)sb[i] * (double)sx[i];
    gp(L[0].rzpart)[t] = acc;
  }
}

// ---- per-request numeric set-up -------------------------------------------------

// Fewer aggregate pairs than this: a wave each, else 16 lanes.  A pair has 30
// to 90 blocks on average but an aggregate's pair with itself thousands, and
// where the pairs do not fill the chip that one is the launch: 59,000 pairs
// 2,900 us with a lane per coarse row, 317 us with a wave; 1.85 M pairs with
// 8, 16, 32 lanes: 4.2, 3.6, 3.5 ms.
constexpr int64_t kGalPairs = 131072;

// Galerkin product of aggregate pair p, 6x6: sum over its fine blocks g = (j, i)
// of Qj^T B Qi, FP64.  G lanes take the blocks in turn, each with all 36 sums
// (a lane per coarse row reads B and Qi six times over: 8.8 instead of 3.6 ms
// for 59.5 M blocks), and a fixed reduce-scatter leaves each lane its share of
// the 36.  What bounds it: the gathers of B and Q, 16 G blocks/s.
template <int G>
__global__ __launch_bounds__(kMB) void k_galerkin(int64_t npairs, int64_t nadjf, int64_t nadjc,
                                                  const int64_t* __restrict__ gptr,
                                                  const int32_t* __restrict__ gblk, const int32_t* __restrict__ gcol,
                                                  const int32_t* __restrict__ adjf, const float* __restrict__ Qf,
                                                  const float* __restrict__ valf, const int32_t* __restrict__ pair_o,
                                                  float* __restrict__ valc) {
  const int64_t p = (int64_t)blockIdx.x * (kMB / G) + threadIdx.x / G;
  const int l = threadIdx.x % G;
  if (p >= npairs) return;   // the same for the G lanes of a pair
  double acc[36];
#pragma unroll
  for (int k = 0; k < 36; ++k) acc[k] = 0.0;
  const int64_t c1 = gptr[p + 1];
  for (int64_t c = gptr[p] + l; c < c1; c += G) {
    const int64_t g = gblk[c];
    const int64_t j = gcol[c];
    const int64_t i = adjf[g];
    const f4v ba = reinterpret_cast<const f4v*>(valf)[g], bb = reinterpret_cast<const f4v*>(valf + 4 * nadjf)[g];
    const float b8 = valf[8 * nadjf + g];
    float qj[18];
    double qi[18];
    const float2* Qj = reinterpret_cast<const float2*>(Qf + 18 * j);
    const float2* Qi = reinterpret_cast<const float2*>(Qf + 18 * i);
#pragma unroll
    for (int k = 0; k < 9; ++k) {
      const float2 a = Qj[k], b = Qi[k];
      qj[2 * k] = a.x;
      qj[2 * k + 1] = a.y;
      qi[2 * k] = b.x;
      qi[2 * k + 1] = b.y;
    }
#pragma unroll
    for (int u = 0; u < 6; ++u) {
      const double q0 = qj[u], q1 = qj[6 + u], q2 = qj[12 + u];
      const double t0 = q0 * ba.x + q1 * ba.w + q2 * bb.z;
      const double t1 = q0 * ba.y + q1 * bb.x + q2 * bb.w;
      const double t2 = q0 * ba.z + q1 * bb.y + q2 * b8;
#pragma unroll
      for (int v = 0; v < 6; ++v) acc[6 * u + v] += t0 * qi[v] + t1 * qi[6 + v] + t2 * qi[12 + v];
    }
  }
  int base = 0, cnt = 36;   // this lane's entries: base .. base + cnt - 1
  int n = 36;
#pragma unroll
  for (int o = G / 2; o > 0; o >>= 1) {
    const int h = (n + 1) / 2;
    const bool up = l & o;
#pragma unroll
    for (int k = 0; k < 18; ++k) {
      if (k >= h) break;
      const double lo = acc[k], hi = k + h < n ? acc[k + h] : 0.0;
      acc[k] = (up ? hi : lo) + __shfl_xor(up ? lo : hi, o, G);
    }
    base += up ? h : 0;
    cnt = up ? cnt - h : min(cnt, h);
    n = h;
  }
#pragma unroll
  for (int k = 0; k < 36; ++k) {
    if (k >= n) break;
    if (k >= cnt) break;
    const int u = (base + k) / 6, v = (base + k) % 6;
    valc[block32_at(nadjc, pair_o[2 * p + u / 3] + v / 3, 3 * (u % 3) + v % 3)] = (float)acc[k];
  }
}

// The smoothed levels of a system for the kernels below, one block per 16 rows
// of any level: levels in one launch, since most of them are small and a
// launch costs 3 us whatever it does.
struct SetLev {
  int64_t N, nadj;
  const int64_t* adj_ptr;
  const int32_t *adj, *dslot;
  const float* val;
  const uint8_t* mask;
  float *dinv, *v, *y;
};
struct SetArgs {
  SetLev lev[kMaxLevels];
  int32_t first[kMaxLevels + 1];   // first block of each level, then the number of blocks
  int32_t n;
  double* part;                    // [blocks][2]
};

__device__ __forceinline__ int set_level(const SetArgs& S, int block) {
  int l = 0;
  while (l + 1 < S.n && block >= S.first[l + 1]) ++l;
  return l;
}

// D^-1, and the start of the power steps: pseudo-random, 0 on masked DoFs
__global__ __launch_bounds__(64) void k_mg_start(SetArgs S) {
  const int l = set_level(S, blockIdx.x);
  const SetLev& E = S.lev[l];
  const int64_t i = (int64_t)(blockIdx.x - S.first[l]) * 3 * kRowNodes + threadIdx.x;
  if (threadIdx.x >= 3 * kRowNodes || i >= 3 * E.N) return;
  const int64_t j = i / 3;
  const int d = (int)(i % 3);
  const float k = E.val[block32_at(E.nadj, E.adj_ptr[j] + E.dslot[j], 4 * d)];
  const float di = (E.mask[i] || !(k > 0.f)) ? 0.f : 1.f / k;
  E.dinv[i] = di;
  uint32_t h = (uint32_t)i * 2654435761u;
  h ^= h >> 15;
  h *= 2246822519u;
  h ^= h >> 13;
  E.v[i] = di > 0.f ? (float)(h & 0xFFFFu) / 65536.f - 0.5f : 0.f;
}

// One power step, D^-1 A, from v to y (or from y to v).  last: A v instead,
// only for the partials (v.A v, v.D v) of the Rayleigh quotient.
__global__ __launch_bounds__(kRowThreads) void k_mg_power(SetArgs S, int from_y, int last) {
  __shared__ float sh[3 * kRowNodes];
  const int l = set_level(S, blockIdx.x);
  const SetLev& E = S.lev[l];
  const int lb = blockIdx.x - S.first[l];
  const auto* __restrict__ x = gp((const float*)(from_y ? E.y : E.v));
  block_rows<float>(E.nadj, row_span(E.N, gp(E.adj_ptr), lb), gp(E.adj), gp(E.val), x, sh);
  if (threadIdx.x >= 64) return;
  const int64_t i = (int64_t)lb * 3 * kRowNodes + threadIdx.x;
  const bool own = threadIdx.x < 3 * kRowNodes && i < 3 * E.N;
  const float di = own ? gp(E.dinv)[i] : 0.f;
  if (!last) {
    if (own) gp(from_y ? E.v : E.y)[i] = di * sh[threadIdx.x];
    return;
  }
  double a = 0.0, b = 0.0;
  if (di > 0.f) {
    a = (double)x[i] * sh[threadIdx.x];
    b = (double)x[i] * x[i] / di;
  }
  a = wave_sum(a);
  b = wave_sum(b);
  if (threadIdx.x == 0) {
    S.part[2 * (int64_t)blockIdx.x] = a;
    S.part[2 * (int64_t)blockIdx.x + 1] = b;
  }
}

// Block per level: the largest eigenvalue of D^-1 A from the partials, and the
// smoother's 1 / theta, 1 / delta.
__global__ __launch_bounds__(kMB) void k_mg_lambda(SetArgs S, float* __restrict__ cheb) {
  __shared__ double sh[kMB];
  const int l = blockIdx.x;
  double a = 0.0, b = 0.0;
#pragma unroll 8
  for (int64_t i = S.first[l] + threadIdx.x; i < S.first[l + 1]; i += kMB) {
    a += S.part[2 * i];
    b += S.part[2 * i + 1];
  }
  a = msum(a, sh);
  b = msum(b, sh);
  if (threadIdx.x == 0) {
    double lmb = b > 0.0 ? a / b : 0.0;
    if (!(lmb > 0.0) || !isfinite(lmb)) lmb = 1.0;   // empty level: any positive scale
    cheb[2 * l] = (float)(1.0 / (0.5 * (kChebHi + kChebLo) * lmb));
    cheb[2 * l + 1] = (float)(1.0 / (0.5 * (kChebHi - kChebLo) * lmb));
  }
}

// Inverse of the coarsest operator, n <= 160, in one block: FP64 Gauss-Jordan on
// the diagonal, in place, each thread a 5x5 piece of the matrix in registers
// (rows ti + 32 r, columns tj + 32 c).  The operator is symmetric and positive
// definite but for rounding, so no pivot is searched for; one that is not
// clearly positive leaves *status = 1, and the host inverts with pivoting.
// Masked DoFs: identity in, zero out.  What bounds it is the chain of n steps,
// a barrier and a division each: 0.7 us a step, 98 us at n = 144 (265 us with a
// pivot search and 16 waves, 250 us with 4).  On the host
// the elimination took 0.8 ms at n = 96 and 2.8 ms at n = 144, with two copies
// and a wait around it.
constexpr int kInvT = 32, kInvR = 5, kInvMax = kInvT * kInvR;
constexpr double kInvTiny = 1e-10;   // of the diagonal's original value

__global__ __launch_bounds__(kInvT * kInvT) void k_mg_inverse(int n, int64_t NL, int64_t nadj,
                                                              const int64_t* __restrict__ adj_ptr,
                                                              const int32_t* __restrict__ adj,
                                                              const float* __restrict__ val,
                                                              const uint8_t* __restrict__ mask,
                                                              float* __restrict__ Ainv, double* __restrict__ status) {
  __shared__ double col[2][kInvMax], row[2][kInvMax];
  __shared__ float tiny[kInvMax];
  __shared__ uint8_t dead[kInvMax];
  constexpr int kT = kInvT * kInvT;
  const int t = threadIdx.x, ti = t / kInvT, tj = t % kInvT;
  for (int i = t; i < n * n; i += kT) Ainv[i] = 0.f;   // the dense matrix passes through the result's memory
  __syncthreads();
  for (int64_t j = ti; j < NL; j += kInvT)
    for (int64_t g = adj_ptr[j] + tj; g < adj_ptr[j + 1]; g += kInvT) {
      const int64_t i = adj[g];
      for (int e = 0; e < 9; ++e) Ainv[(3 * j + e / 3) * n + 3 * i + e % 3] = val[block32_at(nadj, g, e)];
    }
  __syncthreads();
  for (int i = t; i < n; i += kT) {
    const float d = Ainv[i * n + i];
    dead[i] = mask[i] || !(d > 0.f);
    tiny[i] = dead[i] ? 0.f : (float)kInvTiny * d;
  }
  __syncthreads();
  double a[kInvR][kInvR];
#pragma unroll
  for (int r = 0; r < kInvR; ++r)
#pragma unroll
    for (int c = 0; c < kInvR; ++c) {
      const int i = ti + kInvT * r, j = tj + kInvT * c;
      a[r][c] = 0.0;
      if (i < n && j < n) a[r][c] = dead[i] || dead[j] ? (i == j ? 1.0 : 0.0) : (double)Ainv[i * n + j];
    }
  __syncthreads();   // Ainv is written again only after this
  for (int k = 0; k < n; ++k) {
    double* C = col[k & 1];   // two of each: the step before may still be read
    double* R = row[k & 1];
#pragma unroll
    for (int q = 0; q < kInvR; ++q)
      if (q == k / kInvT) {   // column k and row k out, 0 in their place
        if (tj == k % kInvT)
#pragma unroll
          for (int r = 0; r < kInvR; ++r) C[ti + kInvT * r] = a[r][q];
        if (ti == k % kInvT)
#pragma unroll
          for (int c = 0; c < kInvR; ++c) R[tj + kInvT * c] = a[q][c];
        if (tj == k % kInvT)
#pragma unroll
          for (int r = 0; r < kInvR; ++r) a[r][q] = 0.0;
        if (ti == k % kInvT)
#pragma unroll
          for (int c = 0; c < kInvR; ++c) a[q][c] = 0.0;
      }
    __syncthreads();
    const double d = C[k];
    if (!(d > (double)tiny[k])) {   // the same in every thread
      if (t == 0) *status = 1.0;
      return;
    }
    const double inv = 1.0 / d;
    double rs[kInvR];
#pragma unroll
    for (int c = 0; c < kInvR; ++c) rs[c] = tj + kInvT * c == k ? inv : R[tj + kInvT * c] * inv;
#pragma unroll
    for (int r = 0; r < kInvR; ++r) {
      const double f = ti + kInvT * r == k ? -1.0 : C[ti + kInvT * r];
#pragma unroll
      for (int c = 0; c < kInvR; ++c) a[r][c] -= f * rs[c];
    }
  }
#pragma unroll
  for (int r = 0; r < kInvR; ++r)
#pragma unroll
    for (int c = 0; c < kInvR; ++c) {
      const int i = ti + kInvT * r, j = tj + kInvT * c;
      if (i < n && j < n) Ainv[i * n + j] = dead[i] || dead[j] ? 0.f : (float)a[r][c];
    }
  if (t == 0) *status = 0.0;
}

// per block: the largest off-diagonal block norm of node j, then strong flags
__global__ void k_mg_strength(int64_t N, const int64_t* __restrict__ adj_ptr, const int32_t* __restrict__ dslot,
                              const double* __restrict__ val64, double theta, uint8_t* __restrict__ strong) {
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= N) return;
  const int64_t a0 = adj_ptr[j];
  const int64_t R = adj_ptr[j + 1] - a0;
  const double* P = val64 + 9 * a0;    // panel [c][t][d]
  const int64_t self = dslot[j];
  double mx = 0.0;
  for (int64_t t = 0; t < R; ++t) {
    if (t == self) continue;
    double s = 0.0;
    for (int c = 0; c < 3; ++c)
      for (int d = 0; d < 3; ++d) {
        const double v = P[c * 3 * R + 3 * t + d];
        s += v * v;
      }
    mx = fmax(mx, s);
  }
  const double thr = theta * theta * mx;
  for (int64_t t = 0; t < R; ++t) {
    double s = 0.0;
    for (int c = 0; c < 3; ++c)
      for (int d = 0; d < 3; ++d) {
        const double v = P[c * 3 * R + 3 * t + d];
        s += v * v;
      }
    strong[a0 + t] = (t != self && s > 0.0 && s >= thr) ? 1 : 0;
  }
}

// ---- host hierarchy -------------------------------------------------------------

}  // namespace

// Host allocator for the large arrays of the hierarchy build: resize() leaves
// the elements uninitialised, so the first touch of a large array happens
// where it is filled -- in parallel threads -- rather than in a serial zero
// fill.
template <class T>
struct NoInitAlloc : std::allocator<T> {
  using value_type = T;
  template <class U>
  struct rebind {
    using other = NoInitAlloc<U>;
  };
  NoInitAlloc() = default;
  template <class U>
  NoInitAlloc(const NoInitAlloc<U>&) {}
  template <class U>
  void construct(U* p) noexcept {
    ::new (static_cast<void*>(p)) U;
  }
  template <class U, class... A>
  void construct(U* p, A&&... a) {
    ::new (static_cast<void*>(p)) U(std::forward<A>(a)...);
  }
};
template <class T>
using HVec = std::vector<T, NoInitAlloc<T>>;

namespace {

struct HostLevel {
  int64_t N = 0;                   // pseudo-nodes
  std::vector<int64_t> adj_ptr;    // level >= 1 only (level 0: the mesh's)
  std::vector<int32_t> adj, dslot;
  std::vector<uint8_t> mask;       // level >= 1 only
  // transfer (all but the coarsest)
  int64_t nagg = 0;
  std::vector<int32_t> agg;        // [N]
  HVec<float> Q;                   // [N][18]
  std::vector<int32_t> mem_ptr, mem;
  std::vector<int32_t> pair_o;     // [npairs][2]
  std::vector<int64_t> gptr;
  HVec<int32_t> gblk, gcol;
};

// Run f(lo, hi) over [0, n) split across host threads; serial below `grain`
// items (per-aggregate loops pass a small grain: on coarse levels there are
// few aggregates, each with many members).
template <class F>
void parallel_for(int64_t n, F&& f, int64_t grain = 4096) {
  const int64_t nt = std::max<int64_t>(1, std::min<int64_t>(std::thread::hardware_concurrency(), 16));
  if (n < grain || nt == 1) {
    f((int64_t)0, n);
    return;
  }
  std::vector<std::thread> th;
  const int64_t step = (n + nt - 1) / nt;
  for (int64_t t = 0; t < nt; ++t) {
    const int64_t lo = t * step, hi = std::min(n, lo + step);
    if (lo < hi) th.emplace_back([&f, lo, hi]() { f(lo, hi); });
  }
  for (auto& x : th) x.join();
}

// A graph over real nodes: the neighbours of i are idx[e], e in
// [ptr[i], ptr[i+1]), except i itself and, with `flag`, entries flagged 0.
struct Graph {
  const int64_t* ptr = nullptr;
  const int32_t* idx = nullptr;
  const uint8_t* flag = nullptr;
  template <class F>
  void each(int64_t i, F&& f) const {
    for (int64_t e = ptr[i]; e < ptr[i + 1]; ++e) {
      const int32_t j = idx[e];
      if (j == i || (flag && !flag[e])) continue;
      f(j);
    }
  }
};

// The aggregate the neighbours of i (through `from`) belong to most often;
// ties to the smallest id; -1 if none.
int32_t most_coupled(const Graph& g, int64_t i, const std::vector<int32_t>& from, std::vector<int32_t>& buf) {
  buf.clear();
  g.each(i, [&](int32_t j) {
    if (from[j] >= 0) buf.push_back(from[j]);
  });
  if (buf.empty()) return -1;
  std::sort(buf.begin(), buf.end());
  int32_t best = -1;
  size_t bc = 0;
  for (size_t k = 0; k < buf.size();) {
    size_t e = k;
    while (e < buf.size() && buf[e] == buf[k]) ++e;
    if (e - k > bc) {
      bc = e - k;
      best = buf[k];
    }
    k = e;
  }
  return best;
}

// Greedy aggregation over real nodes.  Returns the aggregate count; agg = -1
// for nodes with no neighbour at all.
int64_t aggregate(int64_t n, const Graph& S, const Graph& F, std::vector<int32_t>& agg) {
  agg.assign((size_t)n, -1);
  int64_t na = 0;
  for (int64_t i = 0; i < n; ++i) {   // phase 1: root + all strong neighbours, all unaggregated
    if (agg[i] >= 0) continue;
    bool ok = true, any = false;
    for (int64_t e = S.ptr[i]; e < S.ptr[i + 1]; ++e) {   // stops at the first aggregated one
      const int32_t j = S.idx[e];
      if (j == i || (S.flag && !S.flag[e])) continue;
      any = true;
      if (agg[j] >= 0) {
        ok = false;
        break;
      }
    }
    if (!ok || !any) continue;
    agg[i] = (int32_t)na;
    S.each(i, [&](int32_t j) { agg[j] = (int32_t)na; });
    ++na;
  }
  // phase 2: join the phase-1 aggregate coupled most strongly.  It reads the
  // phase-1 snapshot only, so the nodes are independent (host threads).
  std::vector<int32_t> snap = agg, buf;
  parallel_for(n, [&](int64_t lo, int64_t hi) {
    std::vector<int32_t> b;
    for (int64_t i = lo; i < hi; ++i)
      if (snap[i] < 0) agg[i] = most_coupled(S, i, snap, b);
  });
  for (int64_t i = 0; i < n; ++i) {   // phase 3a: leftovers with unaggregated strong neighbours
    if (agg[i] >= 0) continue;
    bool any = false;
    S.each(i, [&](int32_t j) { any = any || agg[j] < 0; });
    if (!any) continue;
    agg[i] = (int32_t)na;
    S.each(i, [&](int32_t j) {
      if (agg[j] < 0) agg[j] = (int32_t)na;
    });
    ++na;
  }
  for (int64_t i = 0; i < n; ++i) {   // phase 3b: weakly coupled nodes join, isolated ones stay out
    if (agg[i] >= 0) continue;
    const int32_t a = most_coupled(F, i, agg, buf);
    if (a >= 0) {
      agg[i] = a;
    } else {
      bool any = false;
      F.each(i, [&](int32_t) { any = true; });
      if (any) agg[i] = (int32_t)na++;
    }
  }
  return na;
}


// Modified Gram-Schmidt (two passes) of a rows x 6 matrix (row-major) in
// place; R (6x6, row-major) with B = Q R; dropped columns are zeroed in Q and
// their rows in R.
void mgs6(int64_t rows, double* M, double* R, bool* dropped) {
  std::fill(R, R + 36, 0.0);
  for (int u = 0; u < 6; ++u) {
    double n0 = 0.0;
    for (int64_t r = 0; r < rows; ++r) n0 += M[6 * r + u] * M[6 * r + u];
    n0 = std::sqrt(n0);
    for (int pass = 0; pass < 2; ++pass)
      for (int w = 0; w < u; ++w) {
        if (dropped[w]) continue;
        double c = 0.0;
        for (int64_t r = 0; r < rows; ++r) c += M[6 * r + w] * M[6 * r + u];
        for (int64_t r = 0; r < rows; ++r) M[6 * r + u] -= c * M[6 * r + w];
        R[6 * w + u] += c;
      }
    double nv = 0.0;
    for (int64_t r = 0; r < rows; ++r) nv += M[6 * r + u] * M[6 * r + u];
    nv = std::sqrt(nv);
    if (nv > 1e-10 * n0 && nv > 0.0) {
      dropped[u] = false;
      R[6 * u + u] = nv;
      for (int64_t r = 0; r < rows; ++r) M[6 * r + u] /= nv;
    } else {
      dropped[u] = true;
      for (int v = 0; v < 6; ++v) R[6 * u + v] = 0.0;
      for (int64_t r = 0; r < rows; ++r) M[6 * r + u] = 0.0;
    }
  }
}

}  // namespace

struct AmgHost {
  std::vector<HostLevel> lev;      // lev.back(): coarsest
  int64_t N0 = 0;
  double ms = 0.0;
};

// Input of the host build, gathered from the device by amg_gather.
struct AmgInput {
  int64_t N = 0;
  std::vector<int64_t> adj_ptr;
  HVec<int32_t> adj;
  std::vector<int32_t> dslot;
  HVec<uint8_t> strong;            // per block
  std::vector<double> xyz;         // SoA
  std::vector<uint8_t> mask;       // [3N]
};

struct AmgHier {
  struct Lev {
    int64_t N = 0, nadj = 0, nagg = 0, npairs = 0;
    const int64_t* adj_ptr = nullptr;
    const int32_t* adj = nullptr;
    const int32_t* dslot = nullptr;
    const uint8_t* mask = nullptr;
    const int32_t* agg = nullptr;
    const float* Q = nullptr;
    const int32_t* mem_ptr = nullptr;
    const int32_t* mem = nullptr;
    const int32_t* pair_o = nullptr;
    const int64_t* gptr = nullptr;
    const int32_t* gblk = nullptr;
    const int32_t* gcol = nullptr;
  };
  std::vector<Lev> lev;
  std::vector<int64_t> c_adj_ptr;  // host copy of the coarsest pattern
  std::vector<int32_t> c_adj;
  std::vector<uint8_t> c_mask;
  std::vector<std::pair<void*, size_t>> owned;
  size_t bytes = 0;
  double host_ms = 0.0;
};

namespace {

// Build level l+1 from level l.  Real nodes map to `ps` pseudo-nodes each
// (level 0: one; coarser: two).  nullrow(j, c, out6): near-null-space row of
// pseudo-node j, component c.  S, F: strong and full real-node graphs.
// Outputs the coarse level C, its near-null space Bc ([na][6][6]) and the
// aggregate graph (nbp, nbi; each list includes the aggregate itself).
template <class NullRow>
void coarsen(HostLevel& L, const int64_t* adj_ptr, const int32_t* adj, int ps, int64_t n_real, NullRow&& nullrow,
             const Graph& S, const Graph& F, HostLevel& C, std::vector<double>& Bc, std::vector<int64_t>& nbp,
             std::vector<int32_t>& nbi) {
  using clk = std::chrono::steady_clock;
  const bool trace = std::getenv("LLFEM_AMG_TRACE") != nullptr;
  auto tick = [&](const char* what, clk::time_point& t) {
    if (!trace) return;
    const auto now = clk::now();
    std::fprintf(stderr, "[amg]   N %lld %s %.1f ms\n", (long long)L.N, what,
                 std::chrono::duration<double, std::milli>(now - t).count());
    t = now;
  };
  auto tp = clk::now();
  std::vector<int32_t> ragg;
  const int64_t na = aggregate(n_real, S, F, ragg);
  tick("aggregate", tp);
  L.nagg = na;
  L.agg.assign((size_t)L.N, -1);
  for (int64_t a = 0; a < n_real; ++a)
    for (int s = 0; s < ps; ++s) L.agg[ps * a + s] = ragg[a];
  // members (pseudo-nodes, ascending)
  L.mem_ptr.assign((size_t)na + 1, 0);
  for (int64_t j = 0; j < L.N; ++j)
    if (L.agg[j] >= 0) L.mem_ptr[L.agg[j] + 1]++;
  for (int64_t a = 0; a < na; ++a) L.mem_ptr[a + 1] += L.mem_ptr[a];
  L.mem.assign((size_t)L.mem_ptr[na], 0);
  {
    std::vector<int32_t> fill(L.mem_ptr.begin(), L.mem_ptr.end() - 1);
    for (int64_t j = 0; j < L.N; ++j)
      if (L.agg[j] >= 0) L.mem[fill[L.agg[j]]++] = (int32_t)j;
  }
  tick("members", tp);
  // tentative prolongator and coarse near-null space (aggregates in parallel)
  L.Q.resize((size_t)L.N * 18);
  parallel_for(L.N, [&](int64_t lo, int64_t hi) { std::fill(L.Q.begin() + 18 * lo, L.Q.begin() + 18 * hi, 0.f); });
  Bc.assign((size_t)na * 36, 0.0);
  C.N = 2 * na;
  C.mask.assign((size_t)C.N * 3, 0);
  parallel_for(na, [&](int64_t lo, int64_t hi) {
    std::vector<double> M;
    for (int64_t a = lo; a < hi; ++a) {
      const int64_t m0 = L.mem_ptr[a], m1 = L.mem_ptr[a + 1];
      const int64_t rows = 3 * (m1 - m0);
      M.assign((size_t)rows * 6, 0.0);
      for (int64_t m = m0; m < m1; ++m)
        for (int c = 0; c < 3; ++c) nullrow(L.mem[m], c, &M[6 * (3 * (m - m0) + c)]);
      double R[36];
      bool dropped[6];
      mgs6(rows, M.data(), R, dropped);
      for (int64_t m = m0; m < m1; ++m) {
        const int64_t j = L.mem[m];
        for (int c = 0; c < 3; ++c)
          for (int u = 0; u < 6; ++u) L.Q[18 * j + 6 * c + u] = (float)M[6 * (3 * (m - m0) + c) + u];
      }
      for (int k = 0; k < 36; ++k) Bc[36 * a + k] = R[k];
      for (int u = 0; u < 6; ++u) C.mask[6 * a + u] = dropped[u] ? 1 : 0;
    }
  }, 64);
  tick("prolongator", tp);
  // per aggregate: neighbour aggregates (every fine block couples), then the
  // Galerkin contribution lists of its pairs, fine blocks in ascending order.
  // Two passes over the aggregates in parallel (sizes, then contents at
  // offsets from prefix sums): each aggregate's lists depend on it alone, so
  // the result does not depend on the thread count.
  nbp.assign((size_t)na + 1, 0);
  std::vector<int64_t> nblk((size_t)na + 1, 0);
  // neighbour aggregates of a, ascending, into nb (stamp: per-thread scratch)
  auto neighbours = [&](int64_t a, std::vector<int32_t>& stamp, std::vector<int32_t>& nb) {
    nb.clear();
    stamp[a] = (int32_t)a;
    nb.push_back((int32_t)a);
    for (int64_t m = L.mem_ptr[a]; m < L.mem_ptr[a + 1]; ++m) {
      const int64_t j = L.mem[m];
      for (int64_t g = adj_ptr[j]; g < adj_ptr[j + 1]; ++g) {
        const int32_t B = L.agg[adj[g]];
        if (B >= 0 && stamp[B] != a) {
          stamp[B] = (int32_t)a;
          nb.push_back(B);
        }
      }
    }
    std::sort(nb.begin(), nb.end());
  };
  parallel_for(na, [&](int64_t lo, int64_t hi) {
    std::vector<int32_t> stamp((size_t)na, -1), nb;
    for (int64_t a = lo; a < hi; ++a) {
      neighbours(a, stamp, nb);
      nbp[a + 1] = (int64_t)nb.size();
      int64_t c = 0;
      for (int64_t m = L.mem_ptr[a]; m < L.mem_ptr[a + 1]; ++m) {
        const int64_t j = L.mem[m];
        for (int64_t g = adj_ptr[j]; g < adj_ptr[j + 1]; ++g) c += L.agg[adj[g]] >= 0 ? 1 : 0;
      }
      nblk[a + 1] = c;
    }
  }, 64);
  for (int64_t a = 0; a < na; ++a) {
    nbp[a + 1] += nbp[a];
    nblk[a + 1] += nblk[a];
  }
  nbi.assign((size_t)nbp[na], 0);
  L.gptr.assign((size_t)nbp[na] + 1, 0);
  L.gblk.resize((size_t)nblk[na]);   // every element is written below
  L.gcol.resize((size_t)nblk[na]);
  parallel_for(na, [&](int64_t lo, int64_t hi) {
    std::vector<int32_t> stamp((size_t)na, -1), pos((size_t)na, 0), nb;
    std::vector<int64_t> cur;
    for (int64_t a = lo; a < hi; ++a) {
      neighbours(a, stamp, nb);
      const size_t k1 = nb.size();
      std::copy(nb.begin(), nb.end(), nbi.begin() + nbp[a]);
      for (size_t k = 0; k < k1; ++k) pos[nb[k]] = (int32_t)k;
      cur.assign(k1 + 1, 0);
      for (int64_t m = L.mem_ptr[a]; m < L.mem_ptr[a + 1]; ++m) {
        const int64_t j = L.mem[m];
        for (int64_t g = adj_ptr[j]; g < adj_ptr[j + 1]; ++g) {
          const int32_t B = L.agg[adj[g]];
          if (B >= 0) cur[pos[B] + 1]++;
        }
      }
      const int64_t base = nblk[a];
      for (size_t k = 0; k < k1; ++k) {
        cur[k + 1] += cur[k];
        L.gptr[nbp[a] + k + 1] = base + cur[k + 1];
      }
      for (int64_t m = L.mem_ptr[a]; m < L.mem_ptr[a + 1]; ++m) {
        const int64_t j = L.mem[m];
        for (int64_t g = adj_ptr[j]; g < adj_ptr[j + 1]; ++g) {
          const int32_t B = L.agg[adj[g]];
          if (B < 0) continue;
          const int64_t o = base + cur[pos[B]]++;
          L.gblk[o] = (int32_t)g;
          L.gcol[o] = (int32_t)j;
        }
      }
    }
  }, 64);
  tick("galerkin lists", tp);
  // coarse pseudo-node pattern: 2A and 2A+1 both list [2B, 2B+1 for B in nb(A)]
  const int64_t npairs = nbp[na];
  C.adj_ptr.assign((size_t)C.N + 1, 0);
  C.adj.assign((size_t)4 * npairs, 0);
  C.dslot.assign((size_t)C.N, 0);
  L.pair_o.assign((size_t)npairs * 2, 0);
  parallel_for(na, [&](int64_t lo, int64_t hi) {   // each aggregate writes its own ranges
    for (int64_t a = lo; a < hi; ++a) {
      const int64_t r = 2 * (nbp[a + 1] - nbp[a]);
      C.adj_ptr[2 * a] = 4 * nbp[a];
      C.adj_ptr[2 * a + 1] = 4 * nbp[a] + r;
      for (int s = 0; s < 2; ++s) {
        const int64_t o = 4 * nbp[a] + s * r;
        for (int64_t k = 0; k < nbp[a + 1] - nbp[a]; ++k) {
          const int32_t B = nbi[nbp[a] + k];
          C.adj[o + 2 * k] = 2 * B;
          C.adj[o + 2 * k + 1] = 2 * B + 1;
          if (B == a) C.dslot[2 * a + s] = (int32_t)(2 * k + s);
          L.pair_o[2 * (nbp[a] + k) + s] = (int32_t)(o + 2 * k);
        }
      }
    }
  }, 64);
  C.adj_ptr[2 * na] = 4 * nbp[na];
  tick("coarse pattern", tp);
}

}  // namespace

// Strong-coupling flags (GPU) and host copies of the pattern, coordinates and
// support mask: the inputs of the host hierarchy build.
int amg_gather(llfem_ctx* ctx, const SysSpec& sp, const double* d_xyz, AmgInput* in) {
  hipStream_t st = ctx->stream;
  const int64_t N = sp.N, nadj = sp.nadj;
  if (nadj >= ((int64_t)1 << 31)) return fail(LLFEM_EUNSUP, "AMG: more than 2^31 node blocks");
  uint8_t* d_strong = nullptr;
  LLFEM_TRY(dalloc(ctx, &d_strong, (size_t)nadj));
  k_mg_strength<<<nblk(N), kMB, 0, st>>>(N, sp.adj_ptr, sp.dslot, sp.val64, kStrength, d_strong);
  in->N = N;
  in->adj_ptr.resize((size_t)N + 1);
  in->adj.resize((size_t)nadj);
  in->dslot.resize((size_t)N);
  in->strong.resize((size_t)nadj);
  in->xyz.resize((size_t)3 * N);
  in->mask.resize((size_t)3 * N);
  // first touch of the uninitialised block arrays on all host threads, while
  // the strength kernel runs: the copies would otherwise take their page
  // faults one 4 KB page at a time in the runtime's copy loop
  auto touch = [](auto& v) {
    uint8_t* p = reinterpret_cast<uint8_t*>(v.data());
    const int64_t bytes = (int64_t)(v.size() * sizeof(v[0]));
    parallel_for((bytes + 4095) / 4096, [&](int64_t b, int64_t e) {
      for (int64_t i = b; i < e; ++i) p[i * 4096] = 0;
    });
  };
  touch(in->adj);
  touch(in->strong);
  hipError_t e = hipMemcpyAsync(in->adj_ptr.data(), sp.adj_ptr, sizeof(int64_t) * (N + 1), hipMemcpyDeviceToHost, st);
  if (e == hipSuccess) e = hipMemcpyAsync(in->adj.data(), sp.adj, sizeof(int32_t) * nadj, hipMemcpyDeviceToHost, st);
  if (e == hipSuccess) e = hipMemcpyAsync(in->dslot.data(), sp.dslot, sizeof(int32_t) * N, hipMemcpyDeviceToHost, st);
  if (e == hipSuccess) e = hipMemcpyAsync(in->strong.data(), d_strong, (size_t)nadj, hipMemcpyDeviceToHost, st);
  if (e == hipSuccess) e = hipMemcpyAsync(in->xyz.data(), d_xyz, sizeof(double) * 3 * N, hipMemcpyDeviceToHost, st);
  if (e == hipSuccess) e = hipMemcpyAsync(in->mask.data(), sp.fixed, (size_t)3 * N, hipMemcpyDeviceToHost, st);
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  drelease(ctx, d_strong, (size_t)nadj);
  if (e != hipSuccess) return fail(LLFEM_EHIP, std::string("AMG gather: ") + hipGetErrorString(e));
  return LLFEM_OK;
}

// The aggregation hierarchy (CPU only, no device calls: may run on any thread).
namespace {
// every value of v in [lo, hi), checked across host threads
template <class V>
bool all_in(const V& v, int64_t lo, int64_t hi) {
  std::atomic<bool> ok{true};
  parallel_for((int64_t)v.size(), [&](int64_t b, int64_t e) {
    bool o = true;
    for (int64_t i = b; i < e; ++i) o &= v[i] >= lo && v[i] < hi;
    if (!o) ok = false;
  });
  return ok;
}
}  // namespace

int amg_build_host(const AmgInput& in, AmgHost* H) {
  auto t0 = std::chrono::steady_clock::now();
  const int64_t N = in.N;
  H->N0 = N;
  H->lev.clear();
  H->lev.reserve(kMaxLevels + 1);
  H->lev.emplace_back();
  H->lev[0].N = N;
  // rigid-body modes about the centroid, constrained rows zeroed
  double c0[3] = {0, 0, 0};
  for (int k = 0; k < 3; ++k) {
    for (int64_t j = 0; j < N; ++j) c0[k] += in.xyz[(size_t)k * N + j];
    c0[k] /= std::max<int64_t>(N, 1);
  }
  auto rbm_row = [&](int64_t j, int c, double* out) {
    for (int u = 0; u < 6; ++u) out[u] = 0.0;
    if (in.mask[3 * j + c]) return;
    const double r[3] = {in.xyz[j] - c0[0], in.xyz[(size_t)N + j] - c0[1], in.xyz[(size_t)2 * N + j] - c0[2]};
    out[c] = 1.0;
    if (c == 0) { out[4] = r[2]; out[5] = -r[1]; }
    if (c == 1) { out[3] = -r[2]; out[5] = r[0]; }
    if (c == 2) { out[3] = r[1]; out[4] = -r[0]; }
  };
  std::vector<double> Bn, Bc;
  std::vector<int64_t> nbp, nbp_prev;
  std::vector<int32_t> nbi, nbi_prev;
  for (int l = 0;; ++l) {
    HostLevel C;
    if (l == 0) {
      const Graph S{in.adj_ptr.data(), in.adj.data(), in.strong.data()};
      const Graph F{in.adj_ptr.data(), in.adj.data(), nullptr};
      coarsen(H->lev[0], in.adj_ptr.data(), in.adj.data(), 1, N, rbm_row, S, F, C, Bc, nbp, nbi);
    } else {
      const HostLevel& L = H->lev[l];
      const Graph G{nbp_prev.data(), nbi_prev.data(), nullptr};
      auto row = [&](int64_t j, int c, double* out) {   // real node j/2, DoF 3 (j%2) + c
        const double* R = &Bn[(size_t)(j / 2) * 36 + 6 * (3 * (j % 2) + c)];
        for (int u = 0; u < 6; ++u) out[u] = R[u];
      };
      coarsen(H->lev[l], L.adj_ptr.data(), L.adj.data(), 2, L.N / 2, row, G, G, C, Bc, nbp, nbi);
    }
    const int64_t na = H->lev[l].nagg;
    const int64_t n_real = l == 0 ? N : H->lev[l].N / 2;
    if (na == 0) return fail(LLFEM_EUNSUP, "AMG: no aggregates (empty operator)");
    H->lev.push_back(std::move(C));
    if (na <= kCoarseAggs) break;
    if ((int)H->lev.size() >= kMaxLevels || 5 * na > 4 * n_real) {
      if (6 * na > kMaxDense) return fail(LLFEM_EUNSUP, "AMG: coarsening stalled");
      break;
    }
    Bn.swap(Bc);
    nbp_prev.swap(nbp);
    nbi_prev.swap(nbi);
  }
  const auto tc = std::chrono::steady_clock::now();
  // every index the kernels follow stays inside its array
  for (size_t l = 0; l + 1 < H->lev.size(); ++l) {
    const HostLevel& L = H->lev[l];
    const HostLevel& C = H->lev[l + 1];
    const int64_t nadj = l == 0 ? (int64_t)in.adj.size() : L.adj_ptr.back();
    const int64_t cnadj = C.adj_ptr.back();
    bool ok = (int64_t)L.agg.size() == L.N && (int64_t)L.Q.size() == 18 * L.N && C.N == 2 * L.nagg &&
              (int64_t)L.mem_ptr.size() == L.nagg + 1 && L.mem_ptr.back() == (int64_t)L.mem.size() &&
              (int64_t)L.gptr.size() == (int64_t)L.pair_o.size() / 2 + 1 &&
              L.gptr.back() == (int64_t)L.gblk.size() && L.gblk.size() == L.gcol.size() &&
              (int64_t)C.dslot.size() == C.N && (int64_t)C.mask.size() == 3 * C.N;
    ok = ok && all_in(L.agg, -1, L.nagg) && all_in(L.mem, 0, L.N) && all_in(L.gblk, 0, nadj) &&
         all_in(L.gcol, 0, L.N) && all_in(L.pair_o, 0, cnadj - 1) && all_in(C.adj, 0, C.N);
    for (int64_t j = 0; j < C.N && ok; ++j)
      ok = C.adj_ptr[j] <= C.adj_ptr[j + 1] && C.dslot[j] >= 0 && C.dslot[j] < C.adj_ptr[j + 1] - C.adj_ptr[j] &&
           C.adj[C.adj_ptr[j] + C.dslot[j]] == j;
    if (!ok) return fail(LLFEM_EINVAL, "AMG: inconsistent hierarchy at level " + std::to_string(l));
  }
  if (3 * H->lev.back().N > kMaxDense) return fail(LLFEM_EUNSUP, "AMG: coarsest level too large");
  H->ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  if (std::getenv("LLFEM_AMG_TRACE"))
    std::fprintf(stderr, "[amg]   index checks %.1f ms\n",
                 std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - tc).count());
  return LLFEM_OK;
}

void amg_free(llfem_ctx* ctx, AmgHier* h) {
  if (!h) return;
  for (auto& o : h->owned) dfree(ctx, o.first, o.second);
  delete h;
}

int amg_upload(llfem_ctx* ctx, const AmgHost& H, const SysSpec& sp, AmgHier** out) {
  hipStream_t st = ctx->stream;
  AmgHier* h = new AmgHier();
  h->host_ms = H.ms;
  int rc = LLFEM_OK;
  auto up = [&](const auto& v, auto** dst) -> int {
    using T = typename std::decay_t<decltype(v)>::value_type;
    *dst = nullptr;
    if (v.empty()) return LLFEM_OK;
    void* p = nullptr;
    LLFEM_TRY(dmalloc(ctx, &p, sizeof(T) * v.size()));
    h->owned.emplace_back(p, sizeof(T) * v.size());
    h->bytes += sizeof(T) * v.size();
    LLFEM_HIP(hipMemcpyAsync(p, v.data(), sizeof(T) * v.size(), hipMemcpyHostToDevice, st));
    *dst = static_cast<std::remove_const_t<std::remove_pointer_t<std::decay_t<decltype(*dst)>>>*>(p);
    return LLFEM_OK;
  };
  h->lev.resize(H.lev.size());
  for (size_t l = 0; l < H.lev.size() && rc == LLFEM_OK; ++l) {
    const HostLevel& L = H.lev[l];
    AmgHier::Lev& D = h->lev[l];
    D.N = L.N;
    D.nagg = L.nagg;
    D.npairs = (int64_t)L.pair_o.size() / 2;
    if (l == 0) {
      D.adj_ptr = sp.adj_ptr;
      D.adj = sp.adj;
      D.dslot = sp.dslot;
      D.mask = sp.fixed;
      D.nadj = sp.nadj;
    } else {
      D.nadj = L.adj_ptr.back();
      if ((rc = up(L.adj_ptr, &D.adj_ptr)) || (rc = up(L.adj, &D.adj)) || (rc = up(L.dslot, &D.dslot)) ||
          (rc = up(L.mask, &D.mask)))
        break;
    }
    if ((rc = up(L.agg, &D.agg)) || (rc = up(L.Q, &D.Q)) || (rc = up(L.mem_ptr, &D.mem_ptr)) ||
        (rc = up(L.mem, &D.mem)) || (rc = up(L.pair_o, &D.pair_o)) || (rc = up(L.gptr, &D.gptr)) ||
        (rc = up(L.gblk, &D.gblk)) || (rc = up(L.gcol, &D.gcol)))
      break;
  }
  if (rc == LLFEM_OK) {
    const HostLevel& C = H.lev.back();
    h->c_adj_ptr = C.adj_ptr;
    h->c_adj = C.adj;
    h->c_mask = C.mask;
    if (hipStreamSynchronize(st) != hipSuccess) rc = fail(LLFEM_EHIP, "AMG upload failed");
  }
  if (rc != LLFEM_OK) {
    (void)hipStreamSynchronize(st);
    amg_free(ctx, h);
    return rc;
  }
  *out = h;
  return LLFEM_OK;
}

int64_t amg_levels(const AmgHier* h) { return h ? (int64_t)h->lev.size() : 0; }
size_t amg_bytes(const AmgHier* h) { return h ? h->bytes : 0; }
double amg_host_ms(const AmgHier* h) { return h ? h->host_ms : 0.0; }

// ---- per-system numeric levels ----------------------------------------------------

struct AmgSys {
  const AmgHier* h = nullptr;
  void* mem = nullptr;
  size_t bytes = 0;
  std::vector<MgEnt> ent;          // one per level (the last: coarsest)
  double* status = nullptr;        // device word: 1 = k_mg_inverse has left the inverse to the host
  void* solo_tab = nullptr;
  std::vector<char> solo_src;      // host source of solo_tab's upload
  size_t solo_bytes = 0;
  struct Tab {
    MgEnt* ents = nullptr;
    int32_t *smap = nullptr, *vmap = nullptr, *amap = nullptr;
    int nent = 0;
    int64_t nsb = 0, nvb = 0, nab = 0;
    MgEnt* tents = nullptr;          // the levels of tails that begin on this level
    MgTail* tails = nullptr;
    int ntail = 0;
  };
  int tail = 0;                      // first level in the tail kernel
  std::vector<Tab> solo;
};

namespace {

// Chebyshev recurrence coefficients for the interval [lo, hi] x lambda: the
// same for every level and system (only theta and delta scale with lambda).
ChebSet cheb_coefs() {
  const double theta = 0.5 * (kChebHi + kChebLo), delta = 0.5 * (kChebHi - kChebLo);
  const double sigma = theta / delta;
  ChebSet cs{};
  double rho = 1.0 / sigma;
  for (int s = 1; s < kCheb; ++s) {   // pre: step 0 starts from x = 0
    const double rn = 1.0 / (2.0 * sigma - rho);
    cs.pre[s - 1] = {(float)(rn * rho), 0.f, (float)(2.0 * rn)};
    rho = rn;
  }
  rho = 1.0 / sigma;
  cs.post[0] = {0.f, 1.f, 0.f};
  for (int s = 1; s < kCheb; ++s) {
    const double rn = 1.0 / (2.0 * sigma - rho);
    cs.post[s] = {(float)(rn * rho), 0.f, (float)(2.0 * rn)};
    rho = rn;
  }
  return cs;
}

// Launch tables for a set of systems (block -> entry maps per level).
struct TabBuild {
  std::vector<std::vector<MgEnt>> ents, tents;
  std::vector<std::vector<MgTail>> tails;
  std::vector<std::vector<int32_t>> smap, vmap, amap;
};

void tab_add(TabBuild& T, const AmgSys* s, const double* state) {
  const int t = s->tail;
  if ((int)T.ents.size() < t + 1) {
    T.ents.resize(t + 1);
    T.tents.resize(t + 1);
    T.tails.resize(t + 1);
    T.smap.resize(t + 1);
    T.vmap.resize(t + 1);
    T.amap.resize(t + 1);
  }
  for (int l = 0; l < t; ++l) {
    MgEnt e = s->ent[l];
    e.state = state;
    const int32_t id = (int32_t)T.ents[l].size();
    e.sblk0 = (int32_t)T.smap[l].size();
    e.vblk0 = (int32_t)T.vmap[l].size();
    e.ablk0 = (int32_t)T.amap[l].size();
    T.smap[l].insert(T.smap[l].end(), (size_t)e.nsblk, id);
    T.vmap[l].insert(T.vmap[l].end(), (size_t)e.nvblk, id);
    T.amap[l].insert(T.amap[l].end(), (size_t)e.nablk, id);
    T.ents[l].push_back(e);
  }
  T.tails[t].push_back({(int32_t)T.tents[t].size(), (int32_t)(s->ent.size() - t)});
  for (size_t l = t; l < s->ent.size(); ++l) {
    T.tents[t].push_back(s->ent[l]);
    T.tents[t].back().state = state;
  }
}

// The tables in one copy.  src keeps their host source until the caller has
// next waited for the stream.  grow: room for the tables to double.
int tab_upload(llfem_ctx* ctx, const TabBuild& T, bool grow, void** mem, size_t* bytes, std::vector<char>* src,
               std::vector<AmgSys::Tab>* out) {
  size_t need = 0;
  auto al = [](size_t b) { return (b + 255) / 256 * 256; };
  for (size_t l = 0; l < T.ents.size(); ++l)
    need += al(sizeof(MgEnt) * T.ents[l].size()) + al(sizeof(MgEnt) * T.tents[l].size()) +
            al(sizeof(MgTail) * T.tails[l].size()) +
            al(4 * T.smap[l].size()) + al(4 * T.vmap[l].size()) + al(4 * T.amap[l].size());
  need += 256;
  if (*bytes < need) {
    if (*mem) dfree(ctx, *mem, *bytes);
    *mem = nullptr;
    *bytes = 0;
    const size_t room = grow ? need * 2 : need;
    LLFEM_TRY(dmalloc(ctx, mem, room));
    *bytes = room;
  }
  out->assign(T.ents.size(), AmgSys::Tab{});
  src->resize(need);
  size_t ofs = 0;
  auto put = [&](const void* p, size_t b) -> char* {
    if (b) std::memcpy(src->data() + ofs, p, b);
    char* d = static_cast<char*>(*mem) + ofs;
    ofs += al(b);
    return d;
  };
  for (size_t l = 0; l < T.ents.size(); ++l) {
    AmgSys::Tab& t = (*out)[l];
    t.nent = (int)T.ents[l].size();
    t.ntail = (int)T.tails[l].size();
    t.nsb = (int64_t)T.smap[l].size();
    t.nvb = (int64_t)T.vmap[l].size();
    t.nab = (int64_t)T.amap[l].size();
    t.ents = reinterpret_cast<MgEnt*>(put(T.ents[l].data(), sizeof(MgEnt) * T.ents[l].size()));
    t.tents = reinterpret_cast<MgEnt*>(put(T.tents[l].data(), sizeof(MgEnt) * T.tents[l].size()));
    t.tails = reinterpret_cast<MgTail*>(put(T.tails[l].data(), sizeof(MgTail) * T.tails[l].size()));
    t.smap = reinterpret_cast<int32_t*>(put(T.smap[l].data(), 4 * T.smap[l].size()));
    t.vmap = reinterpret_cast<int32_t*>(put(T.vmap[l].data(), 4 * T.vmap[l].size()));
    t.amap = reinterpret_cast<int32_t*>(put(T.amap[l].data(), 4 * T.amap[l].size()));
  }
  LLFEM_HIP(hipMemcpyAsync(*mem, src->data(), ofs, hipMemcpyHostToDevice, ctx->stream));
  return LLFEM_OK;
}

// head: level 0's first Chebyshev step is still to be done
int run_vcycle(llfem_ctx* ctx, const std::vector<AmgSys::Tab>& T, bool head) {
  hipStream_t st = ctx->stream;
  static const ChebSet cs = cheb_coefs();
  const int L = (int)T.size();
  // the iterate starts in y and changes array with each of the 2 kCheb - 1
  // (odd) smoothing steps, so it ends in x
  static_assert((2 * kCheb - 1) % 2 == 1, "the V-cycle's result has to end in x");
  for (int l = 0; l < L; ++l) {
    const AmgSys::Tab& t = T[l];
    if (t.ntail) k_mg_tail<<<(unsigned)t.ntail, kTB, 0, st>>>(t.tails, t.tents, cs, kOverCorrect);
    if (!t.nent) continue;
    int in_y = 1;
    if (l == 0 && head) k_mg_cheb0<<<(unsigned)t.nvb, kMB, 0, st>>>(t.ents, t.vmap, t.nent);
    for (const ChebCoef& c : cs.pre) {
      k_mg_smooth<<<(unsigned)t.nsb, kRowThreads, 0, st>>>(t.ents, t.smap, t.nent, c.ca, c.cbt, c.cbd, in_y, 0);
      in_y ^= 1;
    }
    k_mg_resid<<<(unsigned)t.nsb, kRowThreads, 0, st>>>(t.ents, t.smap, t.nent, in_y);
    k_mg_restrict<<<(unsigned)t.nab, kMB, 0, st>>>(t.ents, t.amap, t.nent, in_y ^ 1);
  }
  for (int l = L - 1; l >= 0; --l) {
    const AmgSys::Tab& t = T[l];
    if (!t.nent) continue;
    int in_y = kCheb % 2;
    k_mg_prolong<<<(unsigned)t.nvb, kMB, 0, st>>>(t.ents, t.vmap, t.nent, kOverCorrect, in_y);
    for (int s = 0; s < kCheb; ++s) {
      const ChebCoef& c = cs.post[s];
      k_mg_smooth<<<(unsigned)t.nsb, kRowThreads, 0, st>>>(t.ents, t.smap, t.nent, c.ca, c.cbt, c.cbd, in_y,
                                                           (l == 0 && s + 1 == kCheb) ? 1 : 0);
      in_y ^= 1;
    }
  }
  LLFEM_HIP(hipGetLastError());
  return LLFEM_OK;
}

// Dense inverse by Gauss-Jordan with partial pivoting (FP64, n <= kMaxDense).
bool invert_dense(int n, std::vector<double>& A) {
  std::vector<int> piv(n);
  std::iota(piv.begin(), piv.end(), 0);
  std::vector<double> I((size_t)n * n, 0.0);
  for (int i = 0; i < n; ++i) I[(size_t)i * n + i] = 1.0;
  for (int k = 0; k < n; ++k) {
    int p = k;
    for (int i = k + 1; i < n; ++i)
      if (std::fabs(A[(size_t)i * n + k]) > std::fabs(A[(size_t)p * n + k])) p = i;
    if (!(std::fabs(A[(size_t)p * n + k]) > 0.0)) return false;
    if (p != k)
      for (int j = 0; j < n; ++j) {
        std::swap(A[(size_t)p * n + j], A[(size_t)k * n + j]);
        std::swap(I[(size_t)p * n + j], I[(size_t)k * n + j]);
      }
    const double inv = 1.0 / A[(size_t)k * n + k];
    for (int j = 0; j < n; ++j) {
      A[(size_t)k * n + j] *= inv;
      I[(size_t)k * n + j] *= inv;
    }
    for (int i = 0; i < n; ++i) {
      if (i == k) continue;
      const double f = A[(size_t)i * n + k];
      if (f == 0.0) continue;
      for (int j = 0; j < n; ++j) {
        A[(size_t)i * n + j] -= f * A[(size_t)k * n + j];
        I[(size_t)i * n + j] -= f * I[(size_t)k * n + j];
      }
    }
  }
  A.swap(I);
  return true;
}

// Inverse of a coarsest operator that k_mg_inverse cannot hold (more than 26
// aggregates: coarsening stalled) or that is near singular.
int host_inverse(llfem_ctx* ctx, const AmgHier* h, const float* val, float* Ainv, double* status) {
  hipStream_t st = ctx->stream;
  const auto& D = h->lev.back();
  const int n = (int)(3 * D.N);
  std::vector<float> cval((size_t)9 * D.nadj);
  LLFEM_HIP(hipMemcpyAsync(cval.data(), val, sizeof(float) * cval.size(), hipMemcpyDeviceToHost, st));
  LLFEM_HIP(hipMemsetAsync(status, 0, sizeof(double), st));
  LLFEM_HIP(hipStreamSynchronize(st));
  std::vector<double> A((size_t)n * n, 0.0);
  for (int64_t j = 0; j < D.N; ++j)
    for (int64_t g = h->c_adj_ptr[j]; g < h->c_adj_ptr[j + 1]; ++g) {
      const int64_t i = h->c_adj[g];
      for (int c = 0; c < 3; ++c)
        for (int d = 0; d < 3; ++d)
          A[(size_t)(3 * j + c) * n + 3 * i + d] = cval[block32_at(D.nadj, g, 3 * c + d)];
    }
  std::vector<uint8_t> dead(n, 0);   // masked DoFs: identity in, zero out
  for (int i = 0; i < n; ++i) dead[i] = h->c_mask[i] || !(A[(size_t)i * n + i] > 0.0);
  for (int i = 0; i < n; ++i)
    if (dead[i]) {
      for (int k = 0; k < n; ++k) A[(size_t)i * n + k] = A[(size_t)k * n + i] = 0.0;
      A[(size_t)i * n + i] = 1.0;
    }
  if (!invert_dense(n, A)) return fail(LLFEM_EINVAL, "AMG: singular coarsest operator");
  std::vector<float> Af((size_t)n * n);
  for (int i = 0; i < n; ++i)
    for (int k = 0; k < n; ++k)
      Af[(size_t)i * n + k] = (dead[i] || dead[k]) ? 0.f : (float)A[(size_t)i * n + k];
  LLFEM_HIP(hipMemcpyAsync(Ainv, Af.data(), sizeof(float) * Af.size(), hipMemcpyHostToDevice, st));
  LLFEM_HIP(hipStreamSynchronize(st));
  return LLFEM_OK;
}

}  // namespace

void amg_sys_free(llfem_ctx* ctx, AmgSys* s) {
  if (!s) return;
  if (s->solo_tab) dfree(ctx, s->solo_tab, s->solo_bytes);
  if (s->mem) dfree(ctx, s->mem, s->bytes);
  delete s;
}

// Numeric levels of one system: Galerkin operators, inverse diagonals,
// Chebyshev bounds, dense coarsest inverse, launch tables for restarts.
// r, z, q: the system's FP32 residual, preconditioned residual and a free
// work vector (level 0's b, x and y); rzpart: where level 0 leaves the
// partial r.z per row block (row_groups(N) of them, as the engine's product).
int amg_sys_create(llfem_ctx* ctx, const AmgHier* h, const float* val32, float* r, float* z, float* q,
                   double* rzpart, AmgSys** out) {
  hipStream_t st = ctx->stream;
  const int L = (int)h->lev.size() - 1;   // coarsest index
  AmgSys* s = new AmgSys();
  s->h = h;
  // memory: level 0 dinv + d; levels 1..L: val, dinv, b, x, y, d; Ainv; reduction scratch
  auto al = [](size_t b) { return (b + 255) / 256 * 256; };
  const int64_t nc = 3 * h->lev[L].N;
  size_t need = al(4 * 3 * (size_t)h->lev[0].N) * 2;
  for (int l = 1; l <= L; ++l)
    need += al(4 * 9 * (size_t)h->lev[l].nadj) + 5 * al(4 * 3 * (size_t)h->lev[l].N);
  need += al(4 * (size_t)nc * nc);
  int64_t nset = 0;   // row blocks of the smoothed levels
  for (int l = 0; l < L; ++l) nset += row_groups(h->lev[l].N);
  need += al(sizeof(double) * (2 * (size_t)nset + (size_t)(L + 1) + 8));
  s->bytes = need;
  int rc = dmalloc(ctx, &s->mem, need);
  if (rc != LLFEM_OK) {
    delete s;
    return rc;
  }
  char* m = static_cast<char*>(s->mem);
  auto take = [&](size_t b) -> char* {
    char* p = m;
    m += al(b);
    return p;
  };
  s->ent.assign(L + 1, MgEnt{});
  std::vector<float*> val(L + 1), dinv(L + 1);
  val[0] = const_cast<float*>(val32);
  for (int l = 0; l <= L; ++l) {
    const auto& D = h->lev[l];
    MgEnt& e = s->ent[l];
    e.N = D.N;
    e.adj_ptr = D.adj_ptr;
    e.adj = D.adj;
    e.nadj = D.nadj;
    e.mask = D.mask;
    if (l == 0) {
      dinv[0] = (float*)take(4 * 3 * (size_t)D.N);
      e.d = (float*)take(4 * 3 * (size_t)D.N);
      e.b = r;
      e.x = z;
      e.y = q;
    } else {
      val[l] = (float*)take(4 * 9 * (size_t)D.nadj);
      dinv[l] = (float*)take(4 * 3 * (size_t)D.N);
      e.b = (float*)take(4 * 3 * (size_t)D.N);
      e.x = (float*)take(4 * 3 * (size_t)D.N);
      e.y = (float*)take(4 * 3 * (size_t)D.N);
      e.d = (float*)take(4 * 3 * (size_t)D.N);
    }
    e.val = val[l];
    e.dinv = dinv[l];
    e.nsblk = (int32_t)row_groups(D.N);   // as the engine's product
    e.nvblk = (int32_t)cap(3 * D.N, kMB, kMaxVB);
    e.agg = D.agg;
    e.Q = D.Q;
    e.mem_ptr = D.mem_ptr;
    e.mem = D.mem;
    e.nagg = D.nagg;
    e.nablk = (int32_t)cap(D.nagg, kMSpN, kMaxAB);
  }
  s->tail = L;
  for (int64_t n = h->lev[L].N; s->tail > 0; --s->tail) {
    n += h->lev[s->tail - 1].N;
    if (n > kTailN) break;
  }
  for (int l = 0; l < L; ++l) {
    s->ent[l].bc = s->ent[l + 1].b;
    s->ent[l].xc = s->ent[l + 1].x;
  }
  s->ent[0].rzpart = rzpart;
  float* Ainv = (float*)take(4 * (size_t)nc * nc);
  double* part = (double*)take(sizeof(double) * (2 * (size_t)nset + (size_t)(L + 1) + 8));
  s->status = part + 2 * nset;
  float* cheb = (float*)(s->status + 1);
  if ((size_t)(m - static_cast<char*>(s->mem)) > s->bytes) {
    amg_sys_free(ctx, s);
    return fail(LLFEM_EINVAL, "AMG: workspace layout overflow");
  }
  // Galerkin operators, inverse diagonals
  for (int l = 0; l < L; ++l) {
    const auto& D = h->lev[l];
    if (D.npairs < kGalPairs)
      k_galerkin<64><<<nblk(64 * D.npairs), kMB, 0, st>>>(D.npairs, D.nadj, h->lev[l + 1].nadj, D.gptr, D.gblk, D.gcol,
                                                          D.adj, D.Q, val[l], D.pair_o, val[l + 1]);
    else
      k_galerkin<16><<<nblk(16 * D.npairs), kMB, 0, st>>>(D.npairs, D.nadj, h->lev[l + 1].nadj, D.gptr, D.gblk, D.gcol,
                                                          D.adj, D.Q, val[l], D.pair_o, val[l + 1]);
  }
  // inverse diagonals; largest eigenvalue of D^-1 A per smoothed level (power
  // steps, Rayleigh quotient)
  SetArgs S{};
  S.n = L;
  S.part = part;
  for (int l = 0; l < L; ++l) {
    const auto& D = h->lev[l];
    S.lev[l] = {D.N, D.nadj, D.adj_ptr, D.adj, D.dslot, val[l], D.mask, dinv[l], s->ent[l].d, s->ent[l].y};
    S.first[l + 1] = S.first[l] + (int32_t)row_groups(D.N);
    s->ent[l].cheb = cheb + 2 * l;
  }
  k_mg_start<<<(unsigned)nset, 64, 0, st>>>(S);
  int from_y = 0;
  for (int k = 0; k < kPowerSteps; ++k, from_y ^= 1) k_mg_power<<<(unsigned)nset, kRowThreads, 0, st>>>(S, from_y, 0);
  k_mg_power<<<(unsigned)nset, kRowThreads, 0, st>>>(S, from_y, 1);
  k_mg_lambda<<<(unsigned)L, kMB, 0, st>>>(S, cheb);
  for (int l = 0; l + 1 < s->tail; ++l) {
    s->ent[l].yc = s->ent[l + 1].y;
    s->ent[l].dc = s->ent[l + 1].d;
    s->ent[l].dinvc = s->ent[l + 1].dinv;
    s->ent[l].chebc = s->ent[l + 1].cheb;
  }
  s->ent[L].Ainv = Ainv;
  s->ent[L].nc = (int32_t)nc;
  if (nc <= kInvMax) {
    const auto& D = h->lev[L];
    k_mg_inverse<<<1, kInvT * kInvT, 0, st>>>((int)nc, D.N, D.nadj, D.adj_ptr, D.adj, val[L], D.mask, Ainv, s->status);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
      amg_sys_free(ctx, s);
      return fail(LLFEM_EHIP, std::string("AMG set-up: ") + hipGetErrorString(e));
    }
  } else if ((rc = host_inverse(ctx, h, val[L], Ainv, s->status)) != LLFEM_OK) {
    amg_sys_free(ctx, s);
    return rc;
  }
  // restart tables (this system alone, always runs)
  TabBuild T;
  tab_add(T, s, nullptr);
  rc = tab_upload(ctx, T, false, &s->solo_tab, &s->solo_bytes, &s->solo_src, &s->solo);
  if (rc != LLFEM_OK) {
    amg_sys_free(ctx, s);
    return rc;
  }
  *out = s;
  return LLFEM_OK;
}

// z = M r for one system (reliable-update restarts); partial r.z as above.
// amg_batch_apply expects amg_head's step done.
int amg_apply_solo(llfem_ctx* ctx, AmgSys* s) { return run_vcycle(ctx, s->solo, true); }

// Level 0's first Chebyshev step, for the kernel that writes its right-hand
// side: *y = *d = theta[0] dinv b.  False: the tail kernel does it.
bool amg_head(const AmgSys* s, float** y, float** d, const float** dinv, const float** theta) {
  if (s->tail == 0) return false;
  const MgEnt& e = s->ent[0];
  *y = e.y;
  *d = e.d;
  *dinv = e.dinv;
  *theta = e.cheb;
  return true;
}

struct AmgBatch {
  std::vector<char> src;
  void* mem = nullptr;
  size_t bytes = 0;
  std::vector<AmgSys::Tab> tab;
};

// Tables of one V-cycle launch over several systems; states[i]: system i's
// state word (its V-cycle runs while the word reads 0).
int amg_batch_build(llfem_ctx* ctx, const std::vector<AmgSys*>& sys, const std::vector<const double*>& states,
                    AmgBatch** b) {
  if (!*b) *b = new AmgBatch();
  TabBuild T;
  for (size_t i = 0; i < sys.size(); ++i) tab_add(T, sys[i], states[i]);
  if (sys.empty()) {
    (*b)->tab.clear();
    return LLFEM_OK;
  }
  return tab_upload(ctx, T, true, &(*b)->mem, &(*b)->bytes, &(*b)->src, &(*b)->tab);
}

int amg_batch_apply(llfem_ctx* ctx, AmgBatch* b) {
  if (!b || b->tab.empty()) return LLFEM_OK;
  return run_vcycle(ctx, b->tab, false);
}

bool amg_batch_any(const AmgBatch* b) { return b && !b->tab.empty(); }

void amg_batch_free(llfem_ctx* ctx, AmgBatch* b) {
  if (!b) return;
  if (b->mem) dfree(ctx, b->mem, b->bytes);
  delete b;
}

const double* amg_status(const AmgSys* s) { return s->status; }

int amg_host_inverse(llfem_ctx* ctx, AmgSys* s) {
  const MgEnt& e = s->ent.back();
  return host_inverse(ctx, s->h, e.val, const_cast<float*>(e.Ainv), s->status);
}

int amg_build(llfem_ctx* ctx, const SysSpec& sp, const double* d_xyz, AmgHier** out) {
  using clk = std::chrono::steady_clock;
  const auto t0 = clk::now();
  AmgInput in;
  LLFEM_TRY(amg_gather(ctx, sp, d_xyz, &in));
  const auto t1 = clk::now();
  AmgHost H;
  LLFEM_TRY(amg_build_host(in, &H));
  const auto t2 = clk::now();
  const int rc = amg_upload(ctx, H, sp, out);
  if (std::getenv("LLFEM_AMG_TRACE")) {   // set-up phases, wall clock
    (void)hipStreamSynchronize(ctx->stream);
    const auto t3 = clk::now();
    auto ms = [](clk::time_point a, clk::time_point b) { return std::chrono::duration<double, std::milli>(b - a).count(); };
    std::fprintf(stderr, "[amg] N %lld: gather %.1f ms, host build %.1f ms, upload %.1f ms\n", (long long)sp.N,
                 ms(t0, t1), ms(t1, t2), ms(t2, t3));
  }
  return rc;
}

// Asynchronous build: the device gather runs at once, the host build on a
// thread of its own, the upload when the caller collects the job.
struct AmgJob {
  std::future<int> fut;
  AmgInput in;
  AmgHost host;
  std::string err;
};

int amg_job_start(llfem_ctx* ctx, const SysSpec& sp, const double* d_xyz, AmgJob** out) {
  AmgJob* j = new AmgJob();
  int rc = amg_gather(ctx, sp, d_xyz, &j->in);
  if (rc != LLFEM_OK) {
    delete j;
    return rc;
  }
  j->fut = std::async(std::launch::async, [j]() {
    const int r = amg_build_host(j->in, &j->host);
    if (r != LLFEM_OK) j->err = llfem_last_error();
    return r;
  });
  *out = j;
  return LLFEM_OK;
}

bool amg_job_ready(AmgJob* j) {
  return j->fut.wait_for(std::chrono::seconds(0)) == std::future_status::ready;
}

void amg_job_drop(AmgJob* j) {
  if (!j) return;
  j->fut.wait();
  delete j;
}

int amg_job_finish(llfem_ctx* ctx, AmgJob* j, const SysSpec& sp, AmgHier** out) {
  int rc = j->fut.get();
  if (rc == LLFEM_OK) rc = amg_upload(ctx, j->host, sp, out);
  else set_error(j->err);
  delete j;
  return rc;
}

}  // namespace llfem
