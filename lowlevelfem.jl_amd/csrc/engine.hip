// Batched mixed-precision PCG engine: FP32 Krylov iterations with FP64
// reliable updates, Jacobi or AMG preconditioner, many systems per launch.
//
// Reference: solveDisplacement(K, f; support, iterative=true, reltol, ...)
// (src/linear.jl:3711-3743): u = u_fixed on the constrained DoFs and
// K_ff u_f = f_f - K_fc u_c by preconditioned CG, converged at
// ||r|| <= reltol ||r0||.  Here the convergence test is made on the TRUE
// FP64 residual ||b - K x|| <= reltol ||b|| (b = the eliminated right-hand
// side), so the mixed-precision result meets the same relative residual as
// the FP64 solver.
//
// Algorithm (reliable updates, Sleijpen & van der Vorst 1996, as used for
// mixed-precision CG in lattice QCD solvers):
//   * CG runs in FP32 on K32 (the assembled panels rounded to FP32) with the
//     residual scaled to unit norm; dot products accumulate in FP64.
//   * The FP32 correction x32 is folded into the FP64 solution and the true
//     residual r = b - K x is recomputed in FP64 whenever the recursive
//     residual has dropped by delta (0.1) since the last update, or reaches
//     the tolerance.  The search direction p is kept (rescaled), so the
//     Krylov process is not restarted and the iteration count stays close to
//     the FP64 solver's.
//
// Batching: every launch covers all RUNNING systems.  Blocks map to systems
// through per-launch tables; each system's rows are split into blocks that
// depend on that system only and its dot products reduce in a fixed order,
// so a system's iterates are bit-identical whether it runs alone or among
// others.  A system that needs a reliable update pauses (its blocks exit at
// once) until the host performs the update between chunks of iterations.
#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "block32.h"
#include "common.h"
#include "engine_policy.h"

namespace llfem {

namespace {

constexpr int kSB = 256;                 // threads per block
constexpr int kVecNodes = kSB;           // nodes per vector block pass
// Vector blocks per system are capped (they stride over the system's nodes).
// The product's are not: 2,048 striding blocks of 8 lanes a row over 36-byte
// records took 627 us at 2.1 M nodes (tet10, 59.5 M blocks), one block per 16
// rows of block32.h's layout 515 us (4.6 TB/s).  Its partials lie in y, which
// is free between updates; more than kFoldMax of them (16 per thread of a
// summing block) are summed by kFoldBlocks blocks first, a 4 to 6 us launch.
constexpr int64_t kMaxVecBlocks = 1024;
constexpr int64_t kFoldMax = 4096;
constexpr int kFoldBlocks = 64;

// scal words of a system; SC_RHOP: r.z that the running iteration began with,
// SC_LAST: iteration count at the last FP64 update, SC_MAXRUN: force an update
// after this many iterations (0: never)
enum { SC_RHO = 0, SC_RHOP, SC_RR, SC_MAXRR, SC_TOL2, SC_DELTA2, SC_STATE, SC_ITER, SC_LAST, SC_MAXRUN, SC_N = 16 };
enum { ST_RUN = 0, ST_PENDING = 1, ST_PAUSED = 2, ST_IDLE = 3 };

struct SysDev {
  int64_t N;               // nodes (3 DoFs each)
  const int64_t* adj_ptr;
  const int32_t* adj;
  int64_t nadj;
  const float* val;        // FP32 node blocks (block32.h)
  const uint8_t* fixed;    // [3N] 1 = constrained
  const float* dinv;       // [N][3] inverse diagonal (0 on constrained DoFs)
  void *x, *r, *z, *p, *q; // Krylov vectors, FP32 or FP64 (the kernels' VT)
  double* scal;            // [SC_N]
  double* spart;           // [nsblk] partials of a product, then [kFoldBlocks] sums of them if nsblk > kFoldMax
  double* part;            // [nvblk][2] (r.r, r.z) of a vector kernel
  float *mgy, *mgd;        // AMG: the V-cycle's first step y = d = mgt[0] mgdinv r goes here (NULL: the tail kernel does it)
  const float *mgdinv, *mgt;
  int32_t sblk0, nsblk, vblk0, nvblk;
  int32_t amg;             // 1: z and the r.z partials (in spart) come from the AMG V-cycle
};

// Sum over the block's four waves in a fixed order; sh may be used again at once.
__device__ __forceinline__ double bsum(double v, double* sh) {
  v = wave_sum(v);
  if (threadIdx.x % 64 == 0) sh[threadIdx.x / 64] = v;
  __syncthreads();
  const double r = (sh[0] + sh[1]) + (sh[2] + sh[3]);
  __syncthreads();
  return r;
}

// system of a block; the map is a dependent load that one system needs none of
__device__ __forceinline__ const SysDev& sys_of(const SysDev* sys, const int32_t* bsys, int nsys) {
  return sys[nsys == 1 ? 0 : bsys[blockIdx.x]];
}

// This thread's share of the sum of q[i * stride], i < n, over the block, eight
// loads under way: one at a time, 3,165 partials took 5 us on an idle chip.
__device__ __forceinline__ double own_strided(const double* q, int n, int stride) {
  double v = 0.0;
  for (int i0 = threadIdx.x; i0 < n; i0 += 8 * kSB) {
    double a[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int i = i0 + k * kSB;
      a[k] = i < n ? q[(int64_t)stride * i] : 0.0;
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) v += a[k];
  }
  return v;
}
__device__ __forceinline__ double sum_strided(const double* q, int n, int stride, double* sh) {
  return bsum(own_strided(q, n, stride), sh);
}

// q = mask(K32 p) for RUNNING systems; partial p.q per block.
template <typename VT>
__global__ __launch_bounds__(kRowThreads) void k_bs_spmv(const SysDev* __restrict__ sys,
                                                         const int32_t* __restrict__ bsys, int nsys) {
  __shared__ VT sh[3 * kRowNodes];
  const SysDev& S = sys_of(sys, bsys, nsys);
  const int lb = blockIdx.x - pinned(S.sblk0);
  const int64_t N = pinned(S.N), nadj = pinned(S.nadj);
  const auto ap = gp(pinned(S.adj_ptr));
  const auto adj = gp(pinned(S.adj));
  const auto val = gp(pinned(S.val));
  const auto* __restrict__ pv = gp(static_cast<const VT*>(pinned(S.p)));
  VT* const q = static_cast<VT*>(pinned(S.q));
  const uint8_t* const fixed = pinned(S.fixed);
  double* const spart = pinned(S.spart);
  const double st = gp(pinned(S.scal))[SC_STATE];
  const RowSpan rs = row_span(N, ap, lb);
  if (st != ST_RUN) return;   // no block writes it here
  const int64_t i = (int64_t)lb * 3 * kRowNodes + threadIdx.x;
  const bool own = threadIdx.x < 3 * kRowNodes && i < 3 * N;
  VT pi = 0;
  uint8_t fi = 1;
  if (own) {   // loaded now, beside the product's
    pi = pv[i];
    fi = gp(fixed)[i];
  }
  block_rows<VT>(nadj, rs, adj, val, pv, sh);
  if (threadIdx.x >= 64) return;
  double d = 0.0;
  if (own) {
    const VT v = fi ? (VT)0 : sh[threadIdx.x];
    gp(q)[i] = v;
    d = (double)pi * (double)v;
  }
  d = wave_sum(d);
  if (threadIdx.x == 0) gp(spart)[lb] = d;
}

// spart of systems with more than kFoldMax product blocks -> kFoldBlocks sums
// of contiguous runs, behind them.  kFoldBlocks blocks per system.
__global__ __launch_bounds__(kSB) void k_bs_fold(const SysDev* __restrict__ sys) {
  __shared__ double sh[kSB / 64];
  const SysDev& S = sys[blockIdx.x / kFoldBlocks];
  if (S.nsblk <= kFoldMax || S.scal[SC_STATE] != ST_RUN) return;
  const int b = blockIdx.x % kFoldBlocks;
  const int per = (S.nsblk + kFoldBlocks - 1) / kFoldBlocks, i1 = min(S.nsblk, (b + 1) * per);
  double v = 0.0;
  for (int i = b * per + threadIdx.x; i < i1; i += kSB) v += S.spart[i];
  v = bsum(v, sh);
  if (threadIdx.x == 0) S.spart[S.nsblk + b] = v;
}

__device__ __forceinline__ double own_spart(const SysDev& S) {
  const double* q = S.spart + (S.nsblk > kFoldMax ? S.nsblk : 0);
  return own_strided(q, S.nsblk > kFoldMax ? kFoldBlocks : S.nsblk, 1);
}

// alpha = rho / p.q; x += alpha p; r -= alpha q; z = Dinv r; partials
// (r.r, r.z).  Thread per node.  Every block sums the product's partials for
// itself, in the same order, instead of reading alpha from a launch of one
// block per system (4 us each for alpha and beta; eight systems on a server
// 41.5 -> 38.8 ms); block 0 keeps the words.  A system flagged PENDING at the
// end of the previous iteration becomes PAUSED here, and one that breaks down
// does so too, while later blocks still read the word: waves of one block may
// read RUN and PAUSED.  So none leaves by itself.  A wave that does not read RUN
// puts NaN into the block's sum in place of its share, and the block leaves as
// one where that sum is not positive: at a breakdown, which it finds by itself,
// or because some wave saw the system paused.  (The word read by one thread and
// handed on through LDS, with a barrier of its own, cost eight systems on a
// server 0.8 %.)
template <typename VT>
__global__ __launch_bounds__(kSB) void k_bs_update(const SysDev* __restrict__ sys, const int32_t* __restrict__ bsys,
                                                   int nsys) {
  __shared__ double sh[kSB / 64];
  const SysDev& S = sys_of(sys, bsys, nsys);
  const int lb = blockIdx.x - S.vblk0;
  const bool keeper = lb == 0 && threadIdx.x == 0;
  const double st = S.scal[SC_STATE];
  const bool run = st == ST_RUN;   // of this wave
  auto* __restrict__ xv = gp(static_cast<VT*>(S.x));
  auto* __restrict__ rv = gp(static_cast<VT*>(S.r));
  auto* __restrict__ zv = gp(static_cast<VT*>(S.z));
  const auto* __restrict__ pv = gp(static_cast<const VT*>(S.p));
  const auto* qv = gp(static_cast<const VT*>(S.q));   // may be mgy
  const auto* __restrict__ dinv = gp(S.dinv);
  int64_t j = (int64_t)lb * kVecNodes + threadIdx.x;
  VT x[3], p[3], r[3], q[3];   // of the node under way; the first one's load beside the partials
  auto load = [&]() {
    if (j < S.N)
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        x[c] = xv[3 * j + c];
        p[c] = pv[3 * j + c];
        r[c] = rv[3 * j + c];
        q[c] = qv[3 * j + c];
      }
  };
  if (run) load();
  const double rho = S.scal[SC_RHO], pq = bsum(run ? own_spart(S) : (double)NAN, sh);
  if (!(pq > 0.0)) {   // paused, or a breakdown (p = 0 or K not SPD on the free set): check the true residual
    if (keeper && (run || st == ST_PENDING)) S.scal[SC_STATE] = ST_PAUSED;
    return;
  }
  if (keeper) S.scal[SC_RHOP] = rho;
  const VT alpha = (VT)(rho / pq);
  double rr = 0.0, rz = 0.0;
  for (; j < S.N; j += (int64_t)S.nvblk * kVecNodes, load()) {
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      xv[3 * j + c] = x[c] + alpha * p[c];
      r[c] -= alpha * q[c];
      rv[3 * j + c] = r[c];
      rr += (double)r[c] * (double)r[c];
    }
    if (S.amg) {
      if (S.mgy)   // q, whose values are used up, is the level's y
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          const int64_t i = 3 * j + c;
          const float v = gp(S.mgt)[0] * gp(S.mgdinv)[i] * (float)r[c];
          gp(S.mgy)[i] = v;
          gp(S.mgd)[i] = v;
        }
      continue;
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const VT z = (VT)dinv[3 * j + c] * r[c];
      zv[3 * j + c] = z;
      rz += (double)r[c] * (double)z;
    }
  }
  rr = bsum(rr, sh);
  rz = bsum(rz, sh);
  if (threadIdx.x == 0) {
    S.part[2 * lb] = rr;
    if (!S.amg) S.part[2 * lb + 1] = rz;
  }
}

// beta = r.z / rho; p = z + beta p; reliable-update / convergence triggers.
// The sums as in k_bs_update; block 0 writes no word that another block reads
// but the state, which only turns from RUN to PENDING here, and both finish
// their iteration: waves of a block that read one and the other stay together.
template <typename VT>
__global__ __launch_bounds__(kSB) void k_bs_pupd(const SysDev* __restrict__ sys, const int32_t* __restrict__ bsys,
                                                 int nsys) {
  __shared__ double sh[kSB / 64];
  const SysDev& S = sys_of(sys, bsys, nsys);
  const double st = S.scal[SC_STATE];
  if (st != ST_RUN && st != ST_PENDING) return;   // the same in every wave
  const int lb = blockIdx.x - S.vblk0;
  auto* __restrict__ pv = gp(static_cast<VT*>(S.p));
  const auto* __restrict__ zv = gp(static_cast<const VT*>(S.z));
  int64_t j = (int64_t)lb * kVecNodes + threadIdx.x;
  VT z[3], p[3];   // of the node under way; the first one's load beside the partials
  auto load = [&]() {
    if (j < S.N)
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        z[c] = zv[3 * j + c];
        p[c] = pv[3 * j + c];
      }
  };
  load();
  const double rho = S.scal[SC_RHOP];
  const double rz = S.amg ? bsum(own_spart(S), sh) : sum_strided(S.part + 1, S.nvblk, 2, sh);
  if (lb == 0) {
    const double rr = sum_strided(S.part, S.nvblk, 2, sh);
    if (threadIdx.x == 0) {
      S.scal[SC_RHO] = rz;
      S.scal[SC_RR] = rr;
      S.scal[SC_ITER] += 1.0;
      const double maxrun = S.scal[SC_MAXRUN];
      if (rr <= S.scal[SC_TOL2] || rr < S.scal[SC_DELTA2] * S.scal[SC_MAXRR] || !(rz > 0.0) ||
          (maxrun > 0.0 && S.scal[SC_ITER] - S.scal[SC_LAST] >= maxrun))
        S.scal[SC_STATE] = ST_PENDING;
    }
  }
  const VT beta = (VT)(rho != 0.0 ? rz / rho : 0.0);
  for (; j < S.N; j += (int64_t)S.nvblk * kVecNodes, load())
#pragma unroll
    for (int c = 0; c < 3; ++c) pv[3 * j + c] = z[c] + beta * p[c];
}

__global__ void k_bs_states(const SysDev* __restrict__ sys, int nsys, double* __restrict__ out) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= nsys) return;
  out[2 * s] = sys[s].scal[SC_STATE];
  out[2 * s + 1] = sys[s].scal[SC_ITER];
}

// ---- single-system kernels of the reliable update ------------------------------

// trial solution xt = xh + x / s (xh is kept until xt is known to be finite); x = 0
template <typename VT>
__global__ void k_ru_trial(int64_t n, VT* __restrict__ x, double inv_s, const double* __restrict__ xh,
                           double* __restrict__ xt) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  xt[i] = xh[i] + (double)x[i] * inv_s;
  x[i] = (VT)0;
}

// y = mask(K64 x) (mask may be NULL), kG lanes a row (panel_lanes).  us with 8,
// 16, 32 lanes: tet4 (14 to 15 blocks a row) 42,875 nodes 11.3, 11.3, 13.4 and
// 753,571 nodes 178, 160, 231; hex8 (26) 68,921 nodes 29.6, 23.4, 24.7 and
// 912,673 nodes 394, 341, 348; tet10 (28) 4,913 nodes 5.0, 4.5, 4.2 and 117,649
// nodes 53.8, 42.7, 41.9; hex27 (61) 91,125 nodes 107, 85, 78.
template <int kG>
__global__ __launch_bounds__(kSB) void k_spmv64(int64_t N, const int64_t* __restrict__ adj_ptr,
                                                const int32_t* __restrict__ adj, const double* __restrict__ val,
                                                const double* __restrict__ x, const uint8_t* __restrict__ fixed,
                                                double* __restrict__ y) {
  const int64_t gt = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t j = gt / kG;
  const int l = (int)(gt % kG);
  double a0 = 0, a1 = 0, a2 = 0;
  if (j < N) {
    const int64_t p0 = adj_ptr[j];
    const int R = (int)(adj_ptr[j + 1] - p0);
    const double* P = val + 9 * p0;
    for (int t = l; t < R; t += kG) {
      const int64_t i = adj[p0 + t];
      const double x0 = x[3 * i], x1 = x[3 * i + 1], x2 = x[3 * i + 2];
      a0 += P[3 * t] * x0 + P[3 * t + 1] * x1 + P[3 * t + 2] * x2;
      a1 += P[3 * R + 3 * t] * x0 + P[3 * R + 3 * t + 1] * x1 + P[3 * R + 3 * t + 2] * x2;
      a2 += P[6 * R + 3 * t] * x0 + P[6 * R + 3 * t + 1] * x1 + P[6 * R + 3 * t + 2] * x2;
    }
  }
#pragma unroll
  for (int o = kG / 2; o > 0; o >>= 1) {
    a0 += __shfl_xor(a0, o, kG);
    a1 += __shfl_xor(a1, o, kG);
    a2 += __shfl_xor(a2, o, kG);
  }
  if (j < N && l == 0) {
    const double a[3] = {a0, a1, a2};
#pragma unroll
    for (int c = 0; c < 3; ++c) y[3 * j + c] = (fixed && fixed[3 * j + c]) ? 0.0 : a[c];
  }
}

// out = mask(b - y) (y may be NULL: out = mask(b)); partial sum of out^2 per block
__global__ __launch_bounds__(kSB) void k_ru_resid(int64_t n, const double* __restrict__ b, const double* __restrict__ y,
                                                  const uint8_t* __restrict__ fixed, double* __restrict__ out,
                                                  double* __restrict__ part) {
  __shared__ double sh[kSB / 64];
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  double v = 0.0;
  if (i < n) {
    v = fixed[i] ? 0.0 : b[i] - (y ? y[i] : 0.0);
    if (out) out[i] = v;
  }
  const double s = bsum(v * v, sh);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// scal[SC_STATE] = v (one thread; an eager write that needs no host copy)
__global__ void k_set_state(double* __restrict__ scal, double v) { scal[SC_STATE] = v; }

__global__ __launch_bounds__(kSB) void k_sum(int64_t n, const double* __restrict__ part, double* __restrict__ out) {
  __shared__ double sh[kSB / 64];
  double v = 0.0;
  for (int64_t i = threadIdx.x; i < n; i += kSB) v += part[i];
  v = bsum(v, sh);
  if (threadIdx.x == 0) out[0] = v;
}

// r = rh * s; p = pscale * p (= z when init); z = Dinv r; partials (r.r, r.z)
template <typename VT>
__global__ __launch_bounds__(kSB) void k_ru_restart(int64_t N, const double* __restrict__ rh, double s, double pscale,
                                                    int init, const float* __restrict__ dinv, VT* __restrict__ r32,
                                                    VT* __restrict__ z32, VT* __restrict__ p32,
                                                    double* __restrict__ part) {
  __shared__ double sh[kSB / 64];
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  double rr = 0.0, rz = 0.0;
  if (j < N) {
    VT r[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      r[c] = (VT)(rh[3 * j + c] * s);
      r32[3 * j + c] = r[c];
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const VT z = (VT)dinv[3 * j + c] * r[c];
      z32[3 * j + c] = z;
      p32[3 * j + c] = init ? z : (VT)pscale * p32[3 * j + c];
      rr += (double)r[c] * (double)r[c];
      rz += (double)r[c] * (double)z;
    }
  }
  rr = bsum(rr, sh);
  rz = bsum(rz, sh);
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = rr;
    part[2 * blockIdx.x + 1] = rz;
  }
}

__global__ __launch_bounds__(kSB) void k_ru_scal(int64_t nb, const double* __restrict__ part, double* __restrict__ scal,
                                                 double tol2, double delta2) {
  __shared__ double sh[kSB / 64];
  double rr = 0.0, rz = 0.0;
  for (int64_t i = threadIdx.x; i < nb; i += kSB) {
    rr += part[2 * i];
    rz += part[2 * i + 1];
  }
  rr = bsum(rr, sh);
  rz = bsum(rz, sh);
  if (threadIdx.x == 0) {
    scal[SC_RHO] = rz;
    scal[SC_RR] = rr;
    scal[SC_MAXRR] = rr;
    scal[SC_TOL2] = tol2;
    scal[SC_DELTA2] = delta2;
    scal[SC_STATE] = ST_RUN;
  }
}

// AMG restart, first half: r = rh * s; p = pscale * p (not on the first
// start); partial r.r per engine vector block (the V-cycle adds r.z).
__global__ __launch_bounds__(kSB) void k_ru_restart_amg(int64_t N, int32_t nvblk, const double* __restrict__ rh,
                                                        double s, double pscale, int init, float* __restrict__ r32,
                                                        float* __restrict__ p32, double* __restrict__ part) {
  __shared__ double sh[kSB / 64];
  double rr = 0.0;
  for (int64_t j = (int64_t)blockIdx.x * kVecNodes + threadIdx.x; j < N; j += (int64_t)nvblk * kVecNodes)
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const float r = (float)(rh[3 * j + c] * s);
      r32[3 * j + c] = r;
      if (!init) p32[3 * j + c] = (float)pscale * p32[3 * j + c];
      rr += (double)r * (double)r;
    }
  rr = bsum(rr, sh);
  if (threadIdx.x == 0) part[2 * blockIdx.x] = rr;
}

// AMG restart without a V-cycle: r = rh * s, and p, z rescaled by pscale.
// z = M r carries over with the same scale only while the true residual is
// close to the rescaled recursive one; the pass also sums the drift
// ||r_true - pscale r_rec||^2 (into part[2 nvblk + block]) so the host can
// tell when z must be recomputed by a V-cycle instead.
__global__ __launch_bounds__(kSB) void k_ru_rescale_amg(int64_t N, int32_t nvblk, const double* __restrict__ rh,
                                                        double s, float pscale, float* __restrict__ r32,
                                                        float* __restrict__ z32, float* __restrict__ p32,
                                                        double* __restrict__ part) {
  __shared__ double sh[kSB / 64];
  double rr = 0.0, rz = 0.0, dd = 0.0;
  for (int64_t j = (int64_t)blockIdx.x * kVecNodes + threadIdx.x; j < N; j += (int64_t)nvblk * kVecNodes)
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const float r = (float)(rh[3 * j + c] * s);
      const float z = pscale * z32[3 * j + c];
      const double dr = (double)r - (double)pscale * (double)r32[3 * j + c];
      r32[3 * j + c] = r;
      z32[3 * j + c] = z;
      p32[3 * j + c] = pscale * p32[3 * j + c];
      rr += (double)r * (double)r;
      rz += (double)r * (double)z;
      dd += dr * dr;
    }
  rr = bsum(rr, sh);
  rz = bsum(rz, sh);
  dd = bsum(dd, sh);
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = rr;
    part[2 * blockIdx.x + 1] = rz;
    part[2 * nvblk + blockIdx.x] = dd;
  }
}

// AMG restart, second half: scalars from the partials (one block); r.z from
// the V-cycle's nrz partials where there was one.
__global__ __launch_bounds__(kSB) void k_ru_scal_amg(int32_t nvblk, const double* __restrict__ part, int64_t nrz,
                                                     const double* __restrict__ rzpart, double* __restrict__ scal,
                                                     double tol2, double delta2, double maxrun) {
  __shared__ double sh[kSB / 64];
  double rr = 0.0, rz = 0.0;
  for (int i = threadIdx.x; i < nvblk; i += kSB) {
    rr += part[2 * i];
    if (nrz == 0) rz += part[2 * i + 1];
  }
  for (int64_t i = threadIdx.x; i < nrz; i += kSB) rz += rzpart[i];
  rr = bsum(rr, sh);
  rz = bsum(rz, sh);
  if (threadIdx.x == 0) {
    scal[SC_RHO] = rz;
    scal[SC_RR] = rr;
    scal[SC_MAXRR] = rr;
    scal[SC_TOL2] = tol2;
    scal[SC_DELTA2] = delta2;
    scal[SC_LAST] = scal[SC_ITER];
    scal[SC_MAXRUN] = maxrun;
    scal[SC_STATE] = ST_RUN;
  }
}

// Jacobi preconditioner: the inverse diagonal of K on the free components,
// zero elsewhere.  (Scalar Jacobi converged faster than the inverse 3x3
// diagonal blocks on the elasticity systems measured.)
__global__ void k_dinv(int64_t N, const int64_t* __restrict__ adj_ptr, const int32_t* __restrict__ dslot,
                       const double* __restrict__ val, const uint8_t* __restrict__ fixed, float* __restrict__ dinv) {
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= N) return;
  const int64_t a0 = adj_ptr[j];
  const int64_t R = adj_ptr[j + 1] - a0;
  const int64_t s = dslot[j];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const double kdd = val[9 * a0 + d * 3 * R + 3 * s + d];   // K[(j,d),(j,d)] = panel[d][s][d]
    const bool free = fixed[3 * j + d] == 0 && kdd != 0.0;
    dinv[3 * j + d] = free ? (float)(1.0 / kdd) : 0.f;
  }
}

// FP32 operator (block32.h) from the FP64 panels: lane t of a node takes its
// blocks t, t + 32, ...
__global__ void k_to32_blocks(int64_t N, int64_t nadj, const int64_t* __restrict__ adj_ptr,
                              const double* __restrict__ val, float* __restrict__ out) {
  const int64_t j = (int64_t)blockIdx.x * blockDim.y + threadIdx.y;
  if (j >= N) return;
  const int64_t a0 = adj_ptr[j];
  const int64_t R = adj_ptr[j + 1] - a0;
  const double* P = val + 9 * a0;
  for (int64_t t = threadIdx.x; t < R; t += blockDim.x) {
    float e[9];
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int d = 0; d < 3; ++d) e[3 * c + d] = (float)P[c * 3 * R + 3 * t + d];
    const int64_t g = a0 + t;
    reinterpret_cast<f4v*>(out)[g] = f4v{e[0], e[1], e[2], e[3]};
    reinterpret_cast<f4v*>(out + 4 * nadj)[g] = f4v{e[4], e[5], e[6], e[7]};
    out[8 * nadj + g] = e[8];
  }
}

__global__ void k_fill_u(int64_t n, const uint8_t* __restrict__ fixed, const double* __restrict__ ufix,
                         const double* __restrict__ x, double* __restrict__ u) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  u[i] = fixed[i] ? (ufix ? ufix[i] : 0.0) : (x ? x[i] : 0.0);
}

inline unsigned blocks(int64_t n, int bs = kSB) { return (unsigned)std::max<int64_t>(1, (n + bs - 1) / bs); }
inline int64_t vec_blocks(int64_t N) {
  return std::max<int64_t>(1, std::min<int64_t>((N + kVecNodes - 1) / kVecNodes, kMaxVecBlocks));
}

void spmv64(hipStream_t st, const SysSpec& sp, const double* x, const uint8_t* mask, double* y) {
  const int lanes = panel_lanes(sp.N, sp.nadj);
  const unsigned g = blocks(sp.N * lanes);
  if (lanes == 32) k_spmv64<32><<<g, kSB, 0, st>>>(sp.N, sp.adj_ptr, sp.adj, sp.val64, x, mask, y);
  else if (lanes == 16) k_spmv64<16><<<g, kSB, 0, st>>>(sp.N, sp.adj_ptr, sp.adj, sp.val64, x, mask, y);
  else k_spmv64<8><<<g, kSB, 0, st>>>(sp.N, sp.adj_ptr, sp.adj, sp.val64, x, mask, y);
}

}  // namespace

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
struct SolveSys {
  SysSpec spec;
  int64_t n = 0, nadj = 0;
  void* mem = nullptr;
  size_t bytes = 0;
  double *b = nullptr, *xh = nullptr, *xt = nullptr, *rh = nullptr, *y = nullptr, *scal = nullptr, *part = nullptr;
  UpdateBook book;          // rollbacks, consecutive non-finite corrections, updates
  int64_t refreshes = 0;    // AMG updates whose z had to be recomputed (drift or r.z <= 0)
  void *x = nullptr, *r = nullptr, *z = nullptr, *p = nullptr, *q = nullptr;   // Krylov vectors (VT)
  float *dinv = nullptr, *val32 = nullptr;
  int64_t npart = 0;
  double bnorm = 0.0, scale = 1.0, relres = 0.0;
  int64_t iters = 0;
  int status = kRunning;
  int32_t sblk0 = 0, nsblk = 0, vblk0 = 0, nvblk = 0;
  AmgSys* amg = nullptr;
};

BatchSolver::BatchSolver(llfem_ctx* c, bool f64_vectors) : ctx_(c), f64v_(f64_vectors) {}

BatchSolver::~BatchSolver() {
  drop_graph();
  if (hslot_) (void)hipHostFree(hslot_);
  for (SolveSys* s : sys_) release(s);
  sys_.clear();
  if (tables_) dfree(ctx_, tables_, tables_bytes_);
  amg_batch_free(ctx_, amgb_);
}

void BatchSolver::release(SolveSys* s) {
  amg_sys_free(ctx_, s->amg);
  if (s->mem) dfree(ctx_, s->mem, s->bytes);
  delete s;
}

size_t BatchSolver::bytes_needed(int64_t N, int64_t nadj, bool f64_vectors) {
  const int64_t n = 3 * N;
  const int64_t nvblk = vec_blocks(N);
  const int64_t npart = std::max<int64_t>(3 * nvblk, blocks(n)) + 64;
  return sizeof(double) * (5 * (size_t)n + SC_N + (size_t)npart) +
         (f64_vectors ? sizeof(double) : sizeof(float)) * 5 * (size_t)n +
         sizeof(float) * ((size_t)n + 9 * (size_t)nadj) + 16 * 256;   // 14 buffers, 256-B aligned
}

// Pinned host slots for the update readbacks (grown on demand).
int BatchSolver::host_slots(size_t n) {
  if (hslot_n_ >= n) return LLFEM_OK;
  if (hslot_) (void)hipHostFree(hslot_);
  hslot_ = nullptr;
  hslot_n_ = 0;
  LLFEM_HIP(hipHostMalloc((void**)&hslot_, sizeof(double) * n, hipHostMallocDefault));
  hslot_n_ = n;
  return LLFEM_OK;
}

// Reliable updates of several systems: fold x32 into xh, recompute the FP64
// residual, test convergence, restart the FP32 recursion.  The host waits a
// fixed number of times per call, whatever the number of systems:
//   1. every system's trial solution and true residual, one readback;
//   2. the decisions (engine_policy.h); rolled-back systems get the residual
//      of their kept solution, one more readback if there are any;
//   3. stop, or restart the recursion; AMG systems that keep a rescaled z
//      read r.z and the drift back, one readback for all of them;
//   4. those whose rescaled z fails the test get a V-cycle.
// Each system's launches are the same as for an update of that system alone.
int BatchSolver::update_many(const std::vector<SolveSys*>& ss, bool init) {
  if (ss.empty()) return LLFEM_OK;
  hipStream_t st = ctx_->stream;
  const size_t m = ss.size();
  LLFEM_TRY(host_slots(4 * m));   // per system: r^2, iterations, r.z, drift^2
  double* h = hslot_;
  // r = b - K x in FP64 for x (NULL: x = 0); ||r||^2 into scal[SC_N - 1]
  auto residual = [&](SolveSys* s, const double* x) {
    const SysSpec& sp = s->spec;
    const int64_t n = s->n;
    if (x) {
      spmv64(st, sp, x, sp.fixed, s->y);
      k_ru_resid<<<blocks(n), kSB, 0, st>>>(n, s->b, s->y, sp.fixed, s->rh, s->part);
    } else {
      k_ru_resid<<<blocks(n), kSB, 0, st>>>(n, s->b, nullptr, sp.fixed, s->rh, s->part);
    }
    k_sum<<<1, kSB, 0, st>>>(blocks(n), s->part, s->scal + SC_N - 1);
  };
  // 1. trial solutions xt = xh + x / scale and their residuals
  for (size_t i = 0; i < m; ++i) {
    SolveSys* s = ss[i];
    const int64_t n = s->n;
    if (!init) {
      if (f64v_) k_ru_trial<double><<<blocks(n), kSB, 0, st>>>(n, (double*)s->x, 1.0 / s->scale, s->xh, s->xt);
      else k_ru_trial<float><<<blocks(n), kSB, 0, st>>>(n, (float*)s->x, 1.0 / s->scale, s->xh, s->xt);
      residual(s, s->xt);
    } else {
      residual(s, nullptr);
    }
    LLFEM_HIP(hipMemcpyAsync(h + 4 * i, s->scal + SC_N - 1, sizeof(double), hipMemcpyDeviceToHost, st));
    LLFEM_HIP(hipMemcpyAsync(h + 4 * i + 1, s->scal + SC_ITER, sizeof(double), hipMemcpyDeviceToHost, st));
    h[4 * i + 2] = 0.0;
    if (init && s->amg)   // the set-up has been enqueued only
      LLFEM_HIP(hipMemcpyAsync(h + 4 * i + 2, amg_status(s->amg), sizeof(double), hipMemcpyDeviceToHost, st));
  }
  LLFEM_HIP(hipStreamSynchronize(st));
  if (init) {
    // LLFEM_AMG_HOST_INVERSE=1 takes every coarsest inverse as left to the host
    // (a host-side switch for testing that path)
    const char* env = std::getenv("LLFEM_AMG_HOST_INVERSE");
    const bool host = env && env[0] == '1';
    for (size_t i = 0; i < m; ++i)
      if (ss[i]->amg && (host || h[4 * i + 2] != 0.0)) LLFEM_TRY(amg_host_inverse(ctx_, ss[i]->amg));
  }
  // 2. adoption or rollback.  LLFEM_ENGINE_FORCE_ROLLBACK=k treats the k-th
  // update's trial as not finite (a host-side switch for testing the
  // rollback path).
  std::vector<uint8_t> fresh(m, init ? 1 : 0);   // restart the Krylov recursion from scratch (p = z)
  if (!init) {
    const char* force_env = std::getenv("LLFEM_ENGINE_FORCE_ROLLBACK");
    const int64_t force_rb = force_env ? (int64_t)std::atoll(force_env) : 0;
    bool any = false;
    for (size_t i = 0; i < m; ++i) {
      SolveSys* s = ss[i];
      double r2 = h[4 * i];
      if (force_rb > 0 && s->book.updates + 1 == force_rb && s->book.rollbacks == 0) r2 = NAN;
      if (adopt_trial(r2, &s->book)) {
        std::swap(s->xh, s->xt);
      } else {
        // rollback: keep xh, restart the recursion from it
        fresh[i] = 1;
        any = true;
        residual(s, s->xh);
        LLFEM_HIP(hipMemcpyAsync(h + 4 * i, s->scal + SC_N - 1, sizeof(double), hipMemcpyDeviceToHost, st));
      }
    }
    if (any) LLFEM_HIP(hipStreamSynchronize(st));
  }
  // 3. stop or restart
  std::vector<uint8_t> check(m, 0);   // AMG systems whose rescaled z is tested
  std::vector<double> tol2(m, 0.0), s_new(m, 0.0), pscale(m, 0.0);
  bool any_check = false;
  for (size_t i = 0; i < m; ++i) {
    SolveSys* s = ss[i];
    const SysSpec& sp = s->spec;
    const int64_t n = s->n;
    const double rn = std::sqrt(h[4 * i]);
    s->iters = (int64_t)h[4 * i + 1];
    if (init) s->bnorm = rn;
    else ++s->book.updates;
    const int status = update_status(rn, s->bnorm, sp.reltol, s->iters, sp.maxiter, s->book);
    if (status != kRunning) {
      s->status = status;
      if (status != kConverged) s->relres = s->bnorm > 0 && std::isfinite(rn) ? rn / s->bnorm : 0.0;
      k_set_state<<<1, 1, 0, st>>>(s->scal, (double)ST_IDLE);
      continue;
    }
    s_new[i] = 1.0 / rn;
    pscale[i] = s_new[i] / s->scale;
    s->scale = s_new[i];
    const double tol = sp.reltol * s->bnorm * s_new[i];
    tol2[i] = tol * tol;
    if (s->amg) {
      const int32_t nvblk = (int32_t)vec_blocks(sp.N);
      double* vpart = s->part;
      if (fresh[i]) {   // z = M r by a V-cycle of this system alone, p = z
        k_ru_restart_amg<<<(unsigned)nvblk, kSB, 0, st>>>(sp.N, nvblk, s->rh, s_new[i], pscale[i], 1, (float*)s->r,
                                                          (float*)s->p, vpart);
        LLFEM_TRY(amg_apply_solo(ctx_, s->amg));
        LLFEM_HIP(hipMemcpyAsync(s->p, s->z, sizeof(float) * n, hipMemcpyDeviceToDevice, st));
      } else {
        k_ru_rescale_amg<<<(unsigned)nvblk, kSB, 0, st>>>(sp.N, nvblk, s->rh, s_new[i], (float)pscale[i],
                                                          (float*)s->r, (float*)s->z, (float*)s->p, vpart);
      }
      k_ru_scal_amg<<<1, kSB, 0, st>>>(nvblk, vpart, fresh[i] ? row_groups(sp.N) : 0, s->y, s->scal, tol2[i],
                                       kDeltaAmg * kDeltaAmg, (double)kMaxRunAmg);
      if (!fresh[i]) {
        // the rescaled z is consistent only if r.z > 0 and the true residual
        // is close to the rescaled recursive one (amg_keep_rescaled)
        k_sum<<<1, kSB, 0, st>>>(nvblk, vpart + 2 * nvblk, s->scal + SC_N - 1);
        LLFEM_HIP(hipMemcpyAsync(h + 4 * i + 2, s->scal + SC_RHO, sizeof(double), hipMemcpyDeviceToHost, st));
        LLFEM_HIP(hipMemcpyAsync(h + 4 * i + 3, s->scal + SC_N - 1, sizeof(double), hipMemcpyDeviceToHost, st));
        check[i] = 1;
        any_check = true;
      }
      continue;
    }
    const int64_t nb = blocks(sp.N);
    if (f64v_)
      k_ru_restart<double><<<(unsigned)nb, kSB, 0, st>>>(sp.N, s->rh, s_new[i], pscale[i], fresh[i] ? 1 : 0, s->dinv,
                                                         (double*)s->r, (double*)s->z, (double*)s->p, s->part);
    else
      k_ru_restart<float><<<(unsigned)nb, kSB, 0, st>>>(sp.N, s->rh, s_new[i], pscale[i], fresh[i] ? 1 : 0, s->dinv,
                                                        (float*)s->r, (float*)s->z, (float*)s->p, s->part);
    k_ru_scal<<<1, kSB, 0, st>>>(nb, s->part, s->scal, tol2[i], kDelta * kDelta);
  }
  // 4. AMG systems whose rescaled z failed: z = M r, restart the direction from it
  if (any_check) {
    LLFEM_HIP(hipStreamSynchronize(st));
    for (size_t i = 0; i < m; ++i) {
      if (!check[i] || amg_keep_rescaled(h[4 * i + 2], h[4 * i + 3], kDriftAmg)) continue;
      SolveSys* s = ss[i];
      const SysSpec& sp = s->spec;
      const int32_t nvblk = (int32_t)vec_blocks(sp.N);
      double* vpart = s->part;
      ++s->refreshes;
      k_ru_restart_amg<<<(unsigned)nvblk, kSB, 0, st>>>(sp.N, nvblk, s->rh, s_new[i], pscale[i], 1, (float*)s->r,
                                                        (float*)s->p, vpart);
      LLFEM_TRY(amg_apply_solo(ctx_, s->amg));
      LLFEM_HIP(hipMemcpyAsync(s->p, s->z, sizeof(float) * s->n, hipMemcpyDeviceToDevice, st));
      k_ru_scal_amg<<<1, kSB, 0, st>>>(nvblk, vpart, row_groups(sp.N), s->y, s->scal, tol2[i], kDeltaAmg * kDeltaAmg,
                                       (double)kMaxRunAmg);
    }
  }
  LLFEM_HIP(hipGetLastError());
  return LLFEM_OK;
}

int BatchSolver::add(const SysSpec& spec, SolveSys** out) {
  hipStream_t st = ctx_->stream;
  SolveSys* s = new SolveSys();
  s->spec = spec;
  s->n = 3 * spec.N;
  s->nadj = spec.nadj;
  s->bytes = bytes_needed(spec.N, spec.nadj, f64v_);
  int rc = dmalloc(ctx_, &s->mem, s->bytes);
  if (rc != LLFEM_OK) {
    delete s;
    return rc;
  }
  const int64_t n = s->n, N = spec.N;
  const int64_t nvblk = vec_blocks(N);
  s->npart = std::max<int64_t>(3 * nvblk, blocks(n)) + 64;   // vector and drift partials
  char* m = static_cast<char*>(s->mem);
  auto take = [&](size_t bytes) -> char* {
    char* p = m;
    m += (bytes + 255) / 256 * 256;
    return p;
  };
  s->b = (double*)take(sizeof(double) * n);
  s->xh = (double*)take(sizeof(double) * n);
  s->xt = (double*)take(sizeof(double) * n);
  s->rh = (double*)take(sizeof(double) * n);
  s->y = (double*)take(sizeof(double) * n);
  s->scal = (double*)take(sizeof(double) * SC_N);
  s->part = (double*)take(sizeof(double) * s->npart);
  const size_t vsz = f64v_ ? sizeof(double) : sizeof(float);
  s->x = take(vsz * n);
  s->r = take(vsz * n);
  s->z = take(vsz * n);
  s->p = take(vsz * n);
  s->q = take(vsz * n);
  s->dinv = (float*)take(sizeof(float) * n);
  s->val32 = (float*)take(sizeof(float) * 9 * spec.nadj);
  if ((size_t)(m - static_cast<char*>(s->mem)) > s->bytes) {
    release(s);
    return fail(LLFEM_EINVAL, "engine: workspace layout overflow");
  }
  // b = mask(f - K u_fixed); x = 0; FP32 operator and inverse diagonal
  k_fill_u<<<blocks(n), kSB, 0, st>>>(n, spec.fixed, spec.ufix, nullptr, s->y);
  spmv64(st, spec, s->y, nullptr, s->rh);
  k_ru_resid<<<blocks(n), kSB, 0, st>>>(n, spec.f, s->rh, spec.fixed, s->b, s->part);
  k_to32_blocks<<<blocks(N, 8), dim3(32, 8), 0, st>>>(N, spec.nadj, spec.adj_ptr, spec.val64, s->val32);
  k_dinv<<<blocks(N), kSB, 0, st>>>(N, spec.adj_ptr, spec.dslot, spec.val64, spec.fixed, s->dinv);
  LLFEM_HIP(hipMemsetAsync(s->xh, 0, sizeof(double) * n, st));
  LLFEM_HIP(hipMemsetAsync(s->x, 0, vsz * n, st));
  LLFEM_HIP(hipMemsetAsync(s->scal, 0, sizeof(double) * SC_N, st));
  s->scale = 1.0;
  if (spec.amg) {
    if (f64v_) {
      release(s);
      return fail(LLFEM_EUNSUP, "engine: the AMG preconditioner runs with FP32 Krylov vectors");
    }
    rc = amg_sys_create(ctx_, spec.amg, s->val32, (float*)s->r, (float*)s->z, (float*)s->q, s->y, &s->amg);
    if (rc != LLFEM_OK) {
      release(s);
      return rc;
    }
  }
  rc = update_many({s}, true);
  if (rc != LLFEM_OK) {
    release(s);
    return rc;
  }
  sys_.push_back(s);
  dirty_ = true;
  *out = s;
  return LLFEM_OK;
}

int BatchSolver::rebuild_tables() {
  std::vector<SysDev> dev;
  std::vector<int32_t> sb, vb;
  live_.clear();
  fold_ = false;
  for (SolveSys* s : sys_) {
    if (s->status != 0) continue;
    const SysSpec& sp = s->spec;
    SysDev d{};
    d.N = sp.N;
    d.adj_ptr = sp.adj_ptr;
    d.adj = sp.adj;
    d.nadj = sp.nadj;
    d.val = s->val32;
    d.fixed = sp.fixed;
    d.dinv = s->dinv;
    d.x = s->x; d.r = s->r; d.z = s->z; d.p = s->p; d.q = s->q;
    d.scal = s->scal;
    d.spart = s->y;
    d.part = s->part;
    d.nsblk = (int32_t)row_groups(sp.N);
    fold_ = fold_ || d.nsblk > kFoldMax;
    d.nvblk = (int32_t)vec_blocks(sp.N);
    d.amg = s->amg ? 1 : 0;
    if (s->amg) (void)amg_head(s->amg, &d.mgy, &d.mgd, &d.mgdinv, &d.mgt);
    d.sblk0 = (int32_t)sb.size();
    d.vblk0 = (int32_t)vb.size();
    const int32_t id = (int32_t)dev.size();
    sb.insert(sb.end(), (size_t)d.nsblk, id);
    vb.insert(vb.end(), (size_t)d.nvblk, id);
    dev.push_back(d);
    live_.push_back(s);
  }
  {
    std::vector<AmgSys*> as;
    std::vector<const double*> st_words;
    for (SolveSys* s : live_)
      if (s->amg) {
        as.push_back(s->amg);
        st_words.push_back(s->scal + SC_STATE);
      }
    LLFEM_TRY(amg_batch_build(ctx_, as, st_words, &amgb_));
  }
  nsys_ = (int)dev.size();
  nsb_ = (int64_t)sb.size();
  nvb_ = (int64_t)vb.size();
  const size_t need = sizeof(SysDev) * dev.size() + sizeof(int32_t) * (sb.size() + vb.size()) +
                      sizeof(double) * 2 * dev.size() + 1024;
  if (tables_bytes_ < need) {
    if (tables_) dfree(ctx_, tables_, tables_bytes_);
    tables_ = nullptr;
    tables_bytes_ = 0;
    LLFEM_TRY(dmalloc(ctx_, &tables_, need * 2));
    tables_bytes_ = need * 2;
  }
  char* m = static_cast<char*>(tables_);
  d_sys_ = reinterpret_cast<SysDev*>(m);
  m += (sizeof(SysDev) * dev.size() + 255) / 256 * 256;
  d_sb_ = reinterpret_cast<int32_t*>(m);
  m += (sizeof(int32_t) * sb.size() + 255) / 256 * 256;
  d_vb_ = reinterpret_cast<int32_t*>(m);
  m += (sizeof(int32_t) * vb.size() + 255) / 256 * 256;
  d_states_ = reinterpret_cast<double*>(m);
  hipStream_t st = ctx_->stream;
  if (!dev.empty()) {
    LLFEM_HIP(hipMemcpyAsync(d_sys_, dev.data(), sizeof(SysDev) * dev.size(), hipMemcpyHostToDevice, st));
    LLFEM_HIP(hipMemcpyAsync(d_sb_, sb.data(), sizeof(int32_t) * sb.size(), hipMemcpyHostToDevice, st));
    LLFEM_HIP(hipMemcpyAsync(d_vb_, vb.data(), sizeof(int32_t) * vb.size(), hipMemcpyHostToDevice, st));
    LLFEM_HIP(hipStreamSynchronize(st));   // host vectors go out of scope
  }
  dirty_ = false;
  return LLFEM_OK;
}

void BatchSolver::drop_graph() {
  if (chunk_exec_) (void)hipGraphExecDestroy(chunk_exec_);
  chunk_exec_ = nullptr;
  chunk_iters_ = 0;
}

// Whether chunks run as a captured graph: on unless LLFEM_ENGINE_GRAPH=0.
static bool engine_graph_enabled() {
  const char* e = std::getenv("LLFEM_ENGINE_GRAPH");
  return !(e && e[0] == '0');
}

int BatchSolver::run(int iters, std::vector<SolveSys*>* finished) {
  hipStream_t st = ctx_->stream;
  if (dirty_) {
    drop_graph();
    LLFEM_TRY(rebuild_tables());
  }
  if (nsys_ == 0) return LLFEM_OK;
  const SysDev* sys = static_cast<const SysDev*>(d_sys_);
  // The chunk's launches (SpMV, updates, V-cycles) depend only on the live
  // set's tables; the per-system state they read and write lives in device
  // memory.  A live set's first chunk is launched as it stands and recorded
  // while the device works on it; the others replay the record.  (Recorded
  // first, with the device idle meanwhile, eight systems on a server with six
  // changes of the set took 41.1 instead of 39.5 ms.)
  const bool graph = engine_graph_enabled();
  const bool replay = graph && chunk_exec_ && chunk_iters_ == iters;
  LLFEM_TRY(host_slots(4 * (size_t)nsys_));   // as much as the updates below need
  if (replay) {
    LLFEM_HIP(hipGraphLaunch(chunk_exec_, st));
  } else {
    drop_graph();
    LLFEM_TRY(launch_chunk(iters));
  }
  k_bs_states<<<blocks(nsys_), kSB, 0, st>>>(sys, nsys_, d_states_);
  LLFEM_HIP(hipMemcpyAsync(hslot_, d_states_, sizeof(double) * 2 * (size_t)nsys_, hipMemcpyDeviceToHost, st));
  if (graph && !replay) {
    hipGraph_t g = nullptr;
    LLFEM_HIP(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
    const int rc = launch_chunk(iters);
    const hipError_t ec = hipStreamEndCapture(st, &g);
    LLFEM_TRY(rc);
    if (ec != hipSuccess) return fail(LLFEM_EHIP, std::string("engine graph capture: ") + hipGetErrorString(ec));
    const hipError_t ei = hipGraphInstantiate(&chunk_exec_, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    if (ei != hipSuccess) {
      chunk_exec_ = nullptr;
      return fail(LLFEM_EHIP, std::string("engine graph instantiate: ") + hipGetErrorString(ei));
    }
    chunk_iters_ = iters;
  }
  LLFEM_HIP(hipStreamSynchronize(st));
  LLFEM_HIP(hipGetLastError());
  const std::vector<double> h(hslot_, hslot_ + 2 * (size_t)nsys_);
  std::vector<SolveSys*> paused;
  for (int i = 0; i < nsys_; ++i) {
    SolveSys* s = live_[i];
    s->iters = (int64_t)h[2 * i + 1];
    const int state = (int)h[2 * i];
    if (state == ST_PENDING || state == ST_PAUSED) paused.push_back(s);
  }
  LLFEM_TRY(update_many(paused, false));
  for (SolveSys* s : paused)
    if (s->status != kRunning) {
      dirty_ = true;
      if (finished) finished->push_back(s);
    }
  return LLFEM_OK;
}

int BatchSolver::launch_chunk(int iters) {
  hipStream_t st = ctx_->stream;
  const SysDev* sys = static_cast<const SysDev*>(d_sys_);
  const unsigned nf = (unsigned)(nsys_ * kFoldBlocks);
  for (int k = 0; k < iters; ++k) {
    if (f64v_) k_bs_spmv<double><<<(unsigned)nsb_, kRowThreads, 0, st>>>(sys, d_sb_, nsys_);
    else k_bs_spmv<float><<<(unsigned)nsb_, kRowThreads, 0, st>>>(sys, d_sb_, nsys_);
    if (fold_) k_bs_fold<<<nf, kSB, 0, st>>>(sys);
    if (f64v_) {
      k_bs_update<double><<<(unsigned)nvb_, kSB, 0, st>>>(sys, d_vb_, nsys_);
    } else {
      k_bs_update<float><<<(unsigned)nvb_, kSB, 0, st>>>(sys, d_vb_, nsys_);
      const bool amg = amg_batch_any(amgb_);
      LLFEM_TRY(amg_batch_apply(ctx_, amgb_));
      if (fold_ && amg) k_bs_fold<<<nf, kSB, 0, st>>>(sys);
    }
    if (f64v_) k_bs_pupd<double><<<(unsigned)nvb_, kSB, 0, st>>>(sys, d_vb_, nsys_);
    else k_bs_pupd<float><<<(unsigned)nvb_, kSB, 0, st>>>(sys, d_vb_, nsys_);
  }
  return LLFEM_OK;
}

// u = u_fixed on constrained DoFs, xh elsewhere; true relative residual
// ||(K u - f)_free|| / ||f_free|| (test/test_dsl.jl:106).
int BatchSolver::finish(SolveSys* s, double* u) {
  hipStream_t st = ctx_->stream;
  const SysSpec& sp = s->spec;
  const int64_t n = s->n;
  k_fill_u<<<blocks(n), kSB, 0, st>>>(n, sp.fixed, sp.ufix, s->xh, u);
  spmv64(st, sp, u, nullptr, s->y);
  k_ru_resid<<<blocks(n), kSB, 0, st>>>(n, sp.f, s->y, sp.fixed, nullptr, s->part);
  k_sum<<<1, kSB, 0, st>>>(blocks(n), s->part, s->scal + SC_N - 1);
  k_ru_resid<<<blocks(n), kSB, 0, st>>>(n, sp.f, nullptr, sp.fixed, nullptr, s->part);
  k_sum<<<1, kSB, 0, st>>>(blocks(n), s->part, s->scal + SC_N - 2);
  double h[2];
  LLFEM_HIP(hipMemcpyAsync(h, s->scal + SC_N - 2, sizeof(h), hipMemcpyDeviceToHost, st));
  LLFEM_HIP(hipStreamSynchronize(st));
  LLFEM_HIP(hipGetLastError());
  s->relres = h[0] > 0 ? std::sqrt(h[1] / h[0]) : std::sqrt(h[1]);
  return LLFEM_OK;
}

void BatchSolver::remove(SolveSys* s) {
  auto it = std::find(sys_.begin(), sys_.end(), s);
  if (it == sys_.end()) return;
  sys_.erase(it);
  (void)hipStreamSynchronize(ctx_->stream);
  release(s);
  dirty_ = true;
}

bool BatchSolver::any_running() const {
  for (SolveSys* s : sys_)
    if (s->status == 0) return true;
  return false;
}

int64_t sys_iterations(const SolveSys* s) { return s->iters; }
int64_t sys_updates(const SolveSys* s) { return s->book.updates; }
int64_t sys_rollbacks(const SolveSys* s) { return s->book.rollbacks; }
int64_t sys_refreshes(const SolveSys* s) { return s->refreshes; }
int sys_status(const SolveSys* s) { return s->status; }
double sys_relres(const SolveSys* s) { return s->relres; }

}  // namespace llfem
