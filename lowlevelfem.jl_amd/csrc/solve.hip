// Dirichlet-eliminated Jacobi-PCG on the device, FP64 or FP32-inner with
// FP64 iterative refinement.
//
// Reference: solveDisplacement(K, f; support, iterative=true, reltol, maxiter,
// preconditioner) (src/linear.jl:3711-3743): u_fixed on the constrained DoFs,
// rhs = f_free - K[free,fixed] u_fixed, u_free = cg(K_ff, rhs; Pl, reltol,
// maxiter) with IterativeSolvers.cg semantics (x0 = 0, converged when
// ||r|| <= reltol ||r0||).  K_ff is applied as the masked operator
// P_f K P_f (no submatrix is extracted); fixed entries stay 0 in every
// Krylov vector.
//
// SpMV runs on the node-panel layout of the assembled K (block CSR of K^T,
// equal to K by symmetry): one int32 column index per 3x3 block, so the
// index stream is 1/9 of scalar CSR.  Dot products reduce per block and then
// in one fixed-order pass, so every run gives bit-identical iterates.
// Scalars (alpha, beta, rho, ||r||, convergence) live on the device; the host
// only polls the convergence flag every few iterations.
#include <chrono>
#include <cmath>
#include <cstring>
#include <mutex>

#include "common.h"

namespace llfem {
namespace {

constexpr int kBS = 256;
constexpr int kWaves = kBS / 64;
constexpr int kG = 8;   // lanes per row the workspace's partial count is sized for (solve_ws_bytes)
// Partials a kernel sums by itself in every block: up to this many cost each
// block about a microsecond out of L2, less than a reduction launch of its
// own.  More of them (large systems) go through k_fold first.
constexpr int64_t kFoldMax = 2048;
constexpr unsigned kFoldBlocks = 64;
constexpr int64_t kMaxPasses = 8;

// S_RHO0 / S_RHO1: r.z of even / odd iterations (the p-update reads one and
// writes the other, so no block sees the new value in place of the old).
enum { S_RHO0 = 0, S_RHO1, S_RR, S_TOL2, S_DONE, S_ITER, S_NS = 8 };

// Sum over the block in a fixed order: a butterfly per wavefront, then the
// wavefronts' sums in order.  One barrier before the result, one after it
// (sh may be reused at once).
__device__ __forceinline__ double block_sum(double v, double* sh) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  double r = sh[0];
#pragma unroll
  for (int w = 1; w < kWaves; ++w) r += sh[w];
  __syncthreads();
  return r;
}

__device__ __forceinline__ double2 block_sum2(double a, double b, double* sh) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    a += __shfl_xor(a, o, 64);
    b += __shfl_xor(b, o, 64);
  }
  if ((threadIdx.x & 63) == 0) {
    sh[threadIdx.x >> 6] = a;
    sh[kWaves + (threadIdx.x >> 6)] = b;
  }
  __syncthreads();
  double ra = sh[0], rb = sh[kWaves];
#pragma unroll
  for (int w = 1; w < kWaves; ++w) {
    ra += sh[w];
    rb += sh[kWaves + w];
  }
  __syncthreads();
  return make_double2(ra, rb);
}

// This thread's share of n partials, or of n pairs of them; the same order in
// every block.  Eight loads under way at a time: one by one, 2,048 partials
// are a chain of eight loads, 0.6 us each on an idle chip.  Loads only, so a
// kernel can issue them before it knows whether the solve is done.
__device__ __forceinline__ double own_partials(int64_t n, const double* __restrict__ part) {
  double s = 0.0;
  for (int64_t i0 = threadIdx.x; i0 < n; i0 += 8 * kBS) {
    double a[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) a[k] = i0 + k * kBS < n ? part[i0 + k * kBS] : 0.0;
#pragma unroll
    for (int k = 0; k < 8; ++k) s += a[k];
  }
  return s;
}
__device__ __forceinline__ double2 own_pairs(int64_t n, const double* __restrict__ part) {
  const double2* const q = reinterpret_cast<const double2*>(part);
  double2 s = make_double2(0.0, 0.0);
  for (int64_t i0 = threadIdx.x; i0 < n; i0 += 8 * kBS) {
    double2 a[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) a[k] = i0 + k * kBS < n ? q[i0 + k * kBS] : make_double2(0.0, 0.0);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      s.x += a[k].x;
      s.y += a[k].y;
    }
  }
  return s;
}
__device__ __forceinline__ double sum_partials(int64_t n, const double* __restrict__ part, double* sh) {
  return block_sum(own_partials(n, part), sh);
}
__device__ __forceinline__ double2 sum_pairs(int64_t n, const double* __restrict__ part, double* sh) {
  const double2 s = own_pairs(n, part);
  return block_sum2(s.x, s.y, sh);
}

// Blocks are dealt round-robin to the 8 XCDs; neighbouring rows share most of
// the x entries they read, so give each XCD a contiguous run of blocks (the
// last gridDim % 8 blocks keep their place).  FP64 panels of 46,575 nodes:
// 23.1 -> 20.8 us; at 2.1 M nodes the same.
__device__ __forceinline__ int64_t xcd_block() {
  const unsigned nb = gridDim.x & ~7u, b = blockIdx.x;
  return b < nb ? (int64_t)(b & 7u) * (nb >> 3) + (b >> 3) : (int64_t)b;
}

// What an SpMV multiplies: a vector as it stands, ...
template <typename VT>
struct Plain {
  using Raw = VT;   // what is loaded of an entry, before begin()
  const VT* __restrict__ x;
  __device__ __forceinline__ void fetch() {}
  __device__ __forceinline__ bool begin(double*) { return true; }
  __device__ __forceinline__ Raw raw(int64_t i) const { return x[i]; }
  __device__ __forceinline__ VT value(Raw v) const { return v; }
  __device__ __forceinline__ void keep(int64_t, VT) const {}
};

// ... or the CG direction p = z + beta p_old, formed while it is gathered: the
// launch that would write it first, and its pass over z and p, are not needed.
// Every block sums the previous update's partials (r.r, r.z) itself; block 0
// keeps the scalars, tests convergence and tells the host.  Each row's owner
// writes its part of p to a second array (neighbours still read p_old).
// Block 0 may set S_DONE while waves of later blocks read it, so such a block
// can lose some of its waves, and what the others then sum and write (p, y and
// the product's partials) means nothing.  No kernel of this solve reads any of
// it: all that follow see S_DONE set, and x is not written here.
template <typename VT>
struct Direction {
  const VT* __restrict__ z;
  const VT* __restrict__ pold;
  VT* __restrict__ pnew;
  double* scal;
  const double* part;   // np pairs (r.r, r.z) of the update before
  int64_t np, it, maxiter;
  volatile double* done_host;
  VT beta;
  double2 own;
  double rho;
  struct Raw {
    VT z, p;
  };
  __device__ __forceinline__ void fetch() {   // the loads of begin()
    if (it == 0) return;
    own = own_pairs(np, part);
    rho = scal[S_RHO0 + (int)((it - 1) & 1)];
  }
  __device__ __forceinline__ bool begin(double* sh) {
    beta = 0;
    if (it == 0) return true;   // p = z, rho from k_init_scal
    const double2 s = block_sum2(own.x, own.y, sh);
    beta = (VT)(s.y / rho);
    const bool done = s.x <= scal[S_TOL2] || it >= maxiter;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      scal[S_RHO0 + (int)(it & 1)] = s.y;
      scal[S_RR] = s.x;
      scal[S_ITER] = (double)it;
      if (done) {
        scal[S_DONE] = 1.0;
        *done_host = 1.0;
      }
    }
    return !done;
  }
  __device__ __forceinline__ Raw raw(int64_t i) const { return {z[i], it == 0 ? (VT)0 : pold[i]}; }
  __device__ __forceinline__ VT value(Raw v) const { return v.z + beta * v.p; }
  __device__ __forceinline__ void keep(int64_t i, VT v) const { pnew[i] = v; }
};

// y = mask(K x); optional partial of dot(x, y).  Node row j uses G lanes, one
// 3x3 block per lane and step.  Bound: HBM for large K, a chain of dependent
// loads (row pointer -> column -> x) for small ones; with G covering a whole
// row the chain is walked once.  FP64, tet10 panels (28 blocks a row): G = 8
// 1013 us, 32 912 us at 2.1 M nodes (4.5 -> 5.0 TB/s of 76 bytes a block);
// 23.0 -> 17.5 us at 46,575 nodes.  A block walks `passes` row groups, so
// that the systems of up to a few 100,000 DoFs leave no more partials than
// the next kernel's blocks sum by themselves.
template <typename MT, typename VT, int G, typename X>
__global__ __launch_bounds__(kBS) void k_spmv(int64_t N, int passes, const int64_t* __restrict__ adj_ptr,
                                             const int32_t* __restrict__ adj, const MT* __restrict__ val, X xs,
                                             const uint8_t* __restrict__ fixed, VT* __restrict__ y,
                                             double* __restrict__ part, const double* __restrict__ scal) {
  __shared__ double sh[2 * kWaves];
  const int64_t lb = xcd_block();
  const int l = (int)(threadIdx.x % G);
  int64_t j = lb * passes * (kBS / G) + threadIdx.x / G;
  int64_t p0 = 0;
  int R = 0;
  auto span = [&]() {
    const int64_t i = j < N ? j : N - 1;
    p0 = adj_ptr[i];
    R = j < N ? (int)(adj_ptr[i + 1] - p0) : 0;
  };
  const double done = scal ? scal[S_DONE] : 0.0;
  xs.fetch();
  span();
  if (done != 0.0) return;
  if (!xs.begin(sh)) return;
  double d = 0.0;
  for (int ps = 0; ps < passes; ++ps, j += kBS / G, span()) {
    VT a0 = 0, a1 = 0, a2 = 0;
    {
      const MT* P = val + 9 * p0;
      for (int s = l; s < R; s += G) {
        const int64_t i = adj[p0 + s];
        const auto r0 = xs.raw(3 * i), r1 = xs.raw(3 * i + 1), r2 = xs.raw(3 * i + 2);
        const VT x0 = xs.value(r0), x1 = xs.value(r1), x2 = xs.value(r2);
        a0 += (VT)P[3 * s] * x0 + (VT)P[3 * s + 1] * x1 + (VT)P[3 * s + 2] * x2;
        a1 += (VT)P[3 * R + 3 * s] * x0 + (VT)P[3 * R + 3 * s + 1] * x1 + (VT)P[3 * R + 3 * s + 2] * x2;
        a2 += (VT)P[6 * R + 3 * s] * x0 + (VT)P[6 * R + 3 * s + 1] * x1 + (VT)P[6 * R + 3 * s + 2] * x2;
      }
    }
#pragma unroll
    for (int o = G / 2; o > 0; o >>= 1) {
      a0 += __shfl_xor(a0, o, G);
      a1 += __shfl_xor(a1, o, G);
      a2 += __shfl_xor(a2, o, G);
    }
    if (j < N && l < 3) {   // lane c writes component c
      const VT r = l == 0 ? a0 : l == 1 ? a1 : a2;
      const int64_t i = 3 * j + l;
      const VT v = (fixed && fixed[i]) ? (VT)0 : r;
      const VT xv = xs.value(xs.raw(i));
      y[i] = v;
      xs.keep(i, xv);
      d += (double)xv * (double)v;
    }
  }
  if (part) {
    const double s = block_sum(d, sh);
    if (threadIdx.x == 0) part[lb] = s;
  }
}

// Fixed-order final reduction of `n` partial rows of width w into out[0..w).
__global__ void k_reduce(int64_t n, int w, const double* __restrict__ part, double* __restrict__ out) {
  __shared__ double sh[kWaves];
  for (int c = 0; c < w; ++c) {
    double s = 0.0;
    for (int64_t i = threadIdx.x; i < n; i += blockDim.x) s += part[i * w + c];
    s = block_sum(s, sh);
    if (threadIdx.x == 0) out[c] = s;
  }
}

// n partials -> gridDim.x partials, each the sum of one contiguous run.
__global__ __launch_bounds__(kBS) void k_fold(int64_t n, const double* __restrict__ part, double* __restrict__ out,
                                             const double* __restrict__ scal) {
  __shared__ double sh[kWaves];
  if (scal[S_DONE] != 0.0) return;
  const int64_t per = (n + gridDim.x - 1) / gridDim.x, i0 = blockIdx.x * per, i1 = min(n, i0 + per);
  double s = 0.0;
  for (int64_t i = i0 + threadIdx.x; i < i1; i += kBS) s += part[i];
  s = block_sum(s, sh);
  if (threadIdx.x == 0) out[blockIdx.x] = s;
}

// alpha = rho / p.q, then x += alpha p; r -= alpha q; z = dinv r; partials
// (r.r, r.z).  Every block sums the np partials of p.q itself (same order,
// same alpha), which takes the reduction and scalar launches between the
// SpMV and this kernel out of the iteration.
template <typename VT>
__global__ __launch_bounds__(kBS) void k_update(int64_t n, const double* __restrict__ scal, int par, int64_t np,
                                               const double* __restrict__ pq, VT* __restrict__ x,
                                               VT* __restrict__ r, const VT* __restrict__ p,
                                               const VT* __restrict__ q, const VT* __restrict__ dinv,
                                               VT* __restrict__ z, double* __restrict__ part) {
  __shared__ double sh[2 * kWaves];
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  VT xi = 0, pi = 0, ri = 0, qi = 0, di = 0;   // of the entry under way; the first one's load beside the partials
  auto load = [&]() {
    if (i < n) {
      xi = x[i];
      pi = p[i];
      ri = r[i];
      qi = q[i];
      di = dinv[i];
    }
  };
  load();
  const double done = scal[S_DONE], rho = scal[S_RHO0 + par], own = own_partials(np, pq);
  if (done != 0.0) return;
  const VT alpha = (VT)(rho / block_sum(own, sh));
  double rr = 0.0, rz = 0.0;
  for (; i < n; i += (int64_t)gridDim.x * blockDim.x, load()) {
    x[i] = xi + alpha * pi;
    ri -= alpha * qi;
    r[i] = ri;
    const VT zi = di * ri;
    z[i] = zi;
    rr += (double)ri * (double)ri;
    rz += (double)ri * (double)zi;
  }
  const double2 s = block_sum2(rr, rz, sh);
  if (threadIdx.x == 0) reinterpret_cast<double2*>(part)[blockIdx.x] = s;
}

// beta = rz / rho, p = z + beta p; block 0 keeps the scalars, tests
// convergence on ||r|| and tells the host (done_host: pinned memory).  A block
// whose waves, some or all, read S_DONE after block 0 set it leaves its part of p
// as it was or writes anything there: no kernel of this solve reads p any more
// then.
template <typename VT>
__global__ __launch_bounds__(kBS) void k_pupd(int64_t n, double* __restrict__ scal, int64_t it, int64_t np,
                                             const double* __restrict__ part, int64_t maxiter,
                                             const VT* __restrict__ z, VT* __restrict__ p,
                                             volatile double* done_host) {
  __shared__ double sh[2 * kWaves];
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  VT zi = 0, pi = 0;   // of the entry under way; the first one's load beside the partials
  auto load = [&]() {
    if (i < n) {
      zi = z[i];
      pi = p[i];
    }
  };
  load();
  const double done = scal[S_DONE], rho = scal[S_RHO0 + (int)(it & 1)];
  const double2 own = own_pairs(np, part);
  if (done != 0.0) return;
  const double2 s = block_sum2(own.x, own.y, sh);   // r.r, r.z
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    scal[S_RHO0 + (int)(~it & 1)] = s.y;
    scal[S_RR] = s.x;
    scal[S_ITER] = (double)(it + 1);
    if (s.x <= scal[S_TOL2] || it + 1 >= maxiter) {
      scal[S_DONE] = 1.0;
      *done_host = 1.0;
    }
  }
  const VT beta = (VT)(s.y / rho);
  for (; i < n; i += (int64_t)gridDim.x * blockDim.x, load()) p[i] = zi + beta * pi;
}

// init: x = 0; r = b; z = dinv r; p = z; partials (r.r, r.z)
template <typename VT>
__global__ __launch_bounds__(kBS) void k_init(int64_t n, VT* __restrict__ x, const VT* __restrict__ b,
                                             VT* __restrict__ r, const VT* __restrict__ dinv, VT* __restrict__ z,
                                             VT* __restrict__ p, double* __restrict__ part) {
  __shared__ double sh[2 * kWaves];
  double rr = 0.0, rz = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    x[i] = 0;
    const VT ri = b[i];
    r[i] = ri;
    const VT zi = dinv[i] * ri;
    z[i] = zi;
    p[i] = zi;
    rr += (double)ri * (double)ri;
    rz += (double)ri * (double)zi;
  }
  const double2 s = block_sum2(rr, rz, sh);
  if (threadIdx.x == 0) reinterpret_cast<double2*>(part)[blockIdx.x] = s;
}

// scalars of the first iteration from the np partials of k_init (one block)
__global__ __launch_bounds__(kBS) void k_init_scal(int64_t np, const double* __restrict__ part, double* scal,
                                                   double rtol, volatile double* done_host) {
  __shared__ double sh[2 * kWaves];
  const double2 s = sum_pairs(np, part, sh);
  if (threadIdx.x != 0) return;
  const double rr = s.x;
  scal[S_RR] = rr;
  scal[S_RHO0] = s.y;
  scal[S_TOL2] = rtol * rtol * rr;
  scal[S_ITER] = 0.0;
  const double done = (rr <= scal[S_TOL2] || rr == 0.0) ? 1.0 : 0.0;
  scal[S_DONE] = done;
  *done_host = done;
}

// diag / Jacobi inverse from the panels; 0 on fixed DoFs
template <typename VT>
__global__ void k_dinv(int64_t N, const int64_t* __restrict__ adj_ptr, const int32_t* __restrict__ dslot,
                       const double* __restrict__ val, const uint8_t* __restrict__ fixed,
                       VT* __restrict__ dinv) {
  int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= N) return;
  const int64_t p0 = adj_ptr[j];
  const int R = (int)(adj_ptr[j + 1] - p0);
  const int s = dslot[j];
  for (int c = 0; c < 3; ++c) {
    const double dv = s >= 0 ? val[9 * p0 + (int64_t)c * 3 * R + 3 * s + c] : 0.0;
    dinv[3 * j + c] = (fixed[3 * j + c] || dv == 0.0) ? (VT)0 : (VT)(1.0 / dv);
  }
}

// r = mask(f - y) (y NULL: mask(f); r NULL: only the norm); partial of r.r
__global__ void k_resid(int64_t n, const double* __restrict__ f, const double* __restrict__ y,
                        const uint8_t* __restrict__ fixed, double* __restrict__ r,
                        double* __restrict__ part) {
  __shared__ double sh[kWaves];
  double rr = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const double v = fixed[i] ? 0.0 : (y ? f[i] - y[i] : f[i]);
    if (r) r[i] = v;
    rr += v * v;
  }
  rr = block_sum(rr, sh);
  if (threadIdx.x == 0) part[blockIdx.x] = rr;
}

__global__ void k_to_f32(int64_t n, const double* __restrict__ a, double scale, float* __restrict__ b) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    b[i] = (float)(a[i] * scale);
}

__global__ void k_axpy_f32(int64_t n, double s, const float* __restrict__ d, double* __restrict__ x) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    x[i] += s * (double)d[i];
}

__global__ void k_masked_set(int64_t n, const uint8_t* __restrict__ fixed, const double* __restrict__ ufix,
                             double* __restrict__ u) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    u[i] = fixed[i] ? (ufix ? ufix[i] : 0.0) : 0.0;
}

__global__ void k_cast_val(int64_t n, const double* __restrict__ a, float* __restrict__ b) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    b[i] = (float)a[i];
}

__global__ void k_axpy(int64_t n, double s, const double* __restrict__ d, double* __restrict__ x) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    x[i] += s * d[i];
}

// Scalar CSC operator (caller-supplied symmetric matrix, used as CSR of K^T),
// G lanes per row (csc_lanes).  A hexahedral or tetrahedral K has 60-90 entries a
// row: 32 lanes walk it in three steps and give a small system (5,400 rows: 675
// blocks instead of 169) a block on every CU.
template <typename MT, typename VT, int G, typename X>
__global__ __launch_bounds__(kBS) void k_spmv_csc(int64_t n, int passes, const int64_t* __restrict__ colptr,
                                                 const int32_t* __restrict__ rowval,
                                                 const MT* __restrict__ val, X xs,
                                                 const uint8_t* __restrict__ fixed, VT* __restrict__ y,
                                                 double* __restrict__ part,
                                                 const double* __restrict__ scal) {
  __shared__ double sh[2 * kWaves];
  const int64_t lb = xcd_block();
  const int l = (int)(threadIdx.x % G);
  int64_t j = lb * passes * (kBS / G) + threadIdx.x / G;
  int64_t p0 = 0, p1 = 0;
  auto span = [&]() {
    const int64_t i = j < n ? j : n - 1;
    p0 = colptr[i];
    p1 = j < n ? colptr[i + 1] : 0;
  };
  const double done = scal ? scal[S_DONE] : 0.0;
  xs.fetch();
  span();
  if (done != 0.0) return;
  if (!xs.begin(sh)) return;
  double d = 0.0;
  for (int ps = 0; ps < passes; ++ps, j += kBS / G, span()) {
    VT acc = 0;
#pragma unroll 4
    for (int64_t p = p0 + l; p < p1; p += G) acc += (VT)val[p] * xs.value(xs.raw(rowval[p]));
#pragma unroll
    for (int o = G / 2; o > 0; o >>= 1) acc += __shfl_xor(acc, o, G);
    if (j < n && l == 0) {
      const VT v = (fixed && fixed[j]) ? (VT)0 : acc;
      const VT xv = xs.value(xs.raw(j));
      y[j] = v;
      xs.keep(j, xv);
      d += (double)xv * (double)v;
    }
  }
  if (part) {
    const double s = block_sum(d, sh);
    if (threadIdx.x == 0) part[lb] = s;
  }
}

// Jacobi inverse of a CSC operator, kG lanes per column; of several stored
// diagonal entries the last one counts.
template <typename VT>
__global__ __launch_bounds__(kBS) void k_dinv_csc(int64_t n, const int64_t* __restrict__ colptr,
                                                  const int32_t* __restrict__ rowval, const double* __restrict__ val,
                                                  const uint8_t* __restrict__ fixed, VT* __restrict__ dinv) {
  const int64_t j = ((int64_t)blockIdx.x * kBS + threadIdx.x) / kG;
  if (j >= n) return;
  const int64_t p1 = colptr[j + 1];
  int64_t at = -1;
  for (int64_t p = colptr[j] + threadIdx.x % kG; p < p1; p += kG)
    if (rowval[p] == j) at = p;
#pragma unroll
  for (int o = kG / 2; o > 0; o >>= 1) at = max(at, (int64_t)__shfl_xor((long long)at, o, kG));
  if (threadIdx.x % kG != 0) return;
  const double dv = at >= 0 ? val[at] : 0.0;
  dinv[j] = (fixed[j] || dv == 0.0) ? (VT)0 : (VT)(1.0 / dv);
}

// Operator views.  Lanes per row of a panel operator: panel_lanes; of a CSC one
// by the average row and the number of rows.  More lanes shorten a row's chain
// of loads, which a small system waits for; a large one has waves enough, and
// what idle lanes and the longer butterfly cost is all that is left.
// us an iteration with 8, 16 and 32 lanes (one process, in turn):
//   below 20 entries 8: 17 entries, 5,000 rows 8.3, 8.5, 8.9, 60,000 12.9, 14.4,
//     16.7, 500,000 47.9, 61.3, 101;
//   20 to 48: 27-point (24) 4,913 rows 9.3, 8.7, 9.1, (26) 27,000 rows 12.1, 11.1, 12.9,
//     216,000 33.7, 32.1, 51.3; tet4 (43) 3,993 rows 9.4, 8.2, 8.4, 73,167 18.8, 18.9,
//     22.9; 16 up to 2^18 rows, then 8: tet4 352,947 rows 57, 64, 85, 680,943 114, 148,
//     205, 27-point 729,000 103, 114, 171;
//   48 to 128: tet10 (80) 3,993 rows 12.8, 10.5, 10.0, 46,875 21.0, 21.7, 21.4; band
//     (61) 5,000 rows 10.1, 10.0, 9.2; 32 up to 2^16 rows, then 16: hex8 (77) 73,167
//     24.2, 23.9, 27.1, 352,947 108, 106, 137, 823,875 229, 215 to 227, 303, band (61)
//     500,000 136, 144, 168, tet10 89,373 38.0, 33.6, 32.1, 273,375 89, 95, 112;
//   from 128: hex27 (148 to 180) 2,187 rows 16.8, 13.4, 11.3, 107,811 64, 67, 60,
//     206,763 160, 156, 149.
inline unsigned row_blocks(int64_t rows, int lanes) { return (unsigned)((rows * lanes + kBS - 1) / kBS); }
inline int csc_lanes(int64_t n, int64_t nnz) {
  if (nnz >= 128 * n) return 32;
  if (nnz >= 48 * n) return n <= (1 << 16) ? 32 : 16;
  return nnz >= 20 * n && n <= (1 << 18) ? 16 : kG;
}

struct PanelOp {
  static constexpr int64_t kFuseMax = 40000;   // DoFs up to which pcg forms the direction inside the SpMV
  int64_t N;
  const int64_t* adj_ptr;
  const int32_t* adj;
  const int32_t* dslot;
  int lanes;
  int64_t ndof() const { return 3 * N; }
  int64_t rows() const { return N; }
  template <typename MT, typename VT, typename X>
  void spmv(hipStream_t st, unsigned grid, int passes, const MT* val, const X& x, const uint8_t* fixed, VT* y,
            double* part, const double* scal) const {
    if (lanes == 32)
      k_spmv<MT, VT, 32, X><<<grid, kBS, 0, st>>>(N, passes, adj_ptr, adj, val, x, fixed, y, part, scal);
    else if (lanes == 16)
      k_spmv<MT, VT, 16, X><<<grid, kBS, 0, st>>>(N, passes, adj_ptr, adj, val, x, fixed, y, part, scal);
    else
      k_spmv<MT, VT, kG, X><<<grid, kBS, 0, st>>>(N, passes, adj_ptr, adj, val, x, fixed, y, part, scal);
  }
  template <typename VT>
  void dinv(hipStream_t st, const double* val, const uint8_t* fixed, VT* d) const {
    k_dinv<VT><<<(unsigned)((N + 255) / 256), 256, 0, st>>>(N, adj_ptr, dslot, val, fixed, d);
  }
};

struct CscOp {
  static constexpr int64_t kFuseMax = 24000;
  int64_t n;
  const int64_t* colptr;
  const int32_t* rowval;
  int lanes;
  int64_t ndof() const { return n; }
  int64_t rows() const { return n; }
  template <typename MT, typename VT, typename X>
  void spmv(hipStream_t st, unsigned grid, int passes, const MT* val, const X& x, const uint8_t* fixed, VT* y,
            double* part, const double* scal) const {
    if (lanes == 32)
      k_spmv_csc<MT, VT, 32, X><<<grid, kBS, 0, st>>>(n, passes, colptr, rowval, val, x, fixed, y, part, scal);
    else if (lanes == 16)
      k_spmv_csc<MT, VT, 16, X><<<grid, kBS, 0, st>>>(n, passes, colptr, rowval, val, x, fixed, y, part, scal);
    else
      k_spmv_csc<MT, VT, kG, X><<<grid, kBS, 0, st>>>(n, passes, colptr, rowval, val, x, fixed, y, part, scal);
  }
  template <typename VT>
  void dinv(hipStream_t st, const double* val, const uint8_t* fixed, VT* d) const {
    k_dinv_csc<VT><<<row_blocks(n, kG), kBS, 0, st>>>(n, colptr, rowval, val, fixed, d);
  }
};

// y = mask(K x) outside the iteration
template <typename Op>
void apply(hipStream_t st, const Op& K, const double* val, const double* x, const uint8_t* fixed, double* y) {
  K.template spmv<double, double>(st, row_blocks(K.rows(), K.lanes), 1, val, Plain<double>{x}, fixed, y, nullptr,
                                  nullptr);
}

inline unsigned vgrid(int64_t n, llfem_ctx* ctx) {
  int64_t g = (n + kBS - 1) / kBS;
  int64_t cap = (int64_t)std::max(ctx->num_cus, 1) * 8;
  return (unsigned)std::max<int64_t>(1, std::min<int64_t>(g, cap));
}

// What the host needs after a solve, in one go: the recursion's iterations,
// r.r and tolerance, and up to two sums of n partials (NULL: 0).
__global__ __launch_bounds__(kBS) void k_report(int64_t n, const double* __restrict__ part1,
                                                const double* __restrict__ part2, const double* __restrict__ scal,
                                                double* out) {
  __shared__ double sh[kWaves];
  const double s1 = part1 ? sum_partials(n, part1, sh) : 0.0;
  const double s2 = part2 ? sum_partials(n, part2, sh) : 0.0;
  if (threadIdx.x != 0) return;
  out[0] = scal[S_ITER];
  out[1] = scal[S_RR];
  out[2] = scal[S_TOL2];
  out[3] = s1;
  out[4] = s2;
}

struct Scratch {   // partial sums + scalars
  double* part;    // of the vector kernels
  double* spart;   // of the SpMV (ndof doubles: at most ndof / 8 blocks, then kFoldBlocks sums of them)
  double* red;
  double* scal;
};

// Jacobi-PCG (IterativeSolvers.cg semantics, x0 = 0) on vectors of type VT; b
// is overwritten (it is the second direction array once r holds it).
// The scalars stay on the device and each kernel sums the partials it needs,
// so an iteration is two launches -- SpMV of the direction formed on the fly,
// update -- up to the operator's kFuseMax DoFs, and three above, where gathering
// two vectors costs the SpMV more than the p-update's own launch and pass.
// Whole solves in ms, three / two launches: panels of 5,400 DoFs 3.39 / 2.73,
// 19,575 6.30 / 5.12, 30,345 7.78 / 6.43, 40,071 8.70 / 7.40, 44,403 14.1 /
// 14.6, 139,725 48.3 / 55.0; CSC 5,400 3.27 / 3.06, 19,575 7.63 / 6.79, 28,611
// 14.3 / 15.0, 30,345 10.4 / 10.1, 37,281 20.2 / 21.6.  With seven launches an
// iteration (separate reductions and scalars, a host wait every 16) the 12x11x40
// tet10 box (139,725 DoFs) to 1e-12 took 50 ms and a 5,400-DoF CSC 4.8 ms, with
// two or three 35.8 and 2.0; loads issued before the partials are summed and the
// done flag is seen, and eight partials under way a thread: 33.4 and 1.9.
// The host keeps two batches queued and looks at the flag after the older one,
// so the device never waits for it.
template <typename Op, typename MT, typename VT>
int pcg(llfem_ctx* ctx, const Op& K, const MT* val, const uint8_t* fixed, const VT* dinv, VT* b,
        VT* x, VT* r, VT* z, VT* p, VT* q, const Scratch& S, double rtol, int64_t maxiter) {
  hipStream_t st = ctx->stream;
  const int64_t n = K.ndof();
  const unsigned gv = vgrid(n, ctx);
  const int64_t groups = row_blocks(K.rows(), K.lanes);
  // up to kMaxPasses row groups a block keep the partials within kFoldMax
  const int64_t need = (groups + kFoldMax - 1) / kFoldMax;
  const int passes = need <= kMaxPasses ? (int)need : 1;
  const unsigned gs = (unsigned)((groups + passes - 1) / passes);
  const bool fold = (int64_t)gs > kFoldMax;
  const bool fuse = n <= Op::kFuseMax;
  volatile double* flag = ctx->h_poll;
  *flag = 0.0;
  k_init<VT><<<gv, kBS, 0, st>>>(n, x, b, r, dinv, z, p, S.part);
  k_init_scal<<<1, kBS, 0, st>>>(gv, S.part, S.scal, rtol, ctx->h_poll);
  VT* dir[2] = {p, b};
  auto direction = [&](int64_t it) {
    return Direction<VT>{z, dir[(it + 1) & 1], dir[it & 1], S.scal, S.part, (int64_t)gv, it, maxiter, ctx->h_poll, 0};
  };
  const int batch = 8;
  int64_t it = 0;
  for (int64_t k = 0;; ++k) {
    for (int i = 0; i < batch && it < maxiter; ++i, ++it) {
      VT* d = fuse ? dir[it & 1] : p;
      if (fuse) K.template spmv<MT, VT>(st, gs, passes, val, direction(it), fixed, q, S.spart, S.scal);
      else K.template spmv<MT, VT>(st, gs, passes, val, Plain<VT>{p}, fixed, q, S.spart, S.scal);
      if (fold) k_fold<<<kFoldBlocks, kBS, 0, st>>>(gs, S.spart, S.spart + gs, S.scal);
      k_update<VT><<<gv, kBS, 0, st>>>(n, S.scal, (int)(it & 1), fold ? (int64_t)kFoldBlocks : (int64_t)gs,
                                       fold ? S.spart + gs : S.spart, x, r, d, q, dinv, z, S.part);
      if (!fuse) k_pupd<VT><<<gv, kBS, 0, st>>>(n, S.scal, it, gv, S.part, maxiter, z, p, ctx->h_poll);
    }
    // the fused SpMV tests the update before it: one more when maxiter is reached
    if (fuse && it >= maxiter && it > 0)
      K.template spmv<MT, VT>(st, gs, passes, val, direction(it), fixed, q, S.spart, S.scal);
    LLFEM_HIP(hipEventRecord(ctx->poll_ev[k & 1], st));
    if (k > 0) LLFEM_HIP(hipEventSynchronize(ctx->poll_ev[(k - 1) & 1]));
    if (*flag != 0.0 || it >= maxiter) break;
  }
  LLFEM_HIP(hipGetLastError());
  return LLFEM_OK;
}

// Iterations and relative recursive residual of a finished pcg from the
// words k_report left.
void pcg_result(const llfem_ctx* ctx, double rtol, int64_t* iters, double* res_rel) {
  const double* h = ctx->h_poll + 1;
  *iters = (int64_t)h[0];
  const double b2 = rtol > 0 ? h[2] / (rtol * rtol) : 0.0;
  *res_rel = b2 > 0 ? std::sqrt(h[1] / b2) : 0.0;
}

__global__ void k_zero(int64_t n, double* __restrict__ a) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    a[i] = 0.0;
}

// Device workspace of solve_device_ws: 8 FP64 vectors of K.ndof(), the
// reduction partials and scalars, and 7 FP32 vectors for the mixed method.
template <typename Op>
size_t solve_ws_bytes(llfem_ctx* ctx, const Op& K, int method) {
  const int64_t n = K.ndof();
  const int64_t nparts = std::max<int64_t>(row_blocks(K.rows(), kG), 2 * (int64_t)vgrid(n, ctx)) + 2;
  const size_t nf = method == LLFEM_PCG_MIXED_REFINE ? 7 : 0;
  return sizeof(double) * (8 * (size_t)n + (size_t)nparts + 8 + S_NS + 8) + sizeof(float) * (nf * (size_t)n + 8);
}

// Full solve on device data: f, ufix (nullable) and u are device vectors of
// K.ndof(); fixed is a device 0/1 mask.  val32 is needed for the mixed method.
// `base` holds solve_ws_bytes(ctx, K, method) bytes; every part of it is
// written before it is read, so it may hold anything on entry.
template <typename Op>
int solve_device_ws(llfem_ctx* ctx, const Op& K, const double* val, const float* val32,
                    const uint8_t* fixed, const double* f, const double* ufix, int method, double reltol,
                    int64_t maxiter, double* u, llfem_stats* stats, void* base) {
  hipStream_t st = ctx->stream;
  const int64_t n = K.ndof();
  const unsigned gv = vgrid(n, ctx);
  const int64_t nparts = std::max<int64_t>(row_blocks(K.rows(), kG), 2 * (int64_t)gv) + 2;
  const bool mixed = (method == LLFEM_PCG_MIXED_REFINE);
  double* b = (double*)base;
  double* x = b + n;
  double* r = x + n;
  double* z = r + n;
  double* p = z + n;
  double* q = p + n;
  double* dinv = q + n;
  double* y = dinv + n;
  Scratch S{y + n, y, y + n + nparts, y + n + nparts + 8};   // y is free while pcg runs
  float* f32 = (float*)(S.scal + S_NS + 8);
  float *b32 = f32, *x32 = b32 + n, *r32 = x32 + n, *z32 = r32 + n, *p32 = z32 + n, *q32 = p32 + n,
        *dinv32 = q32 + n;

  K.template dinv<double>(st, val, fixed, dinv);
  if (mixed) K.template dinv<float>(st, val, fixed, dinv32);
  // u = u_fixed on constrained DoFs; b = mask(f - K u)  (src/linear.jl:3730-3733)
  k_masked_set<<<gv, kBS, 0, st>>>(n, fixed, ufix, u);
  apply(st, K, val, u, nullptr, y);
  k_resid<<<gv, kBS, 0, st>>>(n, f, y, fixed, b, S.part);
  int64_t total_it = 0, refinements = 0;
  bool converged = false;
  if (!mixed) {
    LLFEM_TRY((pcg<Op, double, double>(ctx, K, val, fixed, dinv, b, x, r, z, p, q, S, reltol, maxiter)));
    k_axpy<<<gv, kBS, 0, st>>>(n, 1.0, x, u);
  } else {
    double bn2 = 0.0;
    k_reduce<<<1, kBS, 0, st>>>(gv, 1, S.part, S.red);
    LLFEM_HIP(hipMemcpyAsync(&bn2, S.red, sizeof(double), hipMemcpyDeviceToHost, st));
    LLFEM_HIP(hipStreamSynchronize(st));
    const double bnorm = std::sqrt(bn2);
    // x accumulates the free-DoF correction in FP64; r is the FP64 residual
    k_zero<<<gv, kBS, 0, st>>>(n, x);
    LLFEM_HIP(hipMemcpyAsync(r, b, sizeof(double) * n, hipMemcpyDeviceToDevice, st));
    double rnorm = bnorm;
    const double inner_floor = 1e-5;
    const int max_ref = 40;
    while (refinements < max_ref && total_it < maxiter) {
      if (rnorm <= reltol * bnorm || bnorm == 0.0) { converged = true; break; }
      k_to_f32<<<gv, kBS, 0, st>>>(n, r, 1.0 / rnorm, b32);
      const double need = 0.5 * reltol * bnorm / rnorm;
      const double rin = std::max(inner_floor, std::min(1e-2, need));
      int64_t it = 0;
      double rr = 0.0;
      LLFEM_TRY((pcg<Op, float, float>(ctx, K, val32, fixed, dinv32, b32, x32, r32, z32, p32, q32, S,
                                       rin, maxiter - total_it)));
      k_axpy_f32<<<gv, kBS, 0, st>>>(n, rnorm, x32, x);
      // FP64 residual r = mask(b - K x)
      apply(st, K, val, x, fixed, y);
      k_resid<<<gv, kBS, 0, st>>>(n, b, y, fixed, r, S.part);
      k_report<<<1, kBS, 0, st>>>(gv, S.part, nullptr, S.scal, ctx->h_poll + 1);
      LLFEM_HIP(hipStreamSynchronize(st));
      pcg_result(ctx, rin, &it, &rr);
      total_it += it;
      rnorm = std::sqrt(ctx->h_poll[4]);
      ++refinements;
      if (it == 0) break;
    }
    if (!converged && rnorm <= reltol * bnorm) converged = true;
    k_axpy<<<gv, kBS, 0, st>>>(n, 1.0, x, u);
  }
  // reported residual: ||(K u - f)_free|| / ||f_free|| (test/test_dsl.jl:106)
  apply(st, K, val, u, nullptr, y);
  k_resid<<<gv, kBS, 0, st>>>(n, f, y, fixed, nullptr, S.part);
  k_resid<<<gv, kBS, 0, st>>>(n, f, nullptr, fixed, nullptr, S.part + gv);
  k_report<<<1, kBS, 0, st>>>(gv, S.part, S.part + gv, S.scal, ctx->h_poll + 1);
  LLFEM_HIP(hipStreamSynchronize(st));
  LLFEM_HIP(hipGetLastError());
  if (!mixed) {
    double rr = 0.0;
    pcg_result(ctx, reltol, &total_it, &rr);
    converged = rr <= reltol;
  }
  const double rr2 = ctx->h_poll[4], ff2 = ctx->h_poll[5];
  const double relres = ff2 > 0 ? std::sqrt(rr2 / ff2) : std::sqrt(rr2);
  if (stats) {
    stats->iterations = total_it;
    stats->rollbacks = 0;
    stats->restarts = 0;
    stats->refinements = refinements;
    stats->relres = relres;
  }
  if (!converged)
    return fail(LLFEM_ENOCONV, "cg: maxiter reached (relative residual " + std::to_string(relres) + ")");
  return LLFEM_OK;
}

// solve_device_ws on a workspace allocated for this call.
template <typename Op>
int solve_device(llfem_ctx* ctx, const Op& K, const double* val, const float* val32,
                 const uint8_t* fixed, const double* f, const double* ufix, int method, double reltol,
                 int64_t maxiter, double* u, llfem_stats* stats) {
  const size_t bytes = solve_ws_bytes(ctx, K, method);
  void* base = nullptr;
  LLFEM_TRY(dmalloc(ctx, &base, bytes));
  struct Free {
    llfem_ctx* c; void* p; size_t b;
    ~Free() { (void)hipStreamSynchronize(c->stream); dfree(c, p, b); }
  } guard{ctx, base, bytes};
  return solve_device_ws(ctx, K, val, val32, fixed, f, ufix, method, reltol, maxiter, u, stats, base);
}

__global__ void k_set_fixed(int64_t nfix, const int64_t* __restrict__ idx, int64_t base, int64_t n,
                            const double* __restrict__ vals, uint8_t* __restrict__ mask,
                            double* __restrict__ ufix, int* __restrict__ err) {
  int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nfix) return;
  const int64_t i = idx[k] - base;
  if (i < 0 || i >= n) { atomicOr(err, 1); return; }
  mask[i] = 1;
  ufix[i] = vals ? vals[k] : 0.0;
}

// Upload f, the fixed set and u_fixed; run solve_device; download u.
template <typename Op>
int solve_host(llfem_ctx* ctx, const Op& K, const double* val, const float* val32, int64_t n,
               const double* f, const int64_t* fixed, int64_t nfixed, int32_t one_based,
               const double* u_fixed, int32_t method, double reltol, int64_t maxiter, double* u_out,
               llfem_stats* stats) {
  hipStream_t st = ctx->stream;
  const size_t bytes = sizeof(double) * 3 * (size_t)n + (size_t)n + sizeof(int64_t) * (size_t)(nfixed + 1) +
                       sizeof(double) * (size_t)(nfixed + 1) + 64;
  char* base = nullptr;
  LLFEM_TRY(dmalloc(ctx, (void**)&base, bytes));
  struct Free {
    llfem_ctx* c; void* p; size_t b;
    ~Free() { (void)hipStreamSynchronize(c->stream); dfree(c, p, b); }
  } guard{ctx, base, bytes};
  double* d_f = (double*)base;
  double* d_u = d_f + n;
  double* d_ufix = d_u + n;
  int64_t* d_idx = (int64_t*)(d_ufix + n);
  double* d_vals = (double*)(d_idx + nfixed + 1);
  int* d_err = (int*)(d_vals + nfixed + 1);
  uint8_t* d_mask = (uint8_t*)(d_err + 2);
  LLFEM_HIP(hipMemcpyAsync(d_f, f, sizeof(double) * n, hipMemcpyHostToDevice, st));
  LLFEM_HIP(hipMemsetAsync(d_mask, 0, (size_t)n, st));
  LLFEM_HIP(hipMemsetAsync(d_ufix, 0, sizeof(double) * n, st));
  LLFEM_HIP(hipMemsetAsync(d_err, 0, sizeof(int), st));
  if (nfixed > 0) {
    LLFEM_HIP(hipMemcpyAsync(d_idx, fixed, sizeof(int64_t) * nfixed, hipMemcpyHostToDevice, st));
    if (u_fixed)
      LLFEM_HIP(hipMemcpyAsync(d_vals, u_fixed, sizeof(double) * nfixed, hipMemcpyHostToDevice, st));
    k_set_fixed<<<(unsigned)((nfixed + 255) / 256), 256, 0, st>>>(nfixed, d_idx, one_based ? 1 : 0, n,
                                                                   u_fixed ? d_vals : nullptr, d_mask,
                                                                   d_ufix, d_err);
  }
  int herr = 0;
  LLFEM_HIP(hipMemcpyAsync(&herr, d_err, sizeof(int), hipMemcpyDeviceToHost, st));
  LLFEM_HIP(hipStreamSynchronize(st));
  if (herr) return fail(LLFEM_EINVAL, "solveDisplacement: constrained DoF out of range");
  auto t0 = std::chrono::steady_clock::now();
  int s = solve_device(ctx, K, val, val32, d_mask, d_f, d_ufix, method, reltol, maxiter, d_u, stats);
  if (s != LLFEM_OK && s != LLFEM_ENOCONV) return s;
  LLFEM_TRY(copy_to_host(ctx, u_out, d_u, (size_t)n));
  if (stats)
    stats->total_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  return s;
}

__global__ void k_i64_to_i32(int64_t n, const int64_t* __restrict__ a, int64_t base, int32_t* __restrict__ b) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    b[i] = (int32_t)(a[i] - base);
}

__global__ void k_i64_sub(int64_t n, int64_t* __restrict__ a, int64_t base) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    a[i] -= base;
}

}  // namespace

// Upload f and the fixed set, run one system through the batched engine,
// download u.
int solve_host_reliable(llfem_ctx* ctx, SysSpec sp, bool f64_vectors, const double* f, const int64_t* fixed,
                        int64_t nfixed, int32_t one_based, const double* u_fixed, double* u_out,
                        llfem_stats* stats, llfem_mesh* amg_mesh) {
  hipStream_t st = ctx->stream;
  const int64_t n = 3 * sp.N;
  const size_t bytes = sizeof(double) * 3 * (size_t)n + (size_t)n + sizeof(int64_t) * (size_t)(nfixed + 1) +
                       sizeof(double) * (size_t)(nfixed + 1) + 64;
  char* base = nullptr;
  LLFEM_TRY(dmalloc(ctx, (void**)&base, bytes));
  struct Free {
    llfem_ctx* c; void* p; size_t b;
    ~Free() { (void)hipStreamSynchronize(c->stream); dfree(c, p, b); }
  } guard{ctx, base, bytes};
  double* d_f = (double*)base;
  double* d_u = d_f + n;
  double* d_ufix = d_u + n;
  int64_t* d_idx = (int64_t*)(d_ufix + n);
  double* d_vals = (double*)(d_idx + nfixed + 1);
  int* d_err = (int*)(d_vals + nfixed + 1);
  uint8_t* d_mask = (uint8_t*)(d_err + 2);
  LLFEM_HIP(hipMemcpyAsync(d_f, f, sizeof(double) * n, hipMemcpyHostToDevice, st));
  LLFEM_HIP(hipMemsetAsync(d_mask, 0, (size_t)n, st));
  LLFEM_HIP(hipMemsetAsync(d_ufix, 0, sizeof(double) * n, st));
  LLFEM_HIP(hipMemsetAsync(d_err, 0, sizeof(int), st));
  if (nfixed > 0) {
    LLFEM_HIP(hipMemcpyAsync(d_idx, fixed, sizeof(int64_t) * nfixed, hipMemcpyHostToDevice, st));
    if (u_fixed)
      LLFEM_HIP(hipMemcpyAsync(d_vals, u_fixed, sizeof(double) * nfixed, hipMemcpyHostToDevice, st));
    k_set_fixed<<<(unsigned)((nfixed + 255) / 256), 256, 0, st>>>(nfixed, d_idx, one_based ? 1 : 0, n,
                                                                   u_fixed ? d_vals : nullptr, d_mask,
                                                                   d_ufix, d_err);
  }
  int herr = 0;
  LLFEM_HIP(hipMemcpyAsync(&herr, d_err, sizeof(int), hipMemcpyDeviceToHost, st));
  LLFEM_HIP(hipStreamSynchronize(st));
  if (herr) return fail(LLFEM_EINVAL, "solveDisplacement: constrained DoF out of range");
  auto t0 = std::chrono::steady_clock::now();
  sp.fixed = d_mask;
  sp.f = d_f;
  sp.ufix = d_ufix;
  if (amg_mesh) {
    // the hierarchy of this support, built on first use and kept on the mesh
    uint64_t key = hash_bytes(&one_based, sizeof(one_based));
    key = hash_bytes(&nfixed, sizeof(nfixed), key);
    if (nfixed > 0) key = hash_bytes(fixed, sizeof(int64_t) * (size_t)nfixed, key);
    auto it = amg_mesh->amg.find(key);
    if (it == amg_mesh->amg.end()) {
      uint8_t* keep = nullptr;
      LLFEM_TRY(dalloc(ctx, &keep, (size_t)n));
      LLFEM_HIP(hipMemcpyAsync(keep, d_mask, (size_t)n, hipMemcpyDeviceToDevice, st));
      sp.fixed = keep;
      AmgHier* h = nullptr;
      const int rc = amg_build(ctx, sp, amg_mesh->d_xyz, &h);
      if (rc != LLFEM_OK) {
        (void)hipStreamSynchronize(st);
        dfree(ctx, keep, (size_t)n);
        return rc;
      }
      it = amg_mesh->amg.emplace(key, std::make_pair(h, keep)).first;
    }
    sp.fixed = it->second.second;
    sp.amg = it->second.first;
  }
  BatchSolver eng(ctx, f64_vectors);
  SolveSys* s = nullptr;
  LLFEM_TRY(eng.add(sp, &s));
  const double setup_ms =
      std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  // AMG systems reach the reliable-update trigger every ~10 iterations: short
  // chunks keep a paused system from idling through the rest of a chunk
  const int chunk = sp.amg ? 8 : 32;
  while (sys_status(s) == 0) {
    std::vector<SolveSys*> done;
    LLFEM_TRY(eng.run(chunk, &done));
  }
  LLFEM_TRY(eng.finish(s, d_u));
  LLFEM_TRY(copy_to_host(ctx, u_out, d_u, (size_t)n));
  const int status = sys_status(s);
  if (stats) {
    stats->iterations = sys_iterations(s);
    stats->rollbacks = sys_rollbacks(s);
    stats->restarts = sys_refreshes(s);
    stats->refinements = sys_updates(s);
    stats->relres = sys_relres(s);
    stats->total_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    stats->setup_ms = setup_ms;
  }
  const double rr = sys_relres(s);
  eng.remove(s);
  if (status == -2)
    return fail(LLFEM_ENOCONV, "cg: the FP32 correction was not finite in three successive updates");
  if (status != 1)
    return fail(LLFEM_ENOCONV, "cg: maxiter reached (relative residual " + std::to_string(rr) + ")");
  return LLFEM_OK;
}

// Make sure the mesh's FP32 copy of K exists (mixed-precision solve).
int ensure_k32(llfem_mesh* m) {
  if (m->d_valK32 && m->solver_ready) return LLFEM_OK;
  llfem_ctx* ctx = m->ctx;
  const int64_t nnz = 9 * m->nadj;
  if (!m->d_valK32) LLFEM_TRY(dalloc(ctx, &m->d_valK32, (size_t)nnz));
  k_cast_val<<<vgrid(nnz, ctx), kBS, 0, ctx->stream>>>(nnz, m->d_valK, m->d_valK32);
  m->solver_ready = true;
  return LLFEM_OK;
}

namespace {
// err |= 4: colptr does not start at 0 or ends below it; 1: colptr falls;
// 2: a row index out of range.  The row indices are only read while the ends
// are in order.
__global__ void k_check_csc(int64_t n, const int64_t* __restrict__ colptr, const int32_t* __restrict__ rowval,
                            int* __restrict__ err) {
  const int64_t nnz = colptr[n];
  if (colptr[0] != 0 || nnz < 0) {
    if (blockIdx.x == 0 && threadIdx.x == 0) atomicOr(err, 4);
    return;
  }
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; j < n; j += stride)
    if (colptr[j + 1] < colptr[j]) atomicOr(err, 1);
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < nnz; k += stride)
    if (rowval[k] < 0 || (int64_t)rowval[k] >= n) atomicOr(err, 2);
}

__global__ void k_check_report(int64_t n, const int64_t* __restrict__ colptr, const int* __restrict__ err,
                               double* out) {
  out[0] = (double)*err;
  out[1] = (double)colptr[n];
}

__global__ void k_zero_int(int* a) { *a = 0; }
}  // namespace

}  // namespace llfem

using namespace llfem;

extern "C" {

int llfem_solve(llfem_mesh* m, const double* f, const int64_t* fixed, int64_t nfixed, int32_t one_based,
                const double* u_fixed, int32_t method, double reltol, int64_t maxiter, double* u_out,
                llfem_stats* stats) {
  if (!m || !f || !u_out || (nfixed > 0 && !fixed)) return fail(LLFEM_EINVAL, "llfem_solve: NULL argument");
  if (!m->have_K) return fail(LLFEM_EINVAL, "llfem_solve: no stiffness assembled on this mesh");
  if (method != LLFEM_PCG_JACOBI_FP64 && method != LLFEM_PCG_MIXED_REFINE &&
      method != LLFEM_PCG_MIXED_RELIABLE && method != LLFEM_PCG_F32OP_RELIABLE &&
      method != LLFEM_PCG_AMG_RELIABLE)
    return fail(LLFEM_EUNSUP, "llfem_solve: unknown method");
  if (!(reltol > 0)) return fail(LLFEM_EINVAL, "llfem_solve: reltol must be positive");
  LLFEM_HIP(hipSetDevice(m->ctx->device));
  if (method == LLFEM_PCG_MIXED_RELIABLE || method == LLFEM_PCG_F32OP_RELIABLE ||
      method == LLFEM_PCG_AMG_RELIABLE) {
    SysSpec sp;
    sp.N = m->N;
    sp.nadj = m->nadj;
    sp.adj_ptr = m->d_adj_ptr;
    sp.adj = m->d_adj;
    sp.dslot = m->d_diag_slot;
    sp.val64 = m->d_valK;
    sp.reltol = reltol;
    sp.maxiter = maxiter;
    return solve_host_reliable(m->ctx, sp, method == LLFEM_PCG_F32OP_RELIABLE, f, fixed, nfixed, one_based,
                               u_fixed, u_out, stats, method == LLFEM_PCG_AMG_RELIABLE ? m : nullptr);
  }
  if (method == LLFEM_PCG_MIXED_REFINE) LLFEM_TRY(ensure_k32(m));
  PanelOp K{m->N, m->d_adj_ptr, m->d_adj, m->d_diag_slot, panel_lanes(m->N, m->nadj)};
  return solve_host(m->ctx, K, m->d_valK, m->d_valK32, 3 * m->N, f, fixed, nfixed, one_based, u_fixed,
                    method, reltol, maxiter, u_out, stats);
}

int llfem_solve_csc(llfem_ctx* ctx, int64_t n, const int64_t* colptr, const int64_t* rowval,
                    const double* nzval, int32_t one_based, const double* f, const int64_t* fixed,
                    int64_t nfixed, const double* u_fixed, int32_t method, double reltol, int64_t maxiter,
                    double* u_out, llfem_stats* stats) {
  if (!ctx || !colptr || !rowval || !nzval || !f || !u_out || (nfixed > 0 && !fixed))
    return fail(LLFEM_EINVAL, "llfem_solve_csc: NULL argument");
  if (n <= 0 || n >= ((int64_t)1 << 31)) return fail(LLFEM_EINVAL, "llfem_solve_csc: bad size");
  if (method != LLFEM_PCG_JACOBI_FP64 && method != LLFEM_PCG_MIXED_REFINE)
    return fail(LLFEM_EUNSUP, "llfem_solve_csc: unknown method");
  if (!(reltol > 0)) return fail(LLFEM_EINVAL, "llfem_solve_csc: reltol must be positive");
  const int64_t base = one_based ? 1 : 0;
  const int64_t nnz = colptr[n] - base;
  if (nnz < 0 || colptr[0] != base) return fail(LLFEM_EINVAL, "llfem_solve_csc: bad colptr");
  // the device SpMV trusts these indices: check them here (O(n + nnz))
  for (int64_t j = 0; j < n; ++j)
    if (colptr[j + 1] < colptr[j])
      return fail(LLFEM_EINVAL, "llfem_solve_csc: colptr is not non-decreasing at column " +
                                    std::to_string(j + base));
  for (int64_t k = 0; k < nnz; ++k)
    if (rowval[k] < base || rowval[k] >= n + base)
      return fail(LLFEM_EINVAL, "llfem_solve_csc: row index " + std::to_string(rowval[k]) + " out of range");
  LLFEM_HIP(hipSetDevice(ctx->device));
  hipStream_t st = ctx->stream;
  const size_t bytes = sizeof(int64_t) * (size_t)(n + 1) + sizeof(int64_t) * (size_t)nnz +
                       sizeof(int32_t) * (size_t)nnz + sizeof(double) * (size_t)nnz +
                       (method == LLFEM_PCG_MIXED_REFINE ? sizeof(float) * (size_t)nnz : 0) + 64;
  char* basep = nullptr;
  LLFEM_TRY(dmalloc(ctx, (void**)&basep, bytes));
  struct Free {
    llfem_ctx* c; void* p; size_t b;
    ~Free() { (void)hipStreamSynchronize(c->stream); dfree(c, p, b); }
  } guard{ctx, basep, bytes};
  int64_t* d_cp = (int64_t*)basep;
  int64_t* d_rv64 = d_cp + n + 1;
  double* d_val = (double*)(d_rv64 + nnz);
  int32_t* d_rv = (int32_t*)(d_val + nnz);
  float* d_val32 = (float*)(d_rv + nnz + (nnz & 1));
  LLFEM_HIP(hipMemcpyAsync(d_cp, colptr, sizeof(int64_t) * (n + 1), hipMemcpyHostToDevice, st));
  LLFEM_HIP(hipMemcpyAsync(d_rv64, rowval, sizeof(int64_t) * nnz, hipMemcpyHostToDevice, st));
  LLFEM_HIP(hipMemcpyAsync(d_val, nzval, sizeof(double) * nnz, hipMemcpyHostToDevice, st));
  k_i64_sub<<<vgrid(n + 1, ctx), kBS, 0, st>>>(n + 1, d_cp, base);
  k_i64_to_i32<<<vgrid(nnz, ctx), kBS, 0, st>>>(nnz, d_rv64, base, d_rv);
  if (method == LLFEM_PCG_MIXED_REFINE) k_cast_val<<<vgrid(nnz, ctx), kBS, 0, st>>>(nnz, d_val, d_val32);
  CscOp K{n, d_cp, d_rv, csc_lanes(n, nnz)};
  return solve_host(ctx, K, d_val, d_val32, n, f, fixed, nfixed, one_based, u_fixed, method, reltol,
                    maxiter, u_out, stats);
}

int llfem_solve_csc_noalloc(llfem_ctx* ctx, int64_t n, const int64_t* d_colptr, const int32_t* d_rowval,
                            const double* d_nzval, const double* d_f, const uint8_t* d_fixed,
                            const double* d_u_fixed, double reltol, int64_t maxiter, double* d_u_out,
                            llfem_stats* stats) {
  if (!ctx || !d_colptr || !d_rowval || !d_nzval || !d_f || !d_fixed || !d_u_out)
    return fail(LLFEM_EINVAL, "llfem_solve_csc_noalloc: NULL argument");
  if (n <= 0 || n >= ((int64_t)1 << 31)) return fail(LLFEM_EINVAL, "llfem_solve_csc_noalloc: bad size");
  if (!(reltol > 0)) return fail(LLFEM_EINVAL, "llfem_solve_csc_noalloc: reltol must be positive");
  CscOp K{n, d_colptr, d_rowval, kG};
  // the flag word of the index check sits after the solver's workspace
  const size_t ws = (solve_ws_bytes(ctx, K, LLFEM_PCG_JACOBI_FP64) + 255) & ~(size_t)255;
  if (ws + 256 > kNoAllocScratchBytes)
    return fail(LLFEM_EINVAL, "llfem_solve_csc_noalloc: ndof " + std::to_string(n) + " needs " +
                                  std::to_string(ws + 256) + " bytes of workspace; the maximum is " +
                                  std::to_string(kNoAllocScratchBytes) + " (about " +
                                  std::to_string(kNoAllocScratchBytes / 65) + " DoFs)");
  const int dev = ctx->device;
  void* ws_ptr = nullptr;
  std::mutex* ws_lock = nullptr;
  if (!noalloc_scratch(dev, &ws_ptr, &ws_lock))
    return fail(LLFEM_EINVAL, "llfem_solve_csc_noalloc: no workspace on device " + std::to_string(dev));
  LLFEM_HIP(hipSetDevice(dev));
  std::lock_guard<std::mutex> lk(*ws_lock);
  unsigned char* base = (unsigned char*)ws_ptr;
  int* d_err = (int*)(base + ws);
  hipStream_t st = ctx->stream;
  auto t0 = std::chrono::steady_clock::now();
  // the same index checks as llfem_solve_csc, on the device
  k_zero_int<<<1, 1, 0, st>>>(d_err);
  k_check_csc<<<vgrid(8 * n, ctx), kBS, 0, st>>>(n, d_colptr, d_rowval, d_err);
  k_check_report<<<1, 1, 0, st>>>(n, d_colptr, d_err, ctx->h_poll + 1);
  LLFEM_HIP(hipStreamSynchronize(st));
  LLFEM_HIP(hipGetLastError());
  const int herr = (int)ctx->h_poll[1];
  if (herr & 4) return fail(LLFEM_EINVAL, "llfem_solve_csc_noalloc: bad colptr");
  if (herr & 1) return fail(LLFEM_EINVAL, "llfem_solve_csc_noalloc: colptr is not non-decreasing");
  if (herr & 2) return fail(LLFEM_EINVAL, "llfem_solve_csc_noalloc: row index out of range");
  K.lanes = csc_lanes(n, (int64_t)ctx->h_poll[2]);
  const int s = solve_device_ws(ctx, K, d_nzval, nullptr, d_fixed, d_f, d_u_fixed, LLFEM_PCG_JACOBI_FP64,
                                reltol, maxiter, d_u_out, stats, base);
  if (s != LLFEM_OK && s != LLFEM_ENOCONV) return s;
  LLFEM_HIP(hipStreamSynchronize(st));
  if (stats)
    stats->total_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  return s;
}

}  // extern "C"
