// Load vectors: traction on a set of boundary elements (surface, curve or
// point elements), pressure on a set of 2D face elements, body force on the
// mesh's volume elements.
//
// Reference: loadVector(problem, [load(name; fx, fy, fz)]) (src/linear.jl:3088-3434):
// per boundary element and Gauss point, Ja = |t1 x t2| on a surface,
// |t1| on a curve and 1 at a point (src/linear.jl:3378-3388), from the
// element's Jacobian columns, f1 += H1' * t * Ja * w, then fp[nn2] += f1 in
// element order (src/linear.jl:3408-3413).
//
// Device version: one thread per face element computes the scalar nodal
// integrals s_a = sum_q N_a Ja w (the traction is uniform over the face);
// a second pass gathers them per node in ascending face order (face-node
// incidences prepared on the host), so the summation order matches the
// reference and no atomics are used.
//
// Body force (loadVector on a volume group, src/linear.jl:3054-3068, and
// ∫(Pu ⋅ g; Ω), src/multifield.jl:3496-3748): one thread per element
// integrates N_a g det J w, and one thread per node sums its elements'
// parts over the mesh's (node, element)-sorted incidence lists.  Pressure
// (src/linear.jl:3196-3224): per-face nodal unit normals, their per-node
// average times -p (normalVector + elementsToNodes), then the traction
// interpolated from the nodes and integrated like a traction.
#include <algorithm>
#include <cstring>
#include <numeric>

#include "common.h"

namespace {

// Measure of a boundary element of dimension fd at one point, from its
// Jacobian columns t1 = dx/dxi, t2 = dx/deta (src/linear.jl:3378-3388 for a
// 3D solid): |t1 x t2| on a surface, |t1| on a curve, 1 at a point.
__device__ inline double face_measure(int fd, const double t1[3], const double t2[3]) {
  if (fd == 2) {
    const double xy = t1[0] * t2[1] - t1[1] * t2[0];
    const double yz = t1[1] * t2[2] - t1[2] * t2[1];
    const double zx = t1[2] * t2[0] - t1[0] * t2[2];
    return sqrt(xy * xy + yz * yz + zx * zx);
  }
  if (fd == 1) return sqrt(t1[0] * t1[0] + t1[1] * t1[1] + t1[2] * t1[2]);
  return 1.0;
}

__global__ void k_face_integrals(int64_t F, int nf, int fd, int q, int64_t N, const double* __restrict__ xyz,
                                 const int32_t* __restrict__ fconn, const double* __restrict__ w,
                                 const double* __restrict__ Nref, const double* __restrict__ dN,
                                 double* __restrict__ s) {
  int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= F) return;
  for (int a = 0; a < nf; ++a) s[e * nf + a] = 0.0;
  for (int p = 0; p < q; ++p) {
    double t1[3] = {0, 0, 0}, t2[3] = {0, 0, 0};
    for (int a = 0; a < nf; ++a) {
      const int32_t v = fconn[e * nf + a];
      const double x[3] = {xyz[v], xyz[N + v], xyz[2 * N + v]};
      const double g0 = dN[((size_t)p * nf + a) * 3], g1 = dN[((size_t)p * nf + a) * 3 + 1];
      for (int i = 0; i < 3; ++i) {
        t1[i] += x[i] * g0;
        t2[i] += x[i] * g1;
      }
    }
    const double Ja = face_measure(fd, t1, t2);
    for (int a = 0; a < nf; ++a) s[e * nf + a] += Nref[(size_t)p * nf + a] * Ja * w[p];
  }
}

__global__ void k_face_gather(int64_t nnodes, const int32_t* __restrict__ nodes,
                              const int32_t* __restrict__ ptr, const int32_t* __restrict__ slots,
                              const double* __restrict__ s, double t0, double t1, double t2,
                              double* __restrict__ f) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nnodes) return;
  double acc = 0.0;
  for (int k = ptr[i]; k < ptr[i + 1]; ++k) acc += s[slots[k]];
  const int64_t v = nodes[i];
  f[3 * v] = t0 * acc;
  f[3 * v + 1] = t1 * acc;
  f[3 * v + 2] = t2 * acc;
}

// Physical coordinates of the face Gauss points: thread per (face, point).
__global__ void k_face_points(int64_t F, int nf, int q, int64_t N, const double* __restrict__ xyz,
                              const int32_t* __restrict__ fconn, const double* __restrict__ Nref,
                              double* __restrict__ out) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= F * q) return;
  const int64_t e = t / q;
  const int p = (int)(t - e * q);
  double x[3] = {0.0, 0.0, 0.0};
  for (int a = 0; a < nf; ++a) {
    const int32_t v = fconn[e * nf + a];
    const double h = Nref[(size_t)p * nf + a];
    x[0] += h * xyz[v];
    x[1] += h * xyz[N + v];
    x[2] += h * xyz[2 * N + v];
  }
  for (int i = 0; i < 3; ++i) out[t * 3 + i] = x[i];
}

// Per face element and node a: s3[a][c] = sum_q N_a t_c(q) Ja w_q, the
// traction given per Gauss point (t [F][q][3]).
__global__ void k_face_integrals_gp(int64_t F, int nf, int fd, int q, int64_t N, const double* __restrict__ xyz,
                                    const int32_t* __restrict__ fconn, const double* __restrict__ w,
                                    const double* __restrict__ Nref, const double* __restrict__ dN,
                                    const double* __restrict__ tgp, double* __restrict__ s3) {
  int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= F) return;
  for (int a = 0; a < 3 * nf; ++a) s3[e * nf * 3 + a] = 0.0;
  for (int p = 0; p < q; ++p) {
    double t1[3] = {0, 0, 0}, t2[3] = {0, 0, 0};
    for (int a = 0; a < nf; ++a) {
      const int32_t v = fconn[e * nf + a];
      const double x[3] = {xyz[v], xyz[N + v], xyz[2 * N + v]};
      const double g0 = dN[((size_t)p * nf + a) * 3], g1 = dN[((size_t)p * nf + a) * 3 + 1];
      for (int i = 0; i < 3; ++i) {
        t1[i] += x[i] * g0;
        t2[i] += x[i] * g1;
      }
    }
    const double Ja = face_measure(fd, t1, t2);
    const double* tq = tgp + (e * q + p) * 3;
    for (int a = 0; a < nf; ++a) {
      const double c = Nref[(size_t)p * nf + a] * Ja * w[p];
      for (int i = 0; i < 3; ++i) s3[(e * nf + a) * 3 + i] += c * tq[i];
    }
  }
}

__global__ void k_face_gather3(int64_t nnodes, const int32_t* __restrict__ nodes,
                               const int32_t* __restrict__ ptr, const int32_t* __restrict__ slots,
                               const double* __restrict__ s3, double* __restrict__ f) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nnodes) return;
  double acc[3] = {0.0, 0.0, 0.0};
  for (int k = ptr[i]; k < ptr[i + 1]; ++k)
    for (int c = 0; c < 3; ++c) acc[c] += s3[(size_t)slots[k] * 3 + c];
  const int64_t v = nodes[i];
  for (int c = 0; c < 3; ++c) f[3 * v + c] = acc[c];
}

// ---- volume loads ---------------------------------------------------------
// Per element e of the set (pos[e] >= 0; pos NULL: every element, k = e) and
// node a, with J_q = sum_b x_b dN_b(xi_q)^T on coordinates relative to the
// element's first node and its signed det J (as gmsh's getJacobian gives it):
//   constant force:  s[a][e] = sum_q N_a(xi_q) det J_q w_q
//   per Gauss point: s[3 a + c][e] = sum_q N_a g_c(q) det J_q w_q, g = gp[k][q][3].
// Elements outside the set get zeros.  Connectivity is the mesh's SoA [npe][E].
//
// Constant force, one thread per element: its node coordinates stay in
// registers over the points and the sums leave once, coalesced ([a][E]).  The
// tables are the same for every lane (scalar loads).  Bound: the FP64 point
// sums, 9 npe fma each (E = 331,776 tet10, 15 points: 0.45 G fma).  Adding
// every point's terms to three components in memory instead took 1,971 us
// there; this takes 45 us, and the
// gather of one value per incidence instead of three 21 us instead of 77.
template <int NPE>
__global__ __launch_bounds__(256) void k_body_const(int64_t E, int q, const double4* __restrict__ xyz4,
                                                    const int32_t* __restrict__ conn,
                                                    const int32_t* __restrict__ pos, const double* __restrict__ w,
                                                    const double* __restrict__ Nref, const double* __restrict__ dN,
                                                    double* __restrict__ s) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= E) return;
  double x[NPE], y[NPE], z[NPE], acc[NPE];
  int32_t v[NPE];
#pragma unroll
  for (int a = 0; a < NPE; ++a) v[a] = conn[(int64_t)a * E + e];
#pragma unroll
  for (int a = 0; a < NPE; ++a) {
    const double4 c = xyz4[v[a]];
    x[a] = c.x;
    y[a] = c.y;
    z[a] = c.z;
    acc[a] = 0.0;
  }
#pragma unroll
  for (int a = 1; a < NPE; ++a) {
    x[a] -= x[0];
    y[a] -= y[0];
    z[a] -= z[0];
  }
  if (!pos || pos[e] >= 0) {
    for (int p = 0; p < q; ++p) {
      double J[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
      const double* g = dN + (size_t)p * NPE * 3;
#pragma unroll
      for (int a = 1; a < NPE; ++a) {
        const double g0 = g[3 * a], g1 = g[3 * a + 1], g2 = g[3 * a + 2];
        J[0] += x[a] * g0; J[1] += x[a] * g1; J[2] += x[a] * g2;
        J[3] += y[a] * g0; J[4] += y[a] * g1; J[5] += y[a] * g2;
        J[6] += z[a] * g0; J[7] += z[a] * g1; J[8] += z[a] * g2;
      }
      const double det = J[0] * (J[4] * J[8] - J[5] * J[7]) - J[1] * (J[3] * J[8] - J[5] * J[6]) +
                         J[2] * (J[3] * J[7] - J[4] * J[6]);
      const double dw = det * w[p];
#pragma unroll
      for (int a = 0; a < NPE; ++a) acc[a] += Nref[(size_t)p * NPE + a] * dw;
    }
  }
#pragma unroll
  for (int a = 0; a < NPE; ++a) s[(int64_t)a * E + e] = acc[a];
}

// Any element and either kind of force, one wavefront per element: node
// coordinates in LDS, a lane per point for det J (64 points at a time), then
// a lane per node for the sums over them.  rule: w [q], N [q][npe], dN [q][npe][3].
constexpr int kBodyWaves = 4;

template <bool GP>
__global__ __launch_bounds__(64 * kBodyWaves) void k_body_any(int64_t E, int npe, int q,
                                                              const double4* __restrict__ xyz4,
                                                              const int32_t* __restrict__ conn,
                                                              const int32_t* __restrict__ pos,
                                                              const double* __restrict__ w,
                                                              const double* __restrict__ Nref,
                                                              const double* __restrict__ dN,
                                                              const double* __restrict__ gp_,
                                                              double* __restrict__ s) {
  extern __shared__ double lds[];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  double* rel = lds + (size_t)wave * (3 * npe + 64 * 4);   // x, y, z [npe], then det J w [64], g [64][3]
  double* dw = rel + 3 * npe;
  double* gq = dw + 64;
  const int64_t e = (int64_t)blockIdx.x * kBodyWaves + wave;
  constexpr int C = GP ? 3 : 1;
  const int64_t k = e < E ? (pos ? (int64_t)pos[e] : e) : -1;   // wave-uniform
  if (e < E && k < 0)
    for (int a = lane; a < npe; a += 64)
      for (int c = 0; c < C; ++c) s[(int64_t)(C * a + c) * E + e] = 0.0;
  if (k >= 0) {
    const double4 c0 = xyz4[conn[e]];
    for (int a = lane; a < npe; a += 64) {
      const double4 c = xyz4[conn[(int64_t)a * E + e]];
      rel[a] = c.x - c0.x;
      rel[npe + a] = c.y - c0.y;
      rel[2 * npe + a] = c.z - c0.z;
    }
  }
  for (int p0 = 0; p0 < q; p0 += 64) {
    __syncthreads();
    const int p = p0 + lane;
    if (k >= 0 && p < q) {
      double J[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
      const double* g = dN + (size_t)p * npe * 3;
      for (int a = 1; a < npe; ++a) {
        const double x = rel[a], y = rel[npe + a], z = rel[2 * npe + a];
        const double g0 = g[3 * a], g1 = g[3 * a + 1], g2 = g[3 * a + 2];
        J[0] += x * g0; J[1] += x * g1; J[2] += x * g2;
        J[3] += y * g0; J[4] += y * g1; J[5] += y * g2;
        J[6] += z * g0; J[7] += z * g1; J[8] += z * g2;
      }
      const double det = J[0] * (J[4] * J[8] - J[5] * J[7]) - J[1] * (J[3] * J[8] - J[5] * J[6]) +
                         J[2] * (J[3] * J[7] - J[4] * J[6]);
      dw[lane] = det * w[p];
      if constexpr (GP)
        for (int c = 0; c < 3; ++c) gq[3 * lane + c] = gp_[((size_t)k * q + p) * 3 + c];
    }
    __syncthreads();
    if (k < 0) continue;
    const int np = min(64, q - p0);
    for (int a = lane; a < npe; a += 64) {
      double acc[C];
      for (int c = 0; c < C; ++c) acc[c] = p0 ? s[(int64_t)(C * a + c) * E + e] : 0.0;
      for (int i = 0; i < np; ++i) {
        const double h = Nref[(size_t)(p0 + i) * npe + a] * dw[i];
        if constexpr (GP)
          for (int c = 0; c < 3; ++c) acc[c] += h * gq[3 * i + c];
        else
          acc[0] += h;
      }
      for (int c = 0; c < C; ++c) s[(int64_t)(C * a + c) * E + e] = acc[c];
    }
  }
}

// f[node] = sum of the element parts over the node's incidences in ascending
// element order (the mesh's (node, element)-sorted incidence lists), times
// the constant force where the parts are scalars.  There the set (pos, NULL:
// every element) is asked again: a node that no element of it touches gets 0
// whatever the force, and an infinite one times 0 is none.
template <bool GP>
__global__ __launch_bounds__(256) void k_body_gather(int64_t N, int64_t E, const int32_t* __restrict__ inc_ptr,
                                                     const int32_t* __restrict__ inc_elem,
                                                     const uint8_t* __restrict__ inc_loc,
                                                     const int32_t* __restrict__ pos, const double* __restrict__ s,
                                                     double g0, double g1, double g2, double* __restrict__ f) {
  const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= N) return;
  const int32_t k1 = inc_ptr[v + 1];
  if constexpr (GP) {
    double acc[3] = {0.0, 0.0, 0.0};
    for (int32_t k = inc_ptr[v]; k < k1; ++k)
      for (int c = 0; c < 3; ++c) acc[c] += s[(int64_t)(3 * inc_loc[k] + c) * E + inc_elem[k]];
    for (int c = 0; c < 3; ++c) f[3 * v + c] = acc[c];
  } else {
    double acc = 0.0;
#pragma unroll 4
    for (int32_t k = inc_ptr[v]; k < k1; ++k) acc += s[(int64_t)inc_loc[k] * E + inc_elem[k]];
    bool in = !pos;
    if (pos)
      for (int32_t k = inc_ptr[v]; k < k1 && !in; ++k) in = pos[inc_elem[k]] >= 0;
    f[3 * v] = in ? g0 * acc : 0.0;
    f[3 * v + 1] = in ? g1 * acc : 0.0;
    f[3 * v + 2] = in ? g2 * acc : 0.0;
  }
}

// Physical coordinates of the Gauss points of the elements elems[0..ne) (NULL: all).
__global__ void k_volume_points(int64_t ne, int64_t E, int npe, int q, int64_t N, const double* __restrict__ xyz,
                                const int32_t* __restrict__ conn, const int32_t* __restrict__ elems,
                                const double* __restrict__ Nref, double* __restrict__ out) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= ne * q) return;
  const int64_t k = t / q;
  const int p = (int)(t - k * q);
  const int64_t e = elems ? elems[k] : k;
  double x[3] = {0.0, 0.0, 0.0};
  for (int a = 0; a < npe; ++a) {
    const int32_t v = conn[(int64_t)a * E + e];
    const double h = Nref[(size_t)p * npe + a];
    x[0] += h * xyz[v];
    x[1] += h * xyz[N + v];
    x[2] += h * xyz[2 * N + v];
  }
  for (int i = 0; i < 3; ++i) out[t * 3 + i] = x[i];
}

// ---- pressure ---------------------------------------------------------------
// Unit normal of face e at its own local node k: n = t1 x t2 / |t1 x t2| with
// t1, t2 = sum_a x_a dN_a,xi / dN_a,eta evaluated at node k (dNn [k][a][3]).
__global__ void k_face_node_normals(int64_t F, int nf, int64_t N, const double* __restrict__ xyz,
                                    const int32_t* __restrict__ fconn, const double* __restrict__ dNn,
                                    double* __restrict__ nrm) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= F * nf) return;
  const int64_t e = t / nf;
  const int k = (int)(t - e * nf);
  double t1[3] = {0, 0, 0}, t2[3] = {0, 0, 0};
  for (int a = 0; a < nf; ++a) {
    const int32_t v = fconn[e * nf + a];
    const double x[3] = {xyz[v], xyz[N + v], xyz[2 * N + v]};
    const double g0 = dNn[((size_t)k * nf + a) * 3], g1 = dNn[((size_t)k * nf + a) * 3 + 1];
    for (int i = 0; i < 3; ++i) {
      t1[i] += g0 * x[i];
      t2[i] += g1 * x[i];
    }
  }
  const double nx = t1[1] * t2[2] - t1[2] * t2[1];
  const double ny = t1[2] * t2[0] - t1[0] * t2[2];
  const double nz = t1[0] * t2[1] - t1[1] * t2[0];
  const double len = sqrt(nx * nx + ny * ny + nz * nz);
  nrm[t * 3] = nx / len;
  nrm[t * 3 + 1] = ny / len;
  nrm[t * 3 + 2] = nz / len;
}

// Nodal traction of the pressure on face-set node i (node nodes[i]):
// t_c = (sum over its incidences, ascending face order, of (-n_c) p) * (1 / count),
// p = p_nodal[node] or the constant p.
__global__ void k_pressure_nodal(int64_t nnodes, const int32_t* __restrict__ nodes, const int32_t* __restrict__ ptr,
                                 const int32_t* __restrict__ slots, const double* __restrict__ nrm, double p,
                                 const double* __restrict__ p_nodal, double* __restrict__ tn) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nnodes) return;
  const double pv = p_nodal ? p_nodal[nodes[i]] : p;
  double acc[3] = {0.0, 0.0, 0.0};
  for (int k = ptr[i]; k < ptr[i + 1]; ++k)
    for (int c = 0; c < 3; ++c) acc[c] += (-nrm[(size_t)slots[k] * 3 + c]) * pv;
  const double factor = 1.0 / (double)(ptr[i + 1] - ptr[i]);
  for (int c = 0; c < 3; ++c) tn[i * 3 + c] = acc[c] * factor;
}

// Per face e and node a: s3[e][a][c] = sum_q ((N_a t_c(q)) Ja) w_q with the
// traction interpolated from the nodal values, t(q) = sum_b N_b tn[b].
__global__ void k_face_integrals_nodal(int64_t F, int nf, int q, int64_t N, const double* __restrict__ xyz,
                                       const int32_t* __restrict__ fconn, const double* __restrict__ w,
                                       const double* __restrict__ Nref, const double* __restrict__ dN,
                                       const int32_t* __restrict__ slot_node, const double* __restrict__ tn,
                                       double* __restrict__ s3) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= F) return;
  for (int a = 0; a < 3 * nf; ++a) s3[e * nf * 3 + a] = 0.0;
  for (int p = 0; p < q; ++p) {
    double t1[3] = {0, 0, 0}, t2[3] = {0, 0, 0}, tq[3] = {0, 0, 0};
    for (int a = 0; a < nf; ++a) {
      const int32_t v = fconn[e * nf + a];
      const double x[3] = {xyz[v], xyz[N + v], xyz[2 * N + v]};
      const double g0 = dN[((size_t)p * nf + a) * 3], g1 = dN[((size_t)p * nf + a) * 3 + 1];
      const double h = Nref[(size_t)p * nf + a];
      const double* tb = tn + (size_t)slot_node[e * nf + a] * 3;
      for (int i = 0; i < 3; ++i) {
        t1[i] += x[i] * g0;
        t2[i] += x[i] * g1;
        tq[i] += h * tb[i];
      }
    }
    const double xy = t1[0] * t2[1] - t1[1] * t2[0];
    const double yz = t1[1] * t2[2] - t1[2] * t2[1];
    const double zx = t1[2] * t2[0] - t1[0] * t2[2];
    const double Ja = sqrt(xy * xy + yz * yz + zx * zx);
    for (int a = 0; a < nf; ++a) {
      const double h = Nref[(size_t)p * nf + a];
      for (int i = 0; i < 3; ++i) s3[(e * nf + a) * 3 + i] += ((h * tq[i]) * Ja) * w[p];
    }
  }
}

}  // namespace

using namespace llfem;

namespace {

// Host side of a face set: 0-based connectivity and the face-node incidences
// in ascending face order (nodes, ptr into slots).
struct FacePrep {
  std::vector<int32_t> fc, slots, nodes, ptr;
};

int prepare_faces(const llfem_mesh* m, int32_t face_type, int32_t nf, const int64_t* face_conn, int64_t F,
                  int32_t one_based, int32_t q, FacePrep* P) {
  const int fd = etype_dim(face_type);
  if (fd < 0 || fd > 2)
    return fail(LLFEM_EUNSUP, "loadVector: boundary element type " + std::to_string(face_type) +
                                  " is not a surface, curve or point element");
  if (nf <= 0 || q <= 0 || F < 0) return fail(LLFEM_EINVAL, "loadVector: bad face-set sizes");
  const int64_t base = one_based ? 1 : 0;
  P->fc.resize((size_t)F * nf);
  for (int64_t i = 0; i < F * nf; ++i) {
    const int64_t v = face_conn[i] - base;
    if (v < 0 || v >= m->N) return fail(LLFEM_EINVAL, "loadVector: face node out of range");
    P->fc[i] = (int32_t)v;
  }
  P->slots.resize((size_t)F * nf);
  std::iota(P->slots.begin(), P->slots.end(), 0);
  std::stable_sort(P->slots.begin(), P->slots.end(), [&](int32_t x, int32_t y) { return P->fc[x] < P->fc[y]; });
  P->nodes.clear();
  P->ptr.assign(1, 0);
  for (size_t k = 0; k < P->slots.size(); ++k)
    if (k == 0 || P->fc[P->slots[k]] != P->fc[P->slots[k - 1]]) {
      if (k) P->ptr.push_back((int32_t)k);
      P->nodes.push_back(P->fc[P->slots[k]]);
    }
  P->ptr.push_back((int32_t)P->slots.size());
  return LLFEM_OK;
}

}  // namespace

namespace {

// Host arrays of one call, laid out 256-byte aligned and sent to the device
// in one copy.
class Upload {
 public:
  template <typename T>
  size_t add(const T* p, size_t n) {
    const size_t at = buf_.size();
    buf_.resize(at + WsGuard::aligned(n * sizeof(T)));
    if (n) std::memcpy(buf_.data() + at, p, n * sizeof(T));
    return at;
  }
  size_t bytes() const { return buf_.size(); }
  hipError_t send(char* dev, hipStream_t st) const {
    return buf_.empty() ? hipSuccess : hipMemcpyAsync(dev, buf_.data(), buf_.size(), hipMemcpyHostToDevice, st);
  }

 private:
  std::vector<char> buf_;
};

int load_failed(const char* who, hipError_t e) {
  return fail(LLFEM_EHIP, std::string(who) + ": " + hipGetErrorString(e));
}

// f (3 N, on the device) to the caller
int finish_load(llfem_ctx* ctx, const char* who, const double* d_f, int64_t N, double* f_out) {
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return load_failed(who, e);
  return copy_to_host(ctx, f_out, d_f, 3 * (size_t)N);
}

}  // namespace

extern "C" int llfem_load_traction(llfem_mesh* m, int32_t face_type, int32_t nf,
                                   const int64_t* face_conn, int64_t F, int32_t one_based, int32_t q,
                                   const double* weights, const double* N_ref, const double* dN_ref,
                                   const double traction[3], double* f_out) {
  if (!m || !face_conn || !weights || !N_ref || !dN_ref || !traction || !f_out)
    return fail(LLFEM_EINVAL, "llfem_load_traction: NULL argument");
  FacePrep P;
  LLFEM_TRY(prepare_faces(m, face_type, nf, face_conn, F, one_based, q, &P));
  llfem_ctx* ctx = m->ctx;
  LLFEM_HIP(hipSetDevice(ctx->device));
  hipStream_t st = ctx->stream;
  const int64_t N = m->N, nn = (int64_t)P.nodes.size();
  Upload up;
  const size_t o_fc = up.add(P.fc.data(), P.fc.size()), o_nodes = up.add(P.nodes.data(), P.nodes.size()),
               o_ptr = up.add(P.ptr.data(), P.ptr.size()), o_slots = up.add(P.slots.data(), P.slots.size()),
               o_w = up.add(weights, q), o_N = up.add(N_ref, (size_t)q * nf), o_dN = up.add(dN_ref, (size_t)q * nf * 3);
  const size_t ns = (size_t)F * nf;
  WsGuard ws(ctx);
  LLFEM_TRY(ws.get(up.bytes() + WsGuard::aligned(8 * ns) + WsGuard::aligned(24 * (size_t)N)));
  char* d = ws.take<char>(up.bytes());
  double *d_s = ws.take<double>(ns), *d_f = ws.take<double>(3 * (size_t)N);
  hipError_t e = up.send(d, st);
  e = e ? e : hipMemsetAsync(d_f, 0, sizeof(double) * 3 * N, st);
  if (e != hipSuccess) return load_failed("loadVector upload", e);
  if (F > 0) {
    k_face_integrals<<<(unsigned)((F + 127) / 128), 128, 0, st>>>(
        F, nf, etype_dim(face_type), q, N, m->d_xyz, (const int32_t*)(d + o_fc), (const double*)(d + o_w),
        (const double*)(d + o_N), (const double*)(d + o_dN), d_s);
    k_face_gather<<<(unsigned)((nn + 255) / 256), 256, 0, st>>>(
        nn, (const int32_t*)(d + o_nodes), (const int32_t*)(d + o_ptr), (const int32_t*)(d + o_slots), d_s,
        traction[0], traction[1], traction[2], d_f);
  }
  return finish_load(ctx, "loadVector", d_f, N, f_out);
}

extern "C" int llfem_face_points(llfem_mesh* m, int32_t face_type, int32_t nf, const int64_t* face_conn, int64_t F,
                                 int32_t one_based, int32_t q, const double* N_ref, double* xyz_out) {
  if (!m || !face_conn || !N_ref || !xyz_out) return fail(LLFEM_EINVAL, "llfem_face_points: NULL argument");
  FacePrep P;
  LLFEM_TRY(prepare_faces(m, face_type, nf, face_conn, F, one_based, q, &P));
  llfem_ctx* ctx = m->ctx;
  LLFEM_HIP(hipSetDevice(ctx->device));
  hipStream_t st = ctx->stream;
  const size_t npts = (size_t)F * q;
  Upload up;
  const size_t o_fc = up.add(P.fc.data(), P.fc.size()), o_N = up.add(N_ref, (size_t)q * nf);
  WsGuard ws(ctx);
  LLFEM_TRY(ws.get(up.bytes() + WsGuard::aligned(24 * npts)));
  char* d = ws.take<char>(up.bytes());
  double* d_out = ws.take<double>(3 * npts);
  hipError_t e = up.send(d, st);
  if (e == hipSuccess && npts > 0) {
    k_face_points<<<(unsigned)((npts + 255) / 256), 256, 0, st>>>(F, nf, q, m->N, m->d_xyz,
                                                                  (const int32_t*)(d + o_fc),
                                                                  (const double*)(d + o_N), d_out);
    e = hipGetLastError();
  }
  if (e != hipSuccess) return load_failed("llfem_face_points", e);
  return copy_to_host(ctx, xyz_out, d_out, 3 * npts);
}

extern "C" int llfem_load_traction_gp(llfem_mesh* m, int32_t face_type, int32_t nf, const int64_t* face_conn,
                                      int64_t F, int32_t one_based, int32_t q, const double* weights,
                                      const double* N_ref, const double* dN_ref, const double* t_gp,
                                      double* f_out) {
  if (!m || !face_conn || !weights || !N_ref || !dN_ref || !t_gp || !f_out)
    return fail(LLFEM_EINVAL, "llfem_load_traction_gp: NULL argument");
  FacePrep P;
  LLFEM_TRY(prepare_faces(m, face_type, nf, face_conn, F, one_based, q, &P));
  llfem_ctx* ctx = m->ctx;
  LLFEM_HIP(hipSetDevice(ctx->device));
  hipStream_t st = ctx->stream;
  const int64_t N = m->N, nn = (int64_t)P.nodes.size();
  Upload up;
  const size_t o_fc = up.add(P.fc.data(), P.fc.size()), o_nodes = up.add(P.nodes.data(), P.nodes.size()),
               o_ptr = up.add(P.ptr.data(), P.ptr.size()), o_slots = up.add(P.slots.data(), P.slots.size()),
               o_w = up.add(weights, q), o_N = up.add(N_ref, (size_t)q * nf), o_dN = up.add(dN_ref, (size_t)q * nf * 3);
  const size_t ns = 3 * (size_t)F * nf, nt = 3 * (size_t)F * q;
  WsGuard ws(ctx);
  LLFEM_TRY(ws.get(up.bytes() + WsGuard::aligned(8 * ns) + WsGuard::aligned(8 * nt) +
                   WsGuard::aligned(24 * (size_t)N)));
  char* d = ws.take<char>(up.bytes());
  double *d_s3 = ws.take<double>(ns), *d_t = ws.take<double>(nt), *d_f = ws.take<double>(3 * (size_t)N);
  hipError_t e = up.send(d, st);
  e = e ? e : hipMemcpyAsync(d_t, t_gp, sizeof(double) * nt, hipMemcpyHostToDevice, st);
  e = e ? e : hipMemsetAsync(d_f, 0, sizeof(double) * 3 * N, st);
  if (e != hipSuccess) return load_failed("loadVector upload", e);
  if (F > 0) {
    k_face_integrals_gp<<<(unsigned)((F + 127) / 128), 128, 0, st>>>(
        F, nf, etype_dim(face_type), q, N, m->d_xyz, (const int32_t*)(d + o_fc), (const double*)(d + o_w),
        (const double*)(d + o_N), (const double*)(d + o_dN), d_t, d_s3);
    k_face_gather3<<<(unsigned)((nn + 255) / 256), 256, 0, st>>>(nn, (const int32_t*)(d + o_nodes),
                                                                 (const int32_t*)(d + o_ptr),
                                                                 (const int32_t*)(d + o_slots), d_s3, d_f);
  }
  return finish_load(ctx, "loadVector", d_f, N, f_out);
}

namespace {

// Host side of an element set of the mesh: pos[e] = index of element e in
// elems (or -1), after range and duplicate checks; elems == NULL is every
// element in mesh order (pos and list stay empty).
int prepare_elems(const llfem_mesh* m, const int64_t* elems, int64_t ne, const char* who,
                  std::vector<int32_t>* pos, std::vector<int32_t>* list) {
  if (ne < 0 || (elems == nullptr && ne != 0)) return fail(LLFEM_EINVAL, std::string(who) + ": bad element set");
  pos->clear();
  list->clear();
  if (ne == 0 && elems == nullptr) return LLFEM_OK;
  pos->assign((size_t)m->E, -1);
  list->resize((size_t)ne);
  for (int64_t k = 0; k < ne; ++k) {
    const int64_t e = elems[k];
    if (e < 0 || e >= m->E)
      return fail(LLFEM_EINVAL, std::string(who) + ": element index " + std::to_string(e) + " out of range");
    if ((*pos)[e] >= 0)
      return fail(LLFEM_EINVAL, std::string(who) + ": element " + std::to_string(e) + " listed twice");
    (*pos)[e] = (int32_t)k;
    (*list)[k] = (int32_t)e;
  }
  return LLFEM_OK;
}

}  // namespace

extern "C" int llfem_load_body(llfem_mesh* m, int32_t q, const double* weights, const double* N_ref,
                               const double* dN_ref, const int64_t* elems, int64_t ne, const double g[3],
                               const double* g_gp, double* f_out) {
  if (!m || !weights || !N_ref || !dN_ref || !f_out || (!g && !g_gp))
    return fail(LLFEM_EINVAL, "llfem_load_body: NULL argument");
  if (q <= 0) return fail(LLFEM_EINVAL, "llfem_load_body: bad rule size");
  if (etype_dim(m->etype) != 3)
    return fail(LLFEM_EUNSUP, "llfem_load_body: the mesh's elements are not 3D");
  std::vector<int32_t> pos, list;
  LLFEM_TRY(prepare_elems(m, elems, ne, "llfem_load_body", &pos, &list));
  const bool all = elems == nullptr;
  const int64_t nset = all ? m->E : ne;
  llfem_ctx* ctx = m->ctx;
  LLFEM_HIP(hipSetDevice(ctx->device));
  hipStream_t st = ctx->stream;
  const int64_t N = m->N, E = m->E;
  const int npe = m->npe;
  Upload up;
  const size_t o_w = up.add(weights, q), o_N = up.add(N_ref, (size_t)q * npe), o_dN = up.add(dN_ref, (size_t)q * npe * 3),
               o_pos = up.add(pos.data(), pos.size());
  const size_t ngp = g_gp ? 3 * (size_t)nset * q : 0, ns = (g_gp ? 3 : 1) * (size_t)E * npe;
  WsGuard ws(ctx);
  LLFEM_TRY(ws.get(up.bytes() + WsGuard::aligned(8 * ngp) + WsGuard::aligned(8 * ns) +
                   WsGuard::aligned(24 * (size_t)N)));
  char* d = ws.take<char>(up.bytes());
  double *d_gp = ws.take<double>(ngp), *d_s = ws.take<double>(ns), *d_f = ws.take<double>(3 * (size_t)N);
  hipError_t e = up.send(d, st);
  if (ngp) e = e ? e : hipMemcpyAsync(d_gp, g_gp, sizeof(double) * ngp, hipMemcpyHostToDevice, st);
  if (e != hipSuccess) return load_failed("llfem_load_body upload", e);
  const double *d_w = (const double*)(d + o_w), *d_N = (const double*)(d + o_N), *d_dN = (const double*)(d + o_dN);
  const int32_t* d_pos = all ? nullptr : (const int32_t*)(d + o_pos);
  const unsigned ge = (unsigned)((E + 255) / 256), gw = (unsigned)((E + kBodyWaves - 1) / kBodyWaves),
                 gn = (unsigned)((N + 255) / 256);
  const size_t lds = sizeof(double) * kBodyWaves * (3 * (size_t)npe + 64 * 4);
  if (g_gp) {
    k_body_any<true><<<gw, 64 * kBodyWaves, lds, st>>>(E, npe, q, m->d_xyz4, m->d_conn, d_pos, d_w, d_N, d_dN, d_gp, d_s);
    k_body_gather<true><<<gn, 256, 0, st>>>(N, E, m->d_inc_ptr, m->d_inc_elem, m->d_inc_loc, d_pos, d_s, 0.0, 0.0, 0.0,
                                            d_f);
  } else {
    // up to 10 nodes an element's coordinates and sums fit one thread's registers
    switch (npe) {
      case 4: k_body_const<4><<<ge, 256, 0, st>>>(E, q, m->d_xyz4, m->d_conn, d_pos, d_w, d_N, d_dN, d_s); break;
      case 6: k_body_const<6><<<ge, 256, 0, st>>>(E, q, m->d_xyz4, m->d_conn, d_pos, d_w, d_N, d_dN, d_s); break;
      case 8: k_body_const<8><<<ge, 256, 0, st>>>(E, q, m->d_xyz4, m->d_conn, d_pos, d_w, d_N, d_dN, d_s); break;
      case 10: k_body_const<10><<<ge, 256, 0, st>>>(E, q, m->d_xyz4, m->d_conn, d_pos, d_w, d_N, d_dN, d_s); break;
      default:
        k_body_any<false><<<gw, 64 * kBodyWaves, lds, st>>>(E, npe, q, m->d_xyz4, m->d_conn, d_pos, d_w, d_N, d_dN,
                                                           nullptr, d_s);
    }
    k_body_gather<false><<<gn, 256, 0, st>>>(N, E, m->d_inc_ptr, m->d_inc_elem, m->d_inc_loc, d_pos, d_s, g[0], g[1],
                                             g[2], d_f);
  }
  return finish_load(ctx, "llfem_load_body", d_f, N, f_out);
}

extern "C" int llfem_volume_points(llfem_mesh* m, int32_t q, const double* N_ref, const int64_t* elems, int64_t ne,
                                   double* xyz_out) {
  if (!m || !N_ref || !xyz_out) return fail(LLFEM_EINVAL, "llfem_volume_points: NULL argument");
  if (q <= 0) return fail(LLFEM_EINVAL, "llfem_volume_points: bad rule size");
  std::vector<int32_t> pos, list;
  LLFEM_TRY(prepare_elems(m, elems, ne, "llfem_volume_points", &pos, &list));
  const bool all = elems == nullptr;
  const int64_t nset = all ? m->E : ne;
  llfem_ctx* ctx = m->ctx;
  LLFEM_HIP(hipSetDevice(ctx->device));
  hipStream_t st = ctx->stream;
  const int npe = m->npe;
  const size_t npts = (size_t)nset * q;
  Upload up;
  const size_t o_N = up.add(N_ref, (size_t)q * npe), o_list = up.add(list.data(), list.size());
  WsGuard ws(ctx);
  LLFEM_TRY(ws.get(up.bytes() + WsGuard::aligned(24 * npts)));
  char* d = ws.take<char>(up.bytes());
  double* d_out = ws.take<double>(3 * npts);
  hipError_t e = up.send(d, st);
  if (e == hipSuccess && npts > 0) {
    k_volume_points<<<(unsigned)((npts + 255) / 256), 256, 0, st>>>(nset, m->E, npe, q, m->N, m->d_xyz, m->d_conn,
                                                                     all ? nullptr : (const int32_t*)(d + o_list),
                                                                     (const double*)(d + o_N), d_out);
    e = hipGetLastError();
  }
  if (e != hipSuccess) return load_failed("llfem_volume_points", e);
  return copy_to_host(ctx, xyz_out, d_out, 3 * npts);
}

extern "C" int llfem_load_pressure(llfem_mesh* m, int32_t face_type, int32_t nf, const int64_t* face_conn,
                                   int64_t F, int32_t one_based, int32_t q, const double* weights,
                                   const double* N_ref, const double* dN_ref, const double* dN_nodes, double p,
                                   const double* p_nodal, double* f_out) {
  if (!m || !face_conn || !weights || !N_ref || !dN_ref || !dN_nodes || !f_out)
    return fail(LLFEM_EINVAL, "llfem_load_pressure: NULL argument");
  if (etype_dim(face_type) != 2)
    return fail(LLFEM_EINVAL, "loadVector: pressure can be given on a surface of a 3D solid.");
  FacePrep P;
  LLFEM_TRY(prepare_faces(m, face_type, nf, face_conn, F, one_based, q, &P));
  llfem_ctx* ctx = m->ctx;
  LLFEM_HIP(hipSetDevice(ctx->device));
  hipStream_t st = ctx->stream;
  const int64_t N = m->N, nn = (int64_t)P.nodes.size();
  std::vector<int32_t> slot_node((size_t)F * nf);
  for (int64_t i = 0; i < nn; ++i)
    for (int32_t k = P.ptr[i]; k < P.ptr[i + 1]; ++k) slot_node[P.slots[k]] = (int32_t)i;
  Upload up;
  const size_t o_fc = up.add(P.fc.data(), P.fc.size()), o_nodes = up.add(P.nodes.data(), P.nodes.size()),
               o_ptr = up.add(P.ptr.data(), P.ptr.size()), o_slots = up.add(P.slots.data(), P.slots.size()),
               o_sn = up.add(slot_node.data(), slot_node.size()), o_w = up.add(weights, q),
               o_N = up.add(N_ref, (size_t)q * nf), o_dN = up.add(dN_ref, (size_t)q * nf * 3),
               o_dNn = up.add(dN_nodes, (size_t)nf * nf * 3);
  const size_t ns = 3 * (size_t)F * nf, np = p_nodal ? (size_t)N : 0;
  WsGuard ws(ctx);
  LLFEM_TRY(ws.get(up.bytes() + 2 * WsGuard::aligned(8 * ns) + WsGuard::aligned(24 * (size_t)nn) +
                   WsGuard::aligned(8 * np) + WsGuard::aligned(24 * (size_t)N)));
  char* d = ws.take<char>(up.bytes());
  double *d_nrm = ws.take<double>(ns), *d_s3 = ws.take<double>(ns), *d_tn = ws.take<double>(3 * (size_t)nn),
         *d_p = ws.take<double>(np), *d_f = ws.take<double>(3 * (size_t)N);
  hipError_t e = up.send(d, st);
  if (p_nodal) e = e ? e : hipMemcpyAsync(d_p, p_nodal, sizeof(double) * N, hipMemcpyHostToDevice, st);
  e = e ? e : hipMemsetAsync(d_f, 0, sizeof(double) * 3 * N, st);
  if (e != hipSuccess) return load_failed("loadVector upload", e);
  if (F > 0) {
    const int32_t *d_fc = (const int32_t*)(d + o_fc), *d_nodes = (const int32_t*)(d + o_nodes),
                  *d_ptr = (const int32_t*)(d + o_ptr), *d_slots = (const int32_t*)(d + o_slots);
    k_face_node_normals<<<(unsigned)((F * nf + 255) / 256), 256, 0, st>>>(F, nf, N, m->d_xyz, d_fc,
                                                                          (const double*)(d + o_dNn), d_nrm);
    k_pressure_nodal<<<(unsigned)((nn + 255) / 256), 256, 0, st>>>(nn, d_nodes, d_ptr, d_slots, d_nrm, p,
                                                                   p_nodal ? d_p : nullptr, d_tn);
    k_face_integrals_nodal<<<(unsigned)((F + 127) / 128), 128, 0, st>>>(
        F, nf, q, N, m->d_xyz, d_fc, (const double*)(d + o_w), (const double*)(d + o_N), (const double*)(d + o_dN),
        (const int32_t*)(d + o_sn), d_tn, d_s3);
    k_face_gather3<<<(unsigned)((nn + 255) / 256), 256, 0, st>>>(nn, d_nodes, d_ptr, d_slots, d_s3, d_f);
  }
  return finish_load(ctx, "loadVector", d_f, N, f_out);
}
