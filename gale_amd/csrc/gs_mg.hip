// gs_mg.hip -- geometric multigrid for the inner velocity solve.
//
// Because the Q1 spaces of a regular mesh are nested and the coarse basis
// functions are exactly representable on the fine mesh, the Galerkin coarse
// operator P^T K P equals the coarse Q1 operator integrated with the SAME
// material points and weights omega_p = w_p detJ eta_p.  Its element matrix
// depends on the points only through 27 (3D, 23 of them needed) / 9 (2D) weighted moments
// M[a,b,c] = sum_p omega_p r^a s^b t^c (a,b,c <= 2) in element-local
// coordinates, since every entry of B^T D B is a polynomial of degree <= 2 in
// each local coordinate.  The fine moments come from one pass over the
// particles; each coarser level's moments are an exact polynomial change of
// variables of its children's.  Every level is applied matrix-free from its
// moments (184 B per 3D element instead of 32 B per particle), smoothed by
// Chebyshev-Jacobi, and the coarsest level is solved with a dense inverse.
#include "gs_internal.h"
#include "gs_mg.h"
#include "gs_reduce.h"
#include "gs_tile.h"

#include <math.h>

namespace gs {

__device__ __forceinline__ long long xcd_block_mg(long long b, long long nb) {
  const long long q = nb / 8, rem = nb % 8;
  const long long x = b % 8, i = b / 8;
  return x * q + (x < rem ? x : rem) + i;
}

__device__ __forceinline__ double vcoord_mg(const Geo& g, int d, long long idx) {
#pragma clang fp contract(off)
  if (idx <= 0) return g.lo[d];
  if (idx >= g.res[d]) return g.hi[d];
  return g.lo[d] + ((double)idx / (double)g.res[d]) * (g.hi[d] - g.lo[d]);
}

__device__ __forceinline__ void colour_elem_mg(const Geo& g, int c, long long t, long long* ijk) {
  const long long mx = (g.res[0] - (c & 1) + 1) / 2;
  const long long my = g.dim > 1 ? (g.res[1] - ((c >> 1) & 1) + 1) / 2 : 1;
  const long long a = t % mx, rem = t / mx;
  const long long b = rem % my, cc = rem / my;
  ijk[0] = 2 * a + (c & 1);
  ijk[1] = 2 * b + ((c >> 1) & 1);
  ijk[2] = 2 * cc + ((c >> 2) & 1);
}

static inline unsigned gridn(long long n) { return (unsigned)((n + kBlock - 1) / kBlock); }

// ---------------------------------------------------------------------------
// moments
// ---------------------------------------------------------------------------
template <int DIM>
__global__ void k_moments_fine(Geo g, const double4* __restrict__ pk, const int* __restrict__ off,
                               double* __restrict__ M) {
  constexpr int NM = DIM == 2 ? 9 : 27;
  const long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (e >= g.E) return;
  double m[NM];
#pragma unroll
  for (int k = 0; k < NM; k++) m[k] = 0.0;
  for (int p = off[e]; p < off[e + 1]; p++) {
    const double4 q = pk[p];
    const double r[3] = {1.0, q.x, q.x * q.x};
    const double s[3] = {1.0, q.y, q.y * q.y};
    if (DIM == 2) {
#pragma unroll
      for (int b = 0; b < 3; b++)
#pragma unroll
        for (int a = 0; a < 3; a++) m[a + 3 * b] += q.w * r[a] * s[b];
    } else {
      const double t[3] = {1.0, q.z, q.z * q.z};
#pragma unroll
      for (int c = 0; c < 3; c++)
#pragma unroll
        for (int b = 0; b < 3; b++) {
          const double ws = q.w * s[b] * t[c];
#pragma unroll
          for (int a = 0; a < 3; a++) m[a + 3 * b + 9 * c] += ws * r[a];
        }
    }
  }
#pragma unroll
  for (int k = 0; k < NM; k++)
    if (DIM == 2 || mom_slot(k) >= 0) M[mom_index<double>(g, k, e)] = m[k];
}

// Parent moments from children: child local r_f maps to parent r_c = (r_f + sg)/2,
// sg = -1 for the lower child, +1 for the upper.  Per axis r_c^a = T[a][k] r_f^k.
template <int DIM>
__global__ void k_moments_coarsen(Geo gc, Geo gf, const double* __restrict__ Mf, double* __restrict__ Mc) {
  constexpr int NM = DIM == 2 ? 9 : 27;
  const long long E = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (E >= gc.E) return;
  const long long I = E % gc.res[0], J = (E / gc.res[0]) % gc.res[1], K = DIM == 3 ? E / ((long long)gc.res[0] * gc.res[1]) : 0;
  double acc[NM];
#pragma unroll
  for (int k = 0; k < NM; k++) acc[k] = 0.0;
  for (int ch = 0; ch < (DIM == 2 ? 4 : 8); ch++) {
    const int ox = ch & 1, oy = (ch >> 1) & 1, oz = (ch >> 2) & 1;
    const long long e = (2 * I + ox) + (long long)gf.res[0] * ((2 * J + oy) + (long long)gf.res[1] * (2 * K + oz));
    double T[3][3][3];  // T[axis][a][k]
    const double sg[3] = {ox ? 1.0 : -1.0, oy ? 1.0 : -1.0, oz ? 1.0 : -1.0};
    for (int d = 0; d < 3; d++) {
      const double s = sg[d];
      T[d][0][0] = 1.0; T[d][0][1] = 0.0; T[d][0][2] = 0.0;
      T[d][1][0] = 0.5 * s; T[d][1][1] = 0.5; T[d][1][2] = 0.0;
      T[d][2][0] = 0.25; T[d][2][1] = 0.5 * s; T[d][2][2] = 0.25;  // (r+s)^2/4 = (r^2 + 2 s r + 1)/4
    }
    double m[NM];
    for (int k = 0; k < NM; k++) m[k] = DIM == 2 || mom_slot(k) >= 0 ? Mf[mom_index<double>(gf, k, e)] : 0.0;
    if (DIM == 2) {
      for (int b = 0; b < 3; b++)
        for (int a = 0; a < 3; a++) {
          double v = 0.0;
          for (int kb = 0; kb <= b; kb++)
            for (int ka = 0; ka <= a; ka++) v += T[0][a][ka] * T[1][b][kb] * m[ka + 3 * kb];
          acc[a + 3 * b] += v;
        }
    } else {
      for (int c = 0; c < 3; c++)
        for (int b = 0; b < 3; b++)
          for (int a = 0; a < 3; a++) {
            double v = 0.0;
            for (int kc = 0; kc <= c; kc++)
              for (int kb = 0; kb <= b; kb++)
                for (int ka = 0; ka <= a; ka++)
                  v += T[0][a][ka] * T[1][b][kb] * T[2][c][kc] * m[ka + 3 * kb + 9 * kc];
            acc[a + 3 * b + 9 * c] += v;
          }
    }
  }
#pragma unroll
  for (int k = 0; k < NM; k++)
    if (DIM == 2 || mom_slot(k) >= 0) Mc[mom_index<double>(gc, k, E)] = acc[k];
}

void launch_moments_fine(const Geo& g, const double4* pk, const int* off, double* M, hipStream_t st) {
  if (g.dim == 3)
    hipLaunchKernelGGL(k_moments_fine<3>, dim3(gridn(g.E)), dim3(kBlock), 0, st, g, pk, off, M);
  else
    hipLaunchKernelGGL(k_moments_fine<2>, dim3(gridn(g.E)), dim3(kBlock), 0, st, g, pk, off, M);
}
void launch_moments_coarsen(const Geo& gc, const Geo& gf, const double* Mf, double* Mc, hipStream_t st) {
  if (gc.dim == 3)
    hipLaunchKernelGGL(k_moments_coarsen<3>, dim3(gridn(gc.E)), dim3(kBlock), 0, st, gc, gf, Mf, Mc);
  else
    hipLaunchKernelGGL(k_moments_coarsen<2>, dim3(gridn(gc.E)), dim3(kBlock), 0, st, gc, gf, Mf, Mc);
}

template <typename S, typename T>
__global__ void k_convert(const S* __restrict__ a, T* __restrict__ b, long long n) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    b[i] = (T)a[i];
}
// FP32 copy of a level's moments (the two precisions group the moments
// differently in 3D, so the copy goes through the element and moment index).
template <int DIM>
__global__ void k_mom_d2f(Geo g, const double* __restrict__ a, float* __restrict__ b) {
  constexpr int NM = DIM == 2 ? 9 : 27;
  const long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (e >= g.E) return;
#pragma unroll
  for (int k = 0; k < NM; k++)
    if (DIM == 2 || mom_slot(k) >= 0) b[mom_index<float>(g, k, e)] = (float)a[mom_index<double>(g, k, e)];
}
void launch_mom_d2f(const Geo& g, const double* a, float* b, hipStream_t st) {
  if (g.dim == 3)
    hipLaunchKernelGGL(k_mom_d2f<3>, dim3(gridn(g.E)), dim3(kBlock), 0, st, g, a, b);
  else
    hipLaunchKernelGGL(k_mom_d2f<2>, dim3(gridn(g.E)), dim3(kBlock), 0, st, g, a, b);
}

void launch_d2f(const double* a, float* b, long long n, hipStream_t st) {
  if (n > 0) hipLaunchKernelGGL((k_convert<double, float>), dim3(gridn(n) < 8192 ? gridn(n) : 8192), dim3(kBlock), 0, st, a, b, n);
}

template <typename T>
__global__ void k_fill_mg(T* __restrict__ y, long long n, T v) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    y[i] = v;
}

template <>
void launch_mom_apply<double>(const Geo& g, const double* x, double* y, const double* Mom, const uint8_t* bcflag,
                              double* halo, hipStream_t st) {
  tile_apply_moments(g, x, y, halo, Mom, bcflag, st);
}
template <>
void launch_mom_apply<float>(const Geo& g, const float* x, float* y, const float* Mom, const uint8_t* bcflag,
                             float* halo, hipStream_t st) {
  tile_apply_moments32(g, x, y, halo, Mom, bcflag, st);
}

// diag(K) from moments: node a, component d: sum_p omega (|grad N_a|^2 + (dN_a/dx_d)^2).
template <int DIM>
__global__ void k_mom_diag(Geo g, int c, long long mcount, const double* __restrict__ Mom, double* __restrict__ diag) {
  constexpr int NEN = DIM == 2 ? 4 : 8;
  constexpr int NM = DIM == 2 ? 9 : 27;
  const long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (t >= mcount) return;
  long long ijk[3];
  colour_elem_mg(g, c, t, ijk);
  const long long e = ijk[0] + (long long)g.res[0] * (ijk[1] + (long long)g.res[1] * ijk[2]);
  double inv[3];
  for (int d = 0; d < DIM; d++) inv[d] = 2.0 / (vcoord_mg(g, d, ijk[d] + 1) - vcoord_mg(g, d, ijk[d]));
  const double cN = DIM == 2 ? 0.25 : 0.125;
  double M[NM];
  for (int k = 0; k < NM; k++) M[k] = DIM == 2 || mom_slot(k) >= 0 ? Mom[mom_index<double>(g, k, e)] : 0.0;
  const long long sy = g.nn[0], sz = g.nn[0] * g.nn[1];
  const long long n0 = ijk[0] + sy * ijk[1] + sz * ijk[2];
  for (int a = 0; a < NEN; a++) {
    // (dN_a/dx_d)^2 = (cN inv_d)^2 prod_{d' != d} (1 + s_d' x_d')^2 ; (1 + s x)^2 = 1 + 2 s x + x^2
    double sq[3];
    for (int d = 0; d < DIM; d++) {
      double v = 0.0;
      // polynomial coefficients per axis: axis d contributes only degree 0 (coefficient 1)
      double cf[3][3];
      for (int d2 = 0; d2 < 3; d2++) {
        const double s = ((a >> d2) & 1) ? 1.0 : -1.0;
        if (d2 >= DIM || d2 == d) {
          cf[d2][0] = 1.0; cf[d2][1] = 0.0; cf[d2][2] = 0.0;
        } else {
          cf[d2][0] = 1.0; cf[d2][1] = 2.0 * s; cf[d2][2] = 1.0;
        }
      }
      if (DIM == 2) {
        for (int b = 0; b < 3; b++)
          for (int aa = 0; aa < 3; aa++) v += cf[0][aa] * cf[1][b] * M[aa + 3 * b];
      } else {
        for (int cc = 0; cc < 3; cc++)
          for (int b = 0; b < 3; b++)
            for (int aa = 0; aa < 3; aa++) v += cf[0][aa] * cf[1][b] * cf[2][cc] * M[aa + 3 * b + 9 * cc];
      }
      sq[d] = (cN * inv[d]) * (cN * inv[d]) * v;
    }
    double tot = 0.0;
    for (int d = 0; d < DIM; d++) tot += sq[d];
    const long long nd = n0 + (a & 1) + ((a >> 1) & 1) * sy + ((a >> 2) & 1) * sz;
    for (int d = 0; d < DIM; d++) diag[nd * DIM + d] += tot + sq[d];
  }
}

void launch_mom_diag(const Geo& g, const double* Mom, double* diag, hipStream_t st) {
  const long long n = g.N * g.dim;
  unsigned gb = gridn(n);
  if (gb > 8192) gb = 8192;
  hipLaunchKernelGGL(k_fill_mg<double>, dim3(gb), dim3(kBlock), 0, st, diag, n, 0.0);
  const int ncol = g.dim == 2 ? 4 : 8;
  for (int c = 0; c < ncol; c++) {
    const long long m = colour_count(g, c);
    if (m <= 0) continue;
    if (g.dim == 3)
      hipLaunchKernelGGL(k_mom_diag<3>, dim3(gridn(m)), dim3(kBlock), 0, st, g, c, m, Mom, diag);
    else
      hipLaunchKernelGGL(k_mom_diag<2>, dim3(gridn(m)), dim3(kBlock), 0, st, g, c, m, Mom, diag);
  }
}

// ---------------------------------------------------------------------------
// transfers: P = Q1 interpolation coarse -> fine, R = P^T (full weighting)
// ---------------------------------------------------------------------------
// Lattice indices of node n (x fastest); 32-bit division when the node count
// allows it (64-bit division is a long software sequence on the GPU).
__device__ __forceinline__ void node_ijk(const Geo& g, long long n, long long& i, long long& j, long long& k) {
  if (g.N < (1LL << 31)) {
    const unsigned un = (unsigned)n, nx = (unsigned)g.nn[0], ny = (unsigned)g.nn[1];
    const unsigned q = un / nx;
    i = un - q * nx;
    j = q % ny;
    k = q / ny;
  } else {
    i = n % g.nn[0];
    j = (n / g.nn[0]) % g.nn[1];
    k = n / (g.nn[0] * g.nn[1]);
  }
}
// Full-weighting restriction b_C = R r_F on the coarse level (3 x 3 (x 3)
// stencil, weights 1 and 1/2 per axis).  A thread owns a coarse dof and, in
// 3D, one of its three fine node planes, nine loads in flight; the planes'
// sums meet in LDS.  A coarse level is small, so it is bound by the latency of
// the loads one thread has to wait for: 48^3 -> 24^3 in FP64 takes 3.5 us, one
// thread per node walking all 27 nodes took 8.8.
template <typename T, int DIM>
__global__ __launch_bounds__(DIM == 3 ? 192 : 64) void k_restrict(Geo gc, Geo gf, const T* __restrict__ rf,
                                                                  T* __restrict__ bc,
                                                                  const uint8_t* __restrict__ bcflag_c) {
  __shared__ T part[DIM == 3 ? 2 : 1][64];
  const long long nd = gc.N * DIM;
  const long long i = xcd_block_mg(blockIdx.x, gridDim.x) * 64 + threadIdx.x;
  const int pl = DIM == 3 ? (int)threadIdx.y : 0;
  const bool live = i < nd;
  T s = 0;
  unsigned bf = 0;
  int c = 0;
  if (live) {
    const long long n = i / DIM;
    c = (int)(i - n * DIM);
    long long I, J, K;
    node_ijk(gc, n, I, J, K);
    if (pl == 0 && bcflag_c) bf = bcflag_c[n];
    const long long kk = DIM == 3 ? 2 * K + pl - 1 : 0;
    const bool inz = kk >= 0 && kk < gf.nn[2];
    T v[9];
#pragma unroll
    for (int q = 0; q < 9; q++) {
      const long long ii = 2 * I + q % 3 - 1, jj = 2 * J + q / 3 - 1;
      const bool in = inz && ii >= 0 && ii < gf.nn[0] && jj >= 0 && jj < gf.nn[1];
      v[q] = in ? rf[(ii + gf.nn[0] * (jj + gf.nn[1] * kk)) * DIM + c] : (T)0;
    }
#pragma unroll
    for (int q = 0; q < 9; q++) s += (q % 3 == 1 ? (T)1 : (T)0.5) * (q / 3 == 1 ? (T)1 : (T)0.5) * v[q];
    if (DIM == 3 && pl != 1) s *= (T)0.5;
  }
  if (DIM == 3) {
    if (pl > 0) part[pl - 1][threadIdx.x] = s;
    __syncthreads();
    if (pl > 0 || !live) return;
    s += part[0][threadIdx.x];
    s += part[DIM == 3 ? 1 : 0][threadIdx.x];
  } else if (!live) {
    return;
  }
  bc[i] = ((bf >> c) & 1u) ? (T)0 : s;
}

// x_F += P x_C (Q1 interpolation) on the nodes of the fine level: the up to
// 2^dim coarse parents and the fine value are loaded at once.
template <typename T, int DIM>
__global__ void k_prolong_add(Geo gc, Geo gf, const T* __restrict__ xc, T* __restrict__ xf, const uint8_t* __restrict__ bcflag_f) {
  const long long n = xcd_block_mg(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  if (n >= gf.N) return;
  long long i, j, k;
  node_ijk(gf, n, i, j, k);
  const int nz = (DIM == 3 && (k & 1)) ? 2 : 1, ny = (j & 1) ? 2 : 1, nx = (i & 1) ? 2 : 1;
  const T wz = nz == 2 ? (T)0.5 : (T)1, wy = ny == 2 ? (T)0.5 : (T)1, wx = nx == 2 ? (T)0.5 : (T)1;
  constexpr int NA = DIM == 3 ? 2 : 1;
  T v[NA][2][2][DIM];
  T xv[DIM];
  const unsigned bf = bcflag_f ? bcflag_f[n] : 0u;
#pragma unroll
  for (int d = 0; d < DIM; d++) xv[d] = xf[n * DIM + d];
#pragma unroll
  for (int a = 0; a < NA; a++)
#pragma unroll
    for (int b = 0; b < 2; b++)
#pragma unroll
      for (int cc = 0; cc < 2; cc++) {
        const bool in = a < nz && b < ny && cc < nx;
        const long long K = DIM == 3 ? (k >> 1) + a : 0, J = (j >> 1) + b, I = (i >> 1) + cc;
        const long long cn = in ? I + gc.nn[0] * (J + gc.nn[1] * K) : 0;
#pragma unroll
        for (int d = 0; d < DIM; d++) v[a][b][cc][d] = in ? xc[cn * DIM + d] : (T)0;
      }
  T acc[DIM];
#pragma unroll
  for (int d = 0; d < DIM; d++) acc[d] = 0;
#pragma unroll
  for (int a = 0; a < NA; a++)
#pragma unroll
    for (int b = 0; b < 2; b++)
#pragma unroll
      for (int cc = 0; cc < 2; cc++)
#pragma unroll
        for (int d = 0; d < DIM; d++) acc[d] += wx * wy * wz * v[a][b][cc][d];
#pragma unroll
  for (int d = 0; d < DIM; d++)
    if (!((bf >> d) & 1u)) xf[n * DIM + d] = xv[d] + acc[d];
}

template <typename T>
void launch_restrict(const Geo& gc, const Geo& gf, const T* rf, T* bc, const uint8_t* bcflag_c, hipStream_t st) {
  const dim3 nb((unsigned)((gc.N * gc.dim + 63) / 64));
  if (gc.dim == 3)
    hipLaunchKernelGGL((k_restrict<T, 3>), nb, dim3(64, 3), 0, st, gc, gf, rf, bc, bcflag_c);
  else
    hipLaunchKernelGGL((k_restrict<T, 2>), nb, dim3(64), 0, st, gc, gf, rf, bc, bcflag_c);
}
template <typename T>
void launch_prolong_add(const Geo& gc, const Geo& gf, const T* xc, T* xf, const uint8_t* bcflag_f, hipStream_t st) {
  if (gf.dim == 3)
    hipLaunchKernelGGL((k_prolong_add<T, 3>), dim3(gridn(gf.N)), dim3(kBlock), 0, st, gc, gf, xc, xf, bcflag_f);
  else
    hipLaunchKernelGGL((k_prolong_add<T, 2>), dim3(gridn(gf.N)), dim3(kBlock), 0, st, gc, gf, xc, xf, bcflag_f);
}
template void launch_restrict<double>(const Geo&, const Geo&, const double*, double*, const uint8_t*, hipStream_t);
template void launch_restrict<float>(const Geo&, const Geo&, const float*, float*, const uint8_t*, hipStream_t);
template void launch_prolong_add<double>(const Geo&, const Geo&, const double*, double*, const uint8_t*, hipStream_t);
template void launch_prolong_add<float>(const Geo&, const Geo&, const float*, float*, const uint8_t*, hipStream_t);

// ---------------------------------------------------------------------------
// Chebyshev-Jacobi step: r = b - Ax ; d = alpha d + beta Dinv r ; x += d
// (with x == 0 on entry, "first" uses Ax = 0 and skips reading x / Ax).
// ---------------------------------------------------------------------------
template <typename T>
__global__ void k_cheb(const T* __restrict__ b, const T* __restrict__ Ax, const T* __restrict__ dinv, T* __restrict__ d,
                       T* __restrict__ x, long long n, T alpha, T beta, int first) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
    const T r = first ? b[i] : b[i] - Ax[i];
    const T di = (first ? (T)0 : alpha * d[i]) + beta * dinv[i] * r;
    d[i] = di;
    x[i] = first ? di : x[i] + di;
  }
}
template <typename T>
void launch_cheb(const T* b, const T* Ax, const T* dinv, T* d, T* x, long long n, T alpha, T beta, int first, hipStream_t st) {
  unsigned gb = gridn(n);
  if (gb > 8192) gb = 8192;
  hipLaunchKernelGGL(k_cheb<T>, dim3(gb), dim3(kBlock), 0, st, b, Ax, dinv, d, x, n, alpha, beta, first);
}
template void launch_cheb<double>(const double*, const double*, const double*, double*, double*, long long, double, double, int, hipStream_t);
template void launch_cheb<float>(const float*, const float*, const float*, float*, float*, long long, float, float, int, hipStream_t);

// ---------------------------------------------------------------------------
// Assembled levels
// ---------------------------------------------------------------------------
// A small level is bound by latency, not by bytes: the tiled apply runs 54
// workgroups on 24^3 and needs a second launch for the tile faces.  Here a
// thread owns a row and, in 3D, one of the three node planes (64 x 3 threads;
// the planes' sums meet in LDS), all of its 27 (2D: 18) coefficients and
// neighbour values loaded at once, and the update follows in the same launch.
// At 24^3 in FP64 a smoothing step takes 5 us (apply + face completion: 15),
// reading 30 MB of coefficients from L2 in the place of 3 MB of moments.
template <typename T, int DIM, int KIND, bool X0>
__global__ __launch_bounds__(DIM == 3 ? 192 : 64) void k_stencil_epi(Geo g, const T* __restrict__ A,
                                                                     const T* __restrict__ x, TileEpi<T> ep) {
  constexpr int NB = 9;
  __shared__ T part[DIM == 3 ? 2 : 1][64];
  const long long nd = g.N * DIM;
  // rows of an XCD's blocks are contiguous, so its L2 keeps their coefficients
  const long long i = xcd_block_mg(blockIdx.x, gridDim.x) * 64 + threadIdx.x;
  const int pl = DIM == 3 ? (int)threadIdx.y : 0;
  const bool live = i < nd;
  T s = 0, bi = 0, di0 = 0, xv = 0, dv = 0;
  if (live) {
    const unsigned n = (unsigned)(i / DIM);
    const unsigned nx = (unsigned)g.nn[0], ny = (unsigned)g.nn[1], q = n / nx;
    const int li = (int)(n - q * nx), lj = (int)(q % ny), lk = (int)(q / ny);
    if (pl == 0) {  // the row's own values travel with the coefficients
      bi = ep.b[i];
      if (KIND == 1 || X0) di0 = ep.dinv[i];
      if (!X0 && KIND == 1) {
        xv = x[i];
        if (ep.alpha != 0) dv = ep.d[i];  // a first step does not read d: its buffer may hold anything
      }
    }
    const int kz = DIM == 3 ? lk + pl - 1 : 0;
    const bool inz = DIM == 3 ? kz >= 0 && kz < (int)g.nn[2] : true;
    T c[NB][DIM], v[NB][DIM];
#pragma unroll
    for (int k = 0; k < NB; k++) {
      const int ii = li + k % 3 - 1, jj = lj + k / 3 - 1;
      const bool in = inz && ii >= 0 && ii < (int)nx && jj >= 0 && jj < (int)ny;
      // outside the grid the coefficients are zero: read the row's own node
      const long long m = in ? ii + (long long)nx * (jj + (long long)ny * kz) : (long long)n;
#pragma unroll
      for (int d = 0; d < DIM; d++) {
        c[k][d] = A[((long long)(pl * NB + k) * DIM + d) * nd + i];
        v[k][d] = X0 ? ep.beta0 * ep.dinv[m * DIM + d] * ep.b[m * DIM + d] : x[m * DIM + d];
      }
    }
#pragma unroll
    for (int k = 0; k < NB; k++)
#pragma unroll
      for (int d = 0; d < DIM; d++) s += c[k][d] * v[k][d];
  }
  if (DIM == 3) {
    if (pl > 0) part[pl - 1][threadIdx.x] = s;
    __syncthreads();
    if (pl > 0 || !live) return;
    s += part[0][threadIdx.x];
    s += part[DIM == 3 ? 1 : 0][threadIdx.x];
  } else if (!live) {
    return;
  }
  if (X0) xv = ep.beta0 * di0 * bi;
  if (KIND == 1) {
    const T di = ep.alpha * (X0 ? xv : dv) + ep.beta * di0 * (bi - s);
    ep.d[i] = di;
    ep.xout[i] = xv + di;
  } else {
    ep.r[i] = bi - s;
    if (X0) ep.xout[i] = xv;
  }
}

template <typename T, int DIM>
static void stencil_epi(const Geo& g, const T* A, const T* x, const TileEpi<T>& ep, hipStream_t st) {
  const dim3 nb((unsigned)((g.N * DIM + 63) / 64)), bl(64, DIM == 3 ? 3 : 1);
  if (ep.kind == 1) {
    if (x)
      hipLaunchKernelGGL((k_stencil_epi<T, DIM, 1, false>), nb, bl, 0, st, g, A, x, ep);
    else
      hipLaunchKernelGGL((k_stencil_epi<T, DIM, 1, true>), nb, bl, 0, st, g, A, x, ep);
  } else {
    if (x)
      hipLaunchKernelGGL((k_stencil_epi<T, DIM, 2, false>), nb, bl, 0, st, g, A, x, ep);
    else
      hipLaunchKernelGGL((k_stencil_epi<T, DIM, 2, true>), nb, bl, 0, st, g, A, x, ep);
  }
}
template <typename T>
void launch_stencil_epi(const Geo& g, const T* A, const T* x, const TileEpi<T>& ep, hipStream_t st) {
  if (g.dim == 3)
    stencil_epi<T, 3>(g, A, x, ep, st);
  else
    stencil_epi<T, 2>(g, A, x, ep, st);
}
template void launch_stencil_epi<double>(const Geo&, const double*, const double*, const TileEpi<double>&, hipStream_t);
template void launch_stencil_epi<float>(const Geo&, const float*, const float*, const TileEpi<float>&, hipStream_t);

// Dense coarse solve: x[free[i]] = sum_j Kinv[i][j] b[free[j]], zero on the
// Dirichlet dofs.  16 rows per 1024-thread workgroup, one wavefront per row;
// the gathered right-hand side b[free[j]] is read once per workgroup into
// LDS, and each row is read with 16-byte loads (rows padded to ld, so every
// row starts 16-byte aligned).
template <typename T>
__global__ __launch_bounds__(1024) void k_dense_solve_wide(const T* __restrict__ Kinv, int ld,
                                                           const int* __restrict__ freeidx,
                                                           const int* __restrict__ pos, int nf,
                                                           const T* __restrict__ b, T* __restrict__ x, long long n) {
  constexpr int E = 16 / (int)sizeof(T);
  typedef T vec_t __attribute__((ext_vector_type(E)));
  __shared__ __align__(16) T sb[kDenseWideMax];
  const int row = blockIdx.x * (blockDim.x / 64) + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const bool live = row < nf;
  const vec_t* r = reinterpret_cast<const vec_t*>(Kinv + (long long)(live ? row : 0) * ld);
  // the row's first segment is requested before the right-hand side is
  // staged, and each later one while the previous one is being used (the
  // products and their order are unchanged)
  vec_t vn = {};
  if (live && lane * E < nf) vn = r[lane];
  for (int j = threadIdx.x; j < nf; j += blockDim.x) sb[j] = b[freeidx[j]];
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    if (pos[i] < 0) x[i] = 0;
  __syncthreads();
  if (!live) return;
  T s = 0;
  for (int j0 = lane * E; j0 < nf; j0 += 64 * E) {
    const vec_t v = vn;
    if (j0 + 64 * E < nf) vn = r[(j0 + 64 * E) / E];
#pragma unroll
    for (int e = 0; e < E; e++)
      if (j0 + e < nf) s += v[e] * sb[j0 + e];
  }
  for (int o = 32; o > 0; o >>= 1) s += __shfl_down(s, o, 64);
  if (lane == 0) x[freeidx[row]] = s;
}

// Kinv is symmetric, so a solve can read half of it: a wave takes one 64 x 64
// tile (i, j), j <= i, of the lower triangle and adds both its row sums
// (A x_j) and its column sums (A^T x_i).  Lane l holds the rows l / 8 + 8 k
// and 64 / 8 columns of them, all 16-byte loads of a wave's tile in flight
// together, and a sum goes over eight lanes only.  Slot s of P (nb slots of
// ld values) holds what tile (s, .) or (., s) adds to a row, so every value is
// written once and k_dense_sym_sum adds the slots in order.
template <typename T, int M>
__device__ __forceinline__ T sum8(T (&v)[8], int lane) {
  // on return: the sum over the lanes that differ in bits M, 2M, 4M of v[i],
  // i the three bits (4M: 4, 2M: 2, M: 1) of this lane
#pragma unroll
  for (int h = 4; h > 0; h >>= 1) {
    const bool up = (lane & (h * M)) != 0;
#pragma unroll
    for (int a = 0; a < h; a++) {
      const T send = up ? v[a] : v[a + h], keep = up ? v[a + h] : v[a];
      v[a] = keep + __shfl_xor(send, h * M, 64);
    }
  }
  return v[0];
}
template <typename T>
__global__ __launch_bounds__(256) void k_dense_sym(const T* __restrict__ Kinv, int ld, int ntile,
                                                   const int* __restrict__ freeidx, int nf, const T* __restrict__ b,
                                                   T* __restrict__ P) {
  constexpr int E = 16 / (int)sizeof(T), Q = 64 / (8 * E);
  typedef T vec_t __attribute__((ext_vector_type(E)));
  __shared__ T sx[4][128];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int t = blockIdx.x * 4 + w;
  const bool live = t < ntile;
  int i = (int)((sqrt(8.0 * (double)t + 1.0) - 1.0) * 0.5);
  while ((i + 1) * (i + 2) / 2 <= t) i++;
  while (i * (i + 1) / 2 > t) i--;
  const int j = t - i * (i + 1) / 2;
  const int lr = lane >> 3, lc = lane & 7;
  vec_t v[8][Q];
  if (live) {
    const T* base = Kinv + ((long long)i * 64 + lr) * ld + j * 64 + lc * E;
#pragma unroll
    for (int k = 0; k < 8; k++)
#pragma unroll
      for (int q = 0; q < Q; q++) v[k][q] = *reinterpret_cast<const vec_t*>(base + (long long)8 * k * ld + q * 8 * E);
    const int r = i * 64 + lane, c = j * 64 + lane;
    sx[w][lane] = r < nf ? b[freeidx[r]] : T(0);
    sx[w][64 + lane] = c < nf ? b[freeidx[c]] : T(0);
  }
  __syncthreads();
  if (!live) return;
  T rs[8], cs[8];
#pragma unroll
  for (int k = 0; k < 8; k++) rs[k] = cs[k] = 0;
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const T xr = sx[w][8 * k + lr];
#pragma unroll
    for (int q = 0; q < Q; q++)
#pragma unroll
      for (int e = 0; e < E; e++) {
        rs[k] += v[k][q][e] * sx[w][64 + (q * 8 + lc) * E + e];
        cs[q * E + e] += v[k][q][e] * xr;
      }
  }
  const T rsum = sum8<T, 1>(rs, lane), csum = sum8<T, 8>(cs, lane);
  P[(long long)j * ld + i * 64 + 8 * lc + lr] = rsum;
  if (i != j) P[(long long)i * ld + j * 64 + (lr / E * 8 + lc) * E + lr % E] = csum;
}
template <typename T>
__global__ __launch_bounds__(256) void k_dense_sym_sum(const T* __restrict__ P, int ld, const int* __restrict__ freeidx,
                                                       const int* __restrict__ pos, int nf, T* __restrict__ x,
                                                       long long n) {
  __shared__ T part[8][32];
  const int c = threadIdx.x & 31, g = threadIdx.x >> 5, nb = ld / 64;
  const int e = blockIdx.x * 32 + c;
  T s = 0;
#pragma unroll 8
  for (int k = g; k < nb; k += 8) s += P[(long long)k * ld + e];
  part[g][c] = s;
  for (long long q = blockIdx.x * 256LL + threadIdx.x; q < n; q += (long long)gridDim.x * 256)
    if (pos[q] < 0) x[q] = 0;
  __syncthreads();
  if (g == 0 && e < nf) {
#pragma unroll
    for (int k = 1; k < 8; k++) s += part[k][c];
    x[freeidx[e]] = s;
  }
}

template <typename T>
void launch_dense_solve(const T* Kinv, const int* freeidx, const int* pos, int nf, int ld, double* work, const T* b,
                        T* x, long long n, hipStream_t st) {
  if ((long long)nf * nf * (long long)sizeof(T) >= kDenseSymBytes) {
    const int nb = ld / 64, ntile = nb * (nb + 1) / 2;
    T* P = reinterpret_cast<T*>(work);
    hipLaunchKernelGGL(k_dense_sym<T>, dim3((ntile + 3) / 4), dim3(256), 0, st, Kinv, ld, ntile, freeidx, nf, b, P);
    hipLaunchKernelGGL(k_dense_sym_sum<T>, dim3(ld / 32), dim3(256), 0, st, P, ld, freeidx, pos, nf, x, n);
    return;
  }
  hipLaunchKernelGGL(k_dense_solve_wide<T>, dim3(nf > 0 ? (nf + 15) / 16 : 1), dim3(1024), 0, st, Kinv, ld, freeidx,
                     pos, nf, b, x, n);
}
template void launch_dense_solve<double>(const double*, const int*, const int*, int, int, double*, const double*,
                                         double*, long long, hipStream_t);
template void launch_dense_solve<float>(const float*, const int*, const int*, int, int, double*, const float*, float*,
                                        long long, hipStream_t);

// Power iteration on D^-1 K: x = 1 on the free dofs, then per step
// d = D^-1 (K x), lambda = |d| / |x|, x = d / |d|.  st4 = {lambda, 1 / |d|,
// stopped}; a step whose norms are zero or not finite stops the iteration
// with the last lambda.
__global__ void k_pow_init(double* __restrict__ x, const uint8_t* __restrict__ bc, long long n, double* st4) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    x[i] = bc[i] ? 0.0 : 1.0;
  if (blockIdx.x == 0 && threadIdx.x == 0) st4[0] = 1.0;
}
__global__ void k_pow_dots(const double* __restrict__ x, const double* __restrict__ Ax,
                           const double* __restrict__ dinv, double* __restrict__ d, long long n, Reducer rd) {
  double v[2] = {0.0, 0.0};
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
    const double di = dinv[i] * Ax[i], xi = x[i];
    d[i] = di;
    v[0] += di * di;
    v[1] += xi * xi;
  }
  block_partials<2, false>(v, rd);
}
struct OpPow {
  double* st4;
  __device__ void operator()(const double* t) const {
    if (st4[2] != 0.0) return;
    const double dn = sqrt(t[0]), xn = sqrt(t[1]);
    if (!(xn > 0) || !isfinite(dn)) {
      st4[2] = 1.0;
      return;
    }
    st4[0] = dn / xn;
    st4[1] = 1.0 / dn;
  }
};
__global__ void k_pow_scale(double* __restrict__ x, const double* __restrict__ d, long long n, const double* st4) {
  const double sc = st4[1];
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    x[i] = sc * d[i];
}
void launch_pow_init(double* x, const uint8_t* bc, long long n, double* st4, hipStream_t st) {
  hipLaunchKernelGGL(k_pow_init, dim3(grid_for(n)), dim3(kBlock), 0, st, x, bc, n, st4);
}
void launch_pow_step(double* x, const double* Ax, const double* dinv, double* d, long long n, double* st4, Reducer rd,
                     hipStream_t st) {
  const int nb = reduce_grid(n);
  hipLaunchKernelGGL(k_pow_dots, dim3(nb), dim3(kBlock), 0, st, x, Ax, dinv, d, n, rd);
  reduce_finish<2, false>(rd, nb, OpPow{st4}, st);
  hipLaunchKernelGGL(k_pow_scale, dim3(grid_for(n)), dim3(kBlock), 0, st, x, d, n, st4);
}

}  // namespace gs
