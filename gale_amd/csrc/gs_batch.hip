// gs_batch.hip -- batched solve of many independent 2D Stokes instances in one
// persistent launch (include/gale_batch.h).
//
// Each workgroup takes instances from a queue (largest first) and runs the
// complete reference Uzawa loop for it with workgroup barriers only:
//   K apply     from the instance's assembled 9-point stencil (2x2 blocks,
//               symmetric half: centre and four forward neighbours), one
//               thread per node gathering from its neighbours, so an apply
//               needs one barrier and its consumer (Chebyshev step, residual,
//               dot product) runs in the same pass;
//   G, G^T      closed-form Q1-P0 gradient / divergence (node gather,
//               element loop), as the single-problem kernels;
//   inner solve FP64 flexible CG on K v = b, preconditioned by one FP32
//               geometric multigrid V-cycle per iteration (the instance's
//               Galerkin levels, Chebyshev-Jacobi smoothing, dense coarsest
//               solve), all FP32 K applies;
//   outer loop  Stokes_SLE_UzawaSolver.cxx:553-837 (diagonal Q, the same
//               residual, stopping rule and firewalls), FP64.
// One workgroup per instance is bound by the latency of its passes, so what
// counts is the number of barriers per inner iteration: an apply that
// scattered element forces tile by tile took seven per tile.  One inner
// iteration of a 48^2 instance takes 75 us (186 us with the tiles, at 1024
// threads); the stencils are read from L2 at what one compute unit gets.
#include <hip/hip_runtime.h>
#include <string.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <vector>

#include "../../include/gale_batch.h"
#include "gs_internal.h"
#include "gs_mg.h"
#include "gs_reduce.h"

namespace gs {
struct BatchLevelInfo {
  int nx, ny;
  double lmax;
};
void batch_mark(gs_solver* s);
int32_t batch_mg_info(gs_solver* s, int* nlev, BatchLevelInfo* lv, int max_levels, int* nfc);
int32_t batch_copy_fine(gs_solver* s, double* f, double* dinv, double* Qinv, hipStream_t st);
int32_t batch_copy_level(gs_solver* s, int l, float* dinv32, uint8_t* bcflag, hipStream_t st);
void batch_moments(gs_solver* s, int l, const double** M64, const float** M32);
int32_t batch_copy_dense(gs_solver* s, float* Kinv32, int* freeidx, hipStream_t st);
}  // namespace gs

using namespace gs;

#define BCK(x)                                                                                               \
  do {                                                                                                       \
    hipError_t e_ = (x);                                                                                     \
    if (e_ != hipSuccess) {                                                                                  \
      std::fprintf(stderr, "gale_stokes(batch): HIP error %s at %s:%d\n", hipGetErrorString(e_), __FILE__, \
                   __LINE__);                                                                                \
      return GS_E_HIP;                                                                                       \
    }                                                                                                        \
  } while (0)

namespace {

struct BInst {
  int nx, ny;
  long long node_off, elem_off;
  double hx, hy;
  int lev0, nlev, nfc;  // levels [lev0, lev0 + nlev) in the level table; dense coarsest size (<= 0: none)
  long long kinv_off, free_off;
};

struct BLevel {
  int nx, ny;
  long long node_off;  // into the flat level arrays
  double hx, hy, lmax;
};

struct BArgs {
  const BInst* inst;
  const BLevel* lev;
  const float4* LS;      // FP32 stencils of every level (kStencil per node)
  const double4* FS;     // FP64 stencils of the instances
  const float* Ldinv;    // FP32 masked inverse diagonal of every level
  const uint8_t* Lbc;    // node flags of every level
  float *Lb, *Lx, *Lx2, *Lr, *Ld;  // level work vectors (x ping-pongs between Lx and Lx2)
  const float* Kinv;     // dense coarsest inverses
  const int* freeidx;
  const int* order;  // queue order (largest first)
  int B;
  const double* f;
  const double* dinv;
  const double* Qinv;
  const uint8_t* bc;
  double *u, *vstar, *ft, *cr, *cp, *cAp;
  double *p, *r, *s, *q, *z;
  int* status;
  unsigned long long* itime;  // per instance: device wall-clock ticks of its solve
  int* outer;
  long long* inner;
  double* relres;
  unsigned* queue;
  double *fs, *fq;   // relaxed loop: per-instance rings of window directions and their Schur images
  // parameters
  double tol, irt;
  int max_outer, max_inner, nu;
  double relax;      // > 0: relaxed inner tolerance with a truncated flexible outer loop (0: reference loop)
  int window;        // directions of the flexible outer loop
};
constexpr int kBatchMaxWin = 16;

// The thread's index, opaque to the compiler: each pass over an instance works
// out its own addresses instead of the whole solve's being hoisted in front
// of the iteration loops, where they need more registers than there are.
__device__ __forceinline__ int tid() {
  int t = threadIdx.x;
  asm volatile("" : "+v"(t));
  return t;
}

// Block sums of NV values at once (sh: NV * BS / 64 doubles).
template <int BS, int NV>
__device__ __forceinline__ void block_sums(double (&v)[NV], double* sh) {
#pragma unroll
  for (int k = 0; k < NV; k++) v[k] = wave_sum(v[k]);
  __syncthreads();
  if ((threadIdx.x & 63) == 0)
#pragma unroll
    for (int k = 0; k < NV; k++) sh[k * (BS / 64) + (threadIdx.x >> 6)] = v[k];
  __syncthreads();
  if (NV > 2) {  // one thread per sum: all threads adding all of them would hold NV * BS / 64 values each
    if (threadIdx.x < NV) {
      double t = 0.0;
#pragma unroll
      for (int i = 0; i < BS / 64; i++) t += sh[threadIdx.x * (BS / 64) + i];
      sh[threadIdx.x * (BS / 64)] = t;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NV; k++) v[k] = sh[k * (BS / 64)];
  } else {
#pragma unroll
    for (int k = 0; k < NV; k++) {
      double t = 0.0;
#pragma unroll
      for (int i = 0; i < BS / 64; i++) t += sh[k * (BS / 64) + i];
      v[k] = t;
    }
  }
}
template <int BS>
__device__ __forceinline__ double block_sum(double v, double* sh) {
  double a[1] = {v};
  block_sums<BS, 1>(a, sh);
  return a[0];
}

// Nodal forces of one Q1 element from its 4 nodal velocities and 9 particle
// moments (moment form of the per-particle integration, see gs_tile.hip).
template <typename T>
__device__ __forceinline__ void forces2(const T (&u)[4][2], T ix, T iy, const T (&M)[9], T (&ye)[4][2]) {
  T A[2][2], Bm[2][2];
#pragma unroll
  for (int cc = 0; cc < 2; cc++) {
    const T u0 = u[0][cc], u1 = u[1][cc], u2 = u[2][cc], u3 = u[3][cc];
    const T t1 = (u1 - u0) + (u3 - u2), t2 = (u2 + u3) - (u0 + u1), t3 = (u3 - u2) - (u1 - u0);
    A[cc][0] = ix * t1;
    A[cc][1] = ix * t3;
    Bm[cc][0] = iy * t2;
    Bm[cc][1] = iy * t3;
  }
  const T mxx0 = 2 * (A[0][0] * M[0] + A[0][1] * M[3]);
  const T mxxs = 2 * (A[0][0] * M[3] + A[0][1] * M[6]);
  const T myy0 = 2 * (Bm[1][0] * M[0] + Bm[1][1] * M[1]);
  const T myyr = 2 * (Bm[1][0] * M[1] + Bm[1][1] * M[2]);
  const T txy0 = Bm[0][0] * M[0] + Bm[0][1] * M[1] + A[1][0] * M[0] + A[1][1] * M[3];
  const T txyr = Bm[0][0] * M[1] + Bm[0][1] * M[2] + A[1][0] * M[1] + A[1][1] * M[4];
  const T txys = Bm[0][0] * M[3] + Bm[0][1] * M[4] + A[1][0] * M[3] + A[1][1] * M[6];
#pragma unroll
  for (int a = 0; a < 4; a++) {
    const T ax = (a & 1) ? (T)1 : (T)-1, ay = (a & 2) ? (T)1 : (T)-1;
    ye[a][0] = ix * ax * (mxx0 + ay * mxxs) + iy * ay * (txy0 + ax * txyr);
    ye[a][1] = iy * ay * (myy0 + ax * myyr) + ix * ax * (txy0 + ay * txys);
  }
}

// ---- assembled stencils ----
// Block k of node n couples it to node n + offset k: the node itself, east,
// north-west, north and north-east; the other four are the transposes of the
// neighbours' blocks (K is symmetric).  Rows and columns of Dirichlet dofs
// are zero, and so are blocks towards nodes outside the grid.  S[k * N + n] =
// {xx, xy, yx, yy}: a thread per node reads 16-byte (FP64: 32-byte) entries,
// neighbouring threads neighbouring entries.
constexpr int kStencil = 5;
__device__ __forceinline__ int st_di(int k) { return k == 0 || k == 3 ? 0 : (k == 2 ? -1 : 1); }
__device__ __forceinline__ int st_dj(int k) { return k >= 2 ? 1 : 0; }

template <typename T>
struct T4;
template <>
struct T4<double> {
  using type = double4;
  using pair = double2;
};
template <>
struct T4<float> {
  using type = float4;
  using pair = float2;
};

// Assembles the stencil of an nx x ny grid from its 9 element moments.
template <typename T>
__global__ void k_stencil(int nx, int ny, T ix, T iy, const T* __restrict__ Mom, const uint8_t* __restrict__ bc,
                          typename T4<T>::type* __restrict__ S) {
  const long long N = (long long)(nx + 1) * (ny + 1), E = (long long)nx * ny;
  const long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (t >= N * kStencil) return;
  const int k = (int)(t / N);
  const long long n = t - k * N;
  const int i = (int)(n % (nx + 1)), j = (int)(n / (nx + 1));
  const int i2 = i + st_di(k), j2 = j + st_dj(k);
  T v[2][2] = {{0, 0}, {0, 0}};
  if (i2 >= 0 && i2 <= nx && j2 <= ny) {
    // elements that hold both nodes, row by row
    for (int ej = max(max(j, j2) - 1, 0); ej <= min(min(j, j2), ny - 1); ej++)
      for (int ei = max(max(i, i2) - 1, 0); ei <= min(min(i, i2), nx - 1); ei++) {
        const long long e = ei + (long long)nx * ej;
        const int a = (i - ei) + 2 * (j - ej), b = (i2 - ei) + 2 * (j2 - ej);
        T M[9];
        for (int m = 0; m < 9; m++) M[m] = Mom[m * E + e];
#pragma unroll
        for (int d = 0; d < 2; d++) {
          T u[4][2], ye[4][2];
#pragma unroll
          for (int q = 0; q < 4; q++)
#pragma unroll
            for (int c = 0; c < 2; c++) u[q][c] = q == b && c == d ? (T)1 : (T)0;
          forces2(u, ix, iy, M, ye);
#pragma unroll
          for (int q = 0; q < 4; q++)
            if (q == a) {
              v[0][d] += ye[q][0];
              v[1][d] += ye[q][1];
            }
        }
      }
    const unsigned m1 = bc[n], m2 = bc[i2 + (long long)(nx + 1) * j2];
#pragma unroll
    for (int c = 0; c < 2; c++)
#pragma unroll
      for (int d = 0; d < 2; d++)
        if (((m1 >> c) & 1u) || ((m2 >> d) & 1u)) v[c][d] = 0;
  }
  typename T4<T>::type o;
  o.x = v[0][0];
  o.y = v[0][1];
  o.z = v[1][0];
  o.w = v[1][1];
  S[t] = o;
}

// (K x) of node n = (i, j); w = nodes per row, h = rows, N = w * h.
template <typename T>
__device__ __forceinline__ void st_row(const typename T4<T>::type* __restrict__ S, int w, int h, int N, int n, int i,
                                       int j, const T* __restrict__ x, T& y0, T& y1) {
  typedef typename T4<T>::type V4;
  typedef typename T4<T>::pair V2;
  const V2* x2 = reinterpret_cast<const V2*>(x);
  // A neighbour outside the grid reads the node itself, with a zero block.
  // The loads go in two groups (own blocks with the forward neighbours, then
  // the neighbours' blocks with the backward ones): all 18 of them in flight
  // would take 110 registers in FP64.
  T a0, a1;
  {
    V4 c[kStencil];
    V2 xf[4];
    const V2 xc = x2[n];
#pragma unroll
    for (int k = 0; k < kStencil; k++) c[k] = S[(long long)k * N + n];
#pragma unroll
    for (int k = 1; k < kStencil; k++) {
      const int off = st_di(k) + w * st_dj(k);
      const bool fwd = i + st_di(k) >= 0 && i + st_di(k) < w && j + st_dj(k) < h;
      xf[k - 1] = x2[fwd ? n + off : n];
    }
    a0 = c[0].x * xc.x + c[0].y * xc.y;
    a1 = c[0].z * xc.x + c[0].w * xc.y;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      a0 += c[k + 1].x * xf[k].x + c[k + 1].y * xf[k].y;
      a1 += c[k + 1].z * xf[k].x + c[k + 1].w * xf[k].y;
    }
  }
  if (sizeof(T) == 8) __builtin_amdgcn_sched_barrier(0);
  {
    V4 tr[4];
    V2 xb[4];
#pragma unroll
    for (int k = 1; k < kStencil; k++) {
      const int off = st_di(k) + w * st_dj(k);
      const bool bwd = i - st_di(k) >= 0 && i - st_di(k) < w && j - st_dj(k) >= 0;
      xb[k - 1] = x2[bwd ? n - off : n];
      V4 t = S[(long long)k * N + (bwd ? n - off : n)];
      if (!bwd) {
        t.x = 0; t.y = 0; t.z = 0; t.w = 0;
      }
      tr[k - 1] = t;
    }
#pragma unroll
    for (int k = 0; k < 4; k++) {
      a0 += tr[k].x * xb[k].x + tr[k].z * xb[k].y;
      a1 += tr[k].y * xb[k].x + tr[k].w * xb[k].y;
    }
  }
  y0 = a0;
  y1 = a1;
}

// y = G p (masked), node gather with the closed-form element gradient.
template <int BS>
__device__ void bapply_G(const BInst& I, const double* __restrict__ p, double* __restrict__ y,
                         const uint8_t* __restrict__ bc) {
  const int nx = I.nx, ny = I.ny, nnx = nx + 1;
  const long long N = (long long)(nx + 1) * (ny + 1);
  for (long long n = tid(); n < N; n += BS) {
    const int i = (int)(n % nnx), j = (int)(n / nnx);
    double a0 = 0.0, a1 = 0.0;
    for (int jj = j - 1; jj <= j; jj++) {
      if (jj < 0 || jj >= ny) continue;
      const double sgy = (jj == j - 1) ? 1.0 : -1.0;
      for (int ii = i - 1; ii <= i; ii++) {
        if (ii < 0 || ii >= nx) continue;
        const double sgx = (ii == i - 1) ? 1.0 : -1.0;
        const double pe = p[ii + (long long)nx * jj];
        a0 -= sgx * (I.hy * 0.5) * pe;
        a1 -= sgy * (I.hx * 0.5) * pe;
      }
    }
    y[2 * n] = (bc[n] & 1u) ? 0.0 : a0;
    y[2 * n + 1] = (bc[n] & 2u) ? 0.0 : a1;
  }
  __syncthreads();
}

// q = G^T x (divergence per element)
template <int BS>
__device__ void bapply_Gt(const BInst& I, const double* __restrict__ x, double* __restrict__ q) {
  const int nx = I.nx, nnx = nx + 1;
  const long long E = (long long)nx * I.ny;
  for (long long e = tid(); e < E; e += BS) {
    const long long i = e % nx, j = e / nx;
    const long long n0 = i + (long long)nnx * j;
    const double* u0 = x + n0 * 2;
    const double* u1 = x + (n0 + 1) * 2;
    const double* u2 = x + (n0 + nnx) * 2;
    const double* u3 = x + (n0 + nnx + 1) * 2;
    const double fx = (u1[0] - u0[0]) + (u3[0] - u2[0]);
    const double fy = (u2[1] - u0[1]) + (u3[1] - u1[1]);
    q[e] = -(I.hy * 0.5) * fx - (I.hx * 0.5) * fy;
  }
  __syncthreads();
}

template <int BS>
__device__ double bdot(const double* a, const double* b, long long n, double* sh) {
  double v = 0.0;
  for (long long i = tid(); i < n; i += BS) v += a[i] * b[i];
  return block_sum<BS>(v, sh);
}

struct Inst {
  BInst I;
  long long N2, E;
  const double4* FS;
  const double *f, *dinv, *Qinv;
  const uint8_t* bc;
  double *u, *vstar, *ft, *cr, *cp, *cAp, *p, *r, *s, *q, *z;
  double *fs, *fq;
};

// Chebyshev-Jacobi smoothing on one level (FP32), window [0.1, 1.1] lmax: zero
// = start from x = 0.  x starts in `x` (or in Lx when zero) and ping-pongs;
// returns the buffer that holds it.  Sinkers of 16^2 to 48^2 take 1 to 4 %
// fewer inner iterations from 0.2 lmax (the single solver's bound) and no less
// time: 115 / 334 / 184 / 174 ms for four seeds' batches, 110 / 331 / 177 / 174
// from 0.1.
template <int BS>
__device__ float* bsmooth(const BArgs& A, const BLevel& L, int nu, bool zero, float* x) {
  const int w = L.nx + 1, h = L.ny + 1, N = w * h;
  const float4* S = A.LS + kStencil * L.node_off;
  const float2* dinv = reinterpret_cast<const float2*>(A.Ldinv + 2 * L.node_off);
  const float2* b = reinterpret_cast<const float2*>(A.Lb + 2 * L.node_off);
  float2* d = reinterpret_cast<float2*>(A.Ld + 2 * L.node_off);
  float *xa = A.Lx + 2 * L.node_off, *xb = A.Lx2 + 2 * L.node_off;
  const double emax = 1.1 * L.lmax, emin = 0.1 * L.lmax;
  const double theta = 0.5 * (emax + emin), delta = 0.5 * (emax - emin), sigma = theta / delta;
  double rho_prev = 1.0 / sigma;
  const float b0 = (float)(1.0 / theta);
  int k0 = 0;
  if (zero) {
    float2* x2 = reinterpret_cast<float2*>(xa);
    for (int n = tid(); n < N; n += BS) {
      const float2 bi = b[n], di = dinv[n];
      const float2 v = {b0 * di.x * bi.x, b0 * di.y * bi.y};
      d[n] = v;
      x2[n] = v;
    }
    __syncthreads();
    x = xa;
    k0 = 1;
  }
  for (int k = k0; k < nu; k++) {
    float c1 = 0.f, c2 = b0;
    if (k > 0) {
      const double rho = 1.0 / (2.0 * sigma - rho_prev);
      c1 = (float)(rho * rho_prev);
      c2 = (float)(2.0 * rho / delta);
      rho_prev = rho;
    }
    float* xo = x == xa ? xb : xa;
    for (int n = tid(); n < N; n += BS) {
      const int j = n / w, i = n - j * w;
      float y0, y1;
      const float2 bi = b[n], di = dinv[n], xi = reinterpret_cast<const float2*>(x)[n];
      float2 dv = {0.f, 0.f};
      if (k > 0) dv = d[n];
      st_row<float>(S, w, h, N, n, i, j, x, y0, y1);
      dv.x = c1 * dv.x + c2 * di.x * (bi.x - y0);
      dv.y = c1 * dv.y + c2 * di.y * (bi.y - y1);
      d[n] = dv;
      reinterpret_cast<float2*>(xo)[n] = float2{xi.x + dv.x, xi.y + dv.y};
    }
    __syncthreads();
    x = xo;
  }
  return x;
}

// One V-cycle on the instance's levels: level-0 b in; returns the buffer that
// holds the level-0 x (FP32).
template <int BS>
__device__ float* bvcycle(const BArgs& A, const BInst& I, int nu, float* shf) {
  const int Lc = I.nlev - 1;
  const int Ls = I.nfc > 0 ? Lc - 1 : Lc;  // last smoothed level
  unsigned in2 = 0;                        // bit l: level l's x is in Lx2
  for (int l = 0; l <= Ls; l++) {
    const BLevel F = A.lev[I.lev0 + l];
    float* x = bsmooth<BS>(A, F, l == Lc ? 8 : nu, true, nullptr);
    in2 |= (x == A.Lx2 + 2 * F.node_off ? 1u : 0u) << l;
    if (l == Lc) break;
    const BLevel C = A.lev[I.lev0 + l + 1];
    const int fw = F.nx + 1, fh = F.ny + 1, N = fw * fh;
    const float2* b = reinterpret_cast<const float2*>(A.Lb + 2 * F.node_off);
    float2* r = reinterpret_cast<float2*>(A.Lr + 2 * F.node_off);
    for (int n = tid(); n < N; n += BS) {
      const int j = n / fw, i = n - j * fw;
      float y0, y1;
      const float2 bi = b[n];
      st_row<float>(A.LS + kStencil * F.node_off, fw, fh, N, n, i, j, x, y0, y1);
      r[n] = float2{bi.x - y0, bi.y - y1};
    }
    __syncthreads();
    // full-weighting restriction to the coarse level (masked)
    const int cw = C.nx + 1, NC = cw * (C.ny + 1);
    float2* bcv = reinterpret_cast<float2*>(A.Lb + 2 * C.node_off);
    const uint8_t* cbc = A.Lbc + C.node_off;
    for (int n = tid(); n < NC; n += BS) {
      const int Jc = n / cw, Ic = n - Jc * cw;
      float2 v[9];
#pragma unroll
      for (int q = 0; q < 9; q++) {
        const int i = 2 * Ic + q % 3 - 1, j = 2 * Jc + q / 3 - 1;
        const bool in = i >= 0 && i < fw && j >= 0 && j < fh;
        v[q] = r[in ? i + fw * j : 0];
        if (!in) v[q] = float2{0.f, 0.f};
      }
      float a0 = 0.f, a1 = 0.f;
#pragma unroll
      for (int q = 0; q < 9; q++) {
        const float wt = (q % 3 == 1 ? 1.f : 0.5f) * (q / 3 == 1 ? 1.f : 0.5f);
        a0 += wt * v[q].x;
        a1 += wt * v[q].y;
      }
      const unsigned m = cbc[n];
      bcv[n] = float2{(m & 1u) ? 0.f : a0, (m & 2u) ? 0.f : a1};
    }
    __syncthreads();
  }
  if (I.nfc > 0) {
    const BLevel C = A.lev[I.lev0 + Lc];
    {
      const int nc = 2 * (C.nx + 1) * (C.ny + 1), nf = I.nfc;
      const float* b = A.Lb + 2 * C.node_off;
      float *x = A.Lx + 2 * C.node_off, *bf = A.Lr + 2 * C.node_off;  // bf: b on the free dofs
      const float* K = A.Kinv + I.kinv_off;
      const int* fi = A.freeidx + I.free_off;
      for (int i = tid(); i < nc; i += BS) x[i] = 0.f;
      for (int i = tid(); i < nf; i += BS) bf[i] = b[fi[i]];
      __syncthreads();
      // K is symmetric, so thread -> row reads column entries K[j][row]:
      // neighbouring threads neighbouring values.  Spare threads split the
      // columns; their partial sums are added in order through LDS.
      const int rows = (nf + 63) & ~63;
      const int G = rows <= BS ? BS / rows : 1;
      if (G > 1) {
        const int g = threadIdx.x / rows, row = threadIdx.x - g * rows;
        float acc = 0.f;
        if (g < G && row < nf) {
          const int j0 = (int)((long long)nf * g / G), j1 = (int)((long long)nf * (g + 1) / G);
#pragma unroll 8
          for (int j = j0; j < j1; j++) acc += K[(long long)j * nf + row] * bf[j];
        }
        shf[threadIdx.x] = acc;
        __syncthreads();
        if (threadIdx.x < nf) {
          float t = 0.f;
          for (int q = 0; q < G; q++) t += shf[q * rows + threadIdx.x];
          x[fi[threadIdx.x]] = t;
        }
      } else {
        for (int row = threadIdx.x; row < nf; row += BS) {
          float acc = 0.f;
#pragma unroll 8
          for (int j = 0; j < nf; j++) acc += K[(long long)j * nf + row] * bf[j];
          x[fi[row]] = acc;
        }
      }
      __syncthreads();
    }
  }
  for (int l = Lc - 1; l >= 0; l--) {
    const BLevel F = A.lev[I.lev0 + l], C = A.lev[I.lev0 + l + 1];
    // bilinear prolongation added to the fine iterate (masked)
    const int fw = F.nx + 1, cw = C.nx + 1, NF = fw * (F.ny + 1);
    const float2* xc = reinterpret_cast<const float2*>((((in2 >> (l + 1)) & 1u) ? A.Lx2 : A.Lx) + 2 * C.node_off);
    float* x = (((in2 >> l) & 1u) ? A.Lx2 : A.Lx) + 2 * F.node_off;
    float2* xf = reinterpret_cast<float2*>(x);
    const uint8_t* fbc = A.Lbc + F.node_off;
    for (int n = tid(); n < NF; n += BS) {
      const int j = n / fw, i = n - j * fw;
      // the (up to four) coarse parents; an even index has one with weight 1
      const int ci = i >> 1, cj = j >> 1, di = i & 1, dj = j & 1;
      const float2 v00 = xc[ci + cw * cj], v10 = xc[ci + di + cw * cj], v01 = xc[ci + cw * (cj + dj)],
                   v11 = xc[ci + di + cw * (cj + dj)];
      const float2 xv = xf[n];
      const unsigned m = fbc[n];
      const float a0 = 0.25f * ((v00.x + v10.x) + (v01.x + v11.x)), a1 = 0.25f * ((v00.y + v10.y) + (v01.y + v11.y));
      xf[n] = float2{(m & 1u) ? xv.x : xv.x + a0, (m & 2u) ? xv.y : xv.y + a1};
    }
    __syncthreads();
    x = bsmooth<BS>(A, F, nu, false, x);
    in2 = (in2 & ~(1u << l)) | ((x == A.Lx2 + 2 * F.node_off ? 1u : 0u) << l);
  }
  return ((in2 & 1u) ? A.Lx2 : A.Lx) + 2 * A.lev[I.lev0].node_off;
}

// x = K^-1 b (flexible CG, FP64), stopping at |r| <= rtol |b|.  Returns 0 or
// GS_E_INNER_MAXIT / GS_E_NAN.  z = V-cycle(r) stays in its FP32 level-0
// buffer; the FP32 copy of r that it starts from is written with r.
template <int BS>
__device__ int inner_solve(const BArgs& A, const Inst& W, const double* b, double* x, double rtol, long long* its,
                           double* sh, float* shf) {
  float* b0 = A.Lb + 2 * A.lev[W.I.lev0].node_off;
  const int w = W.I.nx + 1, h = W.I.ny + 1, N = w * h, N2 = 2 * N;
  double bb = 0.0;
  for (int i = tid(); i < N2; i += BS) {
    const double bi = b[i];
    x[i] = 0.0;
    W.cr[i] = bi;
    b0[i] = (float)bi;
    bb += bi * bi;
  }
  bb = block_sum<BS>(bb, sh);
  if (!(bb > 0.0)) return isfinite(bb) ? 0 : GS_E_NAN;
  const double stop = rtol * rtol * bb;
  double rz = 0.0, alpha = 0.0;
  for (int k = 0; k < A.max_inner; k++) {
    const float* z = bvcycle<BS>(A, W.I, A.nu, shf);
    double zs[2] = {0.0, 0.0};  // z.r, z.Ap
    for (int i = tid(); i < N2; i += BS) {
      const double zi = (double)z[i];
      zs[0] += zi * W.cr[i];
      if (k > 0) zs[1] += zi * W.cAp[i];
    }
    block_sums<BS, 2>(zs, sh);
    const double beta = k > 0 && rz != 0.0 ? -alpha * zs[1] / rz : 0.0;
    rz = zs[0];
    for (int i = tid(); i < N2; i += BS) W.cp[i] = k > 0 ? (double)z[i] + beta * W.cp[i] : (double)z[i];
    __syncthreads();
    double pap = 0.0;
    for (int n = tid(); n < N; n += BS) {
      const int j = n / w, i = n - j * w;
      double y0, y1;
      st_row<double>(W.FS, w, h, N, n, i, j, W.cp, y0, y1);
      const double2 pn = reinterpret_cast<const double2*>(W.cp)[n];
      reinterpret_cast<double2*>(W.cAp)[n] = double2{y0, y1};
      pap += pn.x * y0 + pn.y * y1;
    }
    pap = block_sum<BS>(pap, sh);
    alpha = (pap != 0.0 && isfinite(pap)) ? rz / pap : 0.0;
    double rr = 0.0;
    for (int i = tid(); i < N2; i += BS) {
      x[i] += alpha * W.cp[i];
      const double ri = W.cr[i] - alpha * W.cAp[i];
      W.cr[i] = ri;
      b0[i] = (float)ri;
      rr += ri * ri;
    }
    rr = block_sum<BS>(rr, sh);
    (*its)++;
    if (!isfinite(rr)) return GS_E_NAN;
    if (rr <= stop) return 0;
  }
  return GS_E_INNER_MAXIT;
}

// One instance: Stokes_SLE_UzawaSolver.cxx:553-837 (RELAX false), or the same
// solve with inexact inner solves (RELAX true): the inner tolerance is
// relaxed as the outer residual falls,
// rtol_k = min(relax, max(irt, irt |r_0| / |r_k|)) (the inexact-Krylov
// relaxation rule), and the outer iteration is flexible CG on S = G^T K^-1 G
// with each new direction S-orthogonalised against the last `window` ones,
// which keeps it converging with inexact applications of S.  When the
// recursive residual reaches the tolerance, the true residual is recomputed
// from an accurate inner solve u = K^-1 (f - G p) (the reference's STEP 3) and
// the loop resumes from it if needed; a round that stagnates (less than 5 %
// residual drop over 50 iterations) also ends in that check.  Each new round
// relaxes ten times less and the fifth not at all (then the loop is flexible
// CG with the reference inner tolerance).  The reported residual is the true
// one.  Same firewalls in both.
//
// The solve is a sequence of inner solves told apart by `phase`, so that the
// inner solve (and the V-cycle in it) is in the kernel once: inlined at every
// call site it overflowed the registers by 3 KB a thread.
template <int BS, bool RELAX>
__device__ int solve_one(const Inst& W, const BArgs& A, int* outer_out, long long* inner_out, double* relres_out,
                         double* sh, float* shf, double* sqv) {
  const long long N2 = W.N2, E = W.E;
  long long inner = 0;
  const double qRecip = 1.0 / sqrt((double)E);
  *outer_out = 0;
  *inner_out = 0;
  *relres_out = 0.0;
  {
    // zero-force firewall (:476-493)
    double v[2] = {0.0, 0.0};
    for (long long i = tid(); i < N2; i += BS) {
      v[0] += W.dinv[i] != 0.0 ? 1.0 : 0.0;
      v[1] += W.f[i] * W.f[i];
    }
    block_sums<BS, 2>(v, sh);
    if (sqrt(v[1]) / sqrt(v[0] > 0 ? v[0] : 1.0) <= 1e-99) return GS_E_ZERO_FORCE;
  }
  enum { kFirst, kStart, kLoop, kVerify };
  int phase = kFirst, it = 0, err = 0;
  double scale = 1.0, relRes = 0.0, zr = 0.0, zr_prev = 1.0;
  // relaxed loop
  constexpr int kRounds = 5, kStagWin = 50;
  const int m = A.window;
  int round = 0, base = 0, stag_it = 0, slot = 0;
  double relax = A.relax, relax_ref = 0.0, stag_ref = 0.0;
  for (;;) {
    const double* rhs = W.f;
    double* dst = W.vstar;
    double* q = W.q;
    double* sdir = W.s;
    double rt = A.irt;
    if (phase == kFirst) {
      // STEP 1: vstar = K^-1 f; z = G^T vstar - h (h = 0, homogeneous conditions)
      rt = A.tol;
      q = W.z;
    } else if (phase == kStart) {
      // STEP 3: u = K^-1 (f - G p), p = 0; r = G^T u - h
      for (long long e = tid(); e < E; e += BS) W.p[e] = 0.0;
      dst = W.u;
      q = W.r;
    } else if (phase == kVerify) {
      // true residual: u = K^-1 (f - G p) with the reference inner tolerance
      bapply_G<BS>(W.I, W.p, W.ft, W.bc);
      for (long long i = tid(); i < N2; i += BS) W.ft[i] = W.f[i] - W.ft[i];
      __syncthreads();
      rhs = W.ft;
      dst = W.u;
      q = W.r;
    } else {
      rhs = W.ft;
      if (RELAX) {
        for (long long e = tid(); e < E; e += BS) W.z[e] = W.Qinv[e] * W.r[e];
        __syncthreads();
        const int k = it - base, c = k < m ? k : m;
        slot = k % m;
        sdir = W.fs + (long long)slot * E;
        q = W.fq + (long long)slot * E;
        double beta[kBatchMaxWin];
#pragma unroll
        for (int j = 0; j < kBatchMaxWin; j++) beta[j] = 0.0;
        for (long long e = tid(); e < E; e += BS) {
          const double zi = W.z[e];
#pragma unroll
          for (int j = 0; j < kBatchMaxWin; j++)
            if (j < c) beta[j] += zi * W.fq[(long long)j * E + e];
        }
        block_sums<BS, kBatchMaxWin>(beta, sh);
#pragma unroll
        for (int j = 0; j < kBatchMaxWin; j++)
          if (j < c) beta[j] /= sqv[j];
        for (long long e = tid(); e < E; e += BS) {
          double v = W.z[e];
#pragma unroll
          for (int j = 0; j < kBatchMaxWin; j++)
            if (j < c) v -= beta[j] * W.fs[(long long)j * E + e];
          sdir[e] = v;
        }
        if (relax > 0 && relRes > 0) rt = fmin(relax, fmax(A.irt, A.irt * relax_ref / relRes));
      } else {
        zr = 0.0;
        for (long long e = tid(); e < E; e += BS) {
          const double zi = W.Qinv[e] * W.r[e];
          W.z[e] = zi;
          zr += zi * W.r[e];
        }
        zr = block_sum<BS>(zr, sh);
        const double beta = it == 0 ? 0.0 : (zr_prev != 0.0 ? zr / zr_prev : 0.0);
        for (long long e = tid(); e < E; e += BS) W.s[e] = it == 0 ? W.z[e] : W.z[e] + beta * W.s[e];
      }
      __syncthreads();
      bapply_G<BS>(W.I, sdir, W.ft, W.bc);
    }
    err = inner_solve<BS>(A, W, rhs, dst, rt, &inner, sh, shf);
    if (err) {
      if (phase == kFirst || phase == kStart) return err;
      break;
    }
    bapply_Gt<BS>(W.I, dst, q);
    if (phase == kFirst) {
      scale = sqrt(bdot<BS>(W.z, W.z, E, sh)) * qRecip;
      if (!isfinite(scale)) return GS_E_NAN;
      phase = kStart;
      continue;
    }
    if (phase == kLoop) {
      double sv[2] = {0.0, 0.0};  // s.q, s.r
      for (long long e = tid(); e < E; e += BS) {
        const double si = sdir[e];
        sv[0] += si * q[e];
        if (RELAX) sv[1] += si * W.r[e];
      }
      block_sums<BS, 2>(sv, sh);
      const double sq = sv[0];
      if (RELAX && threadIdx.x == 0) sqv[slot] = sq;
      const double num = RELAX ? sv[1] : zr, alpha = num / sq;
      if ((!RELAX && !isfinite(zr)) || !isfinite(sq) || !isfinite(alpha)) {
        err = GS_E_NAN;
        break;
      }
      double rr = 0.0;
      for (long long e = tid(); e < E; e += BS) {
        W.p[e] += alpha * sdir[e];
        const double ri = W.r[e] - alpha * q[e];
        W.r[e] = ri;
        rr += ri * ri;
      }
      for (long long i = tid(); i < N2; i += BS) W.u[i] -= alpha * W.vstar[i];
      rr = block_sum<BS>(rr, sh);
      zr_prev = zr;
      relRes = sqrt(rr) * qRecip / scale;
      if (!isfinite(relRes)) {
        err = GS_E_NAN;
        break;
      }
      if (!(it < A.max_outer)) {
        err = GS_E_MAXIT;
        break;
      }
      it++;
      if (!RELAX) {
        if (!(relRes > A.tol)) break;
        continue;
      }
      if (relRes <= A.tol) {
        phase = kVerify;
      } else if (relax > 0 && it - stag_it >= kStagWin) {
        // stagnation (less than 5 % drop over kStagWin iterations) while still
        // relaxing: end the round, re-check the true residual, relax less
        if (relRes > 0.95 * stag_ref) phase = kVerify;
        stag_ref = relRes;
        stag_it = it;
      }
      continue;
    }
    // kStart, kVerify: r is the true residual
    if (RELAX) {
      relRes = sqrt(bdot<BS>(W.r, W.r, E, sh)) * qRecip / scale;
      if (phase == kVerify) {
        if (!isfinite(relRes)) {
          err = GS_E_NAN;
          break;
        }
        if (relRes <= A.tol) break;
        if (round == kRounds - 1) {
          err = GS_E_MAXIT;
          break;
        }
        round++;
      }
      // each round relaxes ten times less; the last one not at all
      relax = round == kRounds - 1 ? 0.0 : A.relax * pow(0.1, (double)round);
      relax_ref = stag_ref = relRes;
      base = stag_it = it;
    }
    phase = kLoop;
  }
  *outer_out = it;
  *inner_out = inner;
  *relres_out = relRes;
  return err;
}

template <int BS, bool RELAX>
__global__ __launch_bounds__(BS) void k_batch_uzawa(BArgs A) {
  __shared__ double sh[kBatchMaxWin * (BS / 64)];
  __shared__ float shf[BS];
  __shared__ double sqv[kBatchMaxWin];
  __shared__ int cur;
  for (;;) {
    if (threadIdx.x == 0) {
      const unsigned k = atomicAdd(A.queue, 1u);
      cur = k < (unsigned)A.B ? A.order[k] : -1;
    }
    __syncthreads();
    const int i = __builtin_amdgcn_readfirstlane(cur);  // uniform: the instance's pointers and sizes stay in scalar registers
    __syncthreads();
    if (i < 0) return;
    Inst W;
    W.I = A.inst[i];
    const long long no = W.I.node_off, eo = W.I.elem_off;
    W.N2 = 2LL * (W.I.nx + 1) * (W.I.ny + 1);
    W.E = (long long)W.I.nx * W.I.ny;
    W.FS = A.FS + kStencil * no;
    W.f = A.f + 2 * no;
    W.dinv = A.dinv + 2 * no;
    W.Qinv = A.Qinv + eo;
    W.bc = A.bc + no;
    W.u = A.u + 2 * no;
    W.vstar = A.vstar + 2 * no;
    W.ft = A.ft + 2 * no;
    W.cr = A.cr + 2 * no;
    W.cp = A.cp + 2 * no;
    W.cAp = A.cAp + 2 * no;
    W.p = A.p + eo;
    W.r = A.r + eo;
    W.s = A.s + eo;
    W.q = A.q + eo;
    W.z = A.z + eo;
    W.fs = A.fs ? A.fs + (long long)A.window * eo : nullptr;
    W.fq = A.fq ? A.fq + (long long)A.window * eo : nullptr;
    int outer = 0;
    long long inner = 0;
    double rel = 0.0;
    const unsigned long long t0 = wall_clock64();
    const int st = solve_one<BS, RELAX>(W, A, &outer, &inner, &rel, sh, shf, sqv);
    if (threadIdx.x == 0) {
      A.itime[i] = wall_clock64() - t0;
      A.status[i] = st;
      A.outer[i] = outer;
      A.inner[i] = inner;
      A.relres[i] = rel;
    }
    __syncthreads();
  }
}

__global__ void k_zero_queue(unsigned* q) {
  if (threadIdx.x == 0 && blockIdx.x == 0) q[0] = 0u;
}

struct Tile {
  int bs, tx;
};
const Tile kTiles[6] = {{256, 16}, {256, 32}, {512, 32}, {512, 64}, {1024, 32}, {1024, 64}};

}  // namespace

struct gs_batch {
  int B = 0;
  hipStream_t st = nullptr;
  std::vector<BInst> hinst;
  std::vector<BLevel> hlev;
  BInst* inst = nullptr;
  BLevel* lev = nullptr;
  int* order = nullptr;
  long long elems = 0;
  double4* FS = nullptr;
  double *f = nullptr, *dinv = nullptr, *Qinv = nullptr;
  uint8_t* bc = nullptr;
  float4* LS = nullptr;
  float *Ldinv = nullptr, *Lb = nullptr, *Lx = nullptr, *Lr = nullptr, *Ld = nullptr, *Lx2 = nullptr;
  uint8_t* Lbc = nullptr;
  float* Kinv = nullptr;
  int* freeidx = nullptr;
  double *u = nullptr, *vstar = nullptr, *ft = nullptr, *cr = nullptr, *cp = nullptr, *cAp = nullptr;
  double *p = nullptr, *r = nullptr, *s = nullptr, *q = nullptr, *z = nullptr;
  int *status = nullptr, *outer = nullptr;
  unsigned long long* itime = nullptr;
  double clock_khz = 100000.0;  // wall_clock64 rate
  long long* inner = nullptr;
  double* relres = nullptr;
  double *fs = nullptr, *fq = nullptr;  // relaxed loop direction rings (window x elements)
  int fwin = 0;
  unsigned* queue = nullptr;
  // index into kTiles: 512 threads, the most whose vector registers do not
  // spill (217 scalar ones do, to lanes of vector registers).  32 sinkers of
  // 16^2 to 48^2, four seeds, reference loop: 110 / 331 / 177 / 174 ms, against
  // 146 / 443 / 240 / 228 with 256 threads and 127 / 376 / 202 / 201 with 1024;
  // one of 128^2 148 ms, 216 and 146.
  int tile = 2;
  int ncu = 256;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  gs_batch_params gparams{};
  int gtile = -1;
};

template <typename T>
static hipError_t balloc(T** p, long long n) {
  return hipMalloc(reinterpret_cast<void**>(p), sizeof(T) * (n > 0 ? n : 1));
}

static void free_graph(gs_batch* b) {
  if (b->exec) (void)hipGraphExecDestroy(b->exec);
  if (b->graph) (void)hipGraphDestroy(b->graph);
  b->exec = nullptr;
  b->graph = nullptr;
  b->gtile = -1;
}

extern "C" void gs_batch_destroy(gs_batch* b) {
  if (!b) return;
  if (b->st) (void)hipStreamSynchronize(b->st);
  free_graph(b);
  void* ptrs[] = {b->inst, b->lev, b->order, b->FS, b->f, b->dinv, b->Qinv, b->bc, b->LS, b->Ldinv, b->Lb, b->Lx,
                  b->Lr, b->Ld, b->Lx2, b->Lbc, b->Kinv, b->freeidx, b->u, b->vstar, b->ft, b->cr, b->cp,
                  b->cAp, b->p, b->r, b->s, b->q, b->z, b->status, b->outer, b->inner, b->relres, b->queue,
                  b->fs, b->fq, b->itime};
  for (void* p : ptrs)
    if (p) (void)hipFree(p);
  if (b->e0) (void)hipEventDestroy(b->e0);
  if (b->e1) (void)hipEventDestroy(b->e1);
  if (b->st) (void)hipStreamDestroy(b->st);
  delete b;
}

extern "C" int32_t gs_batch_create(int32_t count, const gs_problem_desc* descs, gs_batch** out) {
  if (!out || count < 1 || !descs) return GS_E_INVALID;
  *out = nullptr;
  int nd = 0;
  if (hipGetDeviceCount(&nd) != hipSuccess || nd < 1) return GS_E_NO_DEVICE;
  for (int i = 0; i < count; i++)
    if (descs[i].dim != 2 || descs[i].res[0] < 1 || descs[i].res[1] < 1) return GS_E_INVALID;
  gs_batch* b = new gs_batch();
  b->B = count;
  std::vector<gs_problem*> pbs(count, nullptr);
  std::vector<gs_solver*> svs(count, nullptr);
  auto fail = [&](int32_t s) {
    for (int i = 0; i < count; i++) {
      if (svs[i]) gs_solver_destroy(svs[i]);
      if (pbs[i]) gs_problem_destroy(pbs[i]);
    }
    gs_batch_destroy(b);
    return s;
  };
  if (hipStreamCreate(&b->st) != hipSuccess || hipEventCreate(&b->e0) != hipSuccess ||
      hipEventCreate(&b->e1) != hipSuccess)
    return fail(GS_E_HIP);
  {
    hipDeviceProp_t prop;
    int dev = 0;
    if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&prop, dev) == hipSuccess &&
        prop.multiProcessorCount > 0)
      b->ncu = prop.multiProcessorCount;
    int khz = 0;
    if (hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev) == hipSuccess && khz > 0)
      b->clock_khz = khz;
  }
  // per-instance setup through the single-problem path: particle location,
  // constitutive pass, right-hand side, multigrid levels (Galerkin moments,
  // Chebyshev bounds, dense coarsest inverse)
  gs_uzawa_params up{};
  up.tolerance = 1e-6;
  up.max_iterations = 1;
  up.preconditioner = GS_PC_DIAGONAL;
  up.precision = GS_PREC_MIXED;
  up.inner_preconditioner = GS_INNER_MULTIGRID;
  constexpr int kMaxLev = 16;
  std::vector<std::vector<BatchLevelInfo>> info(count, std::vector<BatchLevelInfo>(kMaxLev));
  b->hinst.resize(count);
  long long no = 0, eo = 0, lno = 0, ko = 0, fo = 0;
  for (int i = 0; i < count; i++) {
    const gs_problem_desc& d = descs[i];
    int32_t s = gs_problem_create(&d, &pbs[i]);
    if (s != GS_OK) return fail(s);
    if ((s = gs_solver_create(pbs[i], &up, &svs[i])) != GS_OK) return fail(s);
    batch_mark(svs[i]);
    if ((s = gs_solver_setup(svs[i], nullptr, nullptr, 0)) != GS_OK) return fail(s);
    int nl = 0, nfc = 0;
    if ((s = batch_mg_info(svs[i], &nl, info[i].data(), kMaxLev, &nfc)) != GS_OK) return fail(s);
    BInst& I = b->hinst[i];
    I.nx = d.res[0];
    I.ny = d.res[1];
    I.node_off = no;
    I.elem_off = eo;
    I.hx = (d.hi[0] - d.lo[0]) / d.res[0];
    I.hy = (d.hi[1] - d.lo[1]) / d.res[1];
    I.lev0 = (int)b->hlev.size();
    I.nlev = nl;
    I.nfc = nfc;
    I.kinv_off = ko;
    I.free_off = fo;
    if (nfc > 0) {
      ko += (long long)nfc * nfc;
      fo += nfc;
    }
    no += (long long)(I.nx + 1) * (I.ny + 1);
    eo += (long long)I.nx * I.ny;
    for (int l = 0; l < nl; l++) {
      BLevel L{};
      L.nx = info[i][l].nx;
      L.ny = info[i][l].ny;
      L.node_off = lno;
      L.hx = (d.hi[0] - d.lo[0]) / L.nx;
      L.hy = (d.hi[1] - d.lo[1]) / L.ny;
      L.lmax = info[i][l].lmax;
      b->hlev.push_back(L);
      lno += (long long)(L.nx + 1) * (L.ny + 1);
    }
  }
  b->elems = eo;
  const long long N2 = 2 * no, L2 = 2 * lno;
  if (balloc(&b->inst, count) || balloc(&b->lev, (long long)b->hlev.size()) || balloc(&b->order, count) ||
      balloc(&b->FS, kStencil * no) || balloc(&b->f, N2) || balloc(&b->dinv, N2) || balloc(&b->Qinv, eo) ||
      balloc(&b->bc, no) || balloc(&b->LS, kStencil * lno) || balloc(&b->Ldinv, L2) || balloc(&b->Lb, L2) ||
      balloc(&b->Lx, L2) || balloc(&b->Lr, L2) || balloc(&b->Ld, L2) || balloc(&b->Lx2, L2) ||
      balloc(&b->Lbc, lno) || balloc(&b->Kinv, ko) || balloc(&b->freeidx, fo) || balloc(&b->u, N2) ||
      balloc(&b->vstar, N2) || balloc(&b->ft, N2) || balloc(&b->cr, N2) ||
      balloc(&b->cp, N2) || balloc(&b->cAp, N2) || balloc(&b->p, eo) || balloc(&b->r, eo) || balloc(&b->s, eo) ||
      balloc(&b->q, eo) || balloc(&b->z, eo) || balloc(&b->status, count) || balloc(&b->outer, count) ||
      balloc(&b->inner, count) || balloc(&b->relres, count) || balloc(&b->queue, 1) || balloc(&b->itime, count))
    return fail(GS_E_HIP);
  for (int i = 0; i < count; i++) {
    const BInst& I = b->hinst[i];
    int32_t s = batch_copy_fine(svs[i], b->f + 2 * I.node_off, b->dinv + 2 * I.node_off, b->Qinv + I.elem_off, b->st);
    for (int l = 0; l < I.nlev && s == GS_OK; l++) {
      const BLevel& L = b->hlev[I.lev0 + l];
      s = batch_copy_level(svs[i], l, b->Ldinv + 2 * L.node_off, b->Lbc + L.node_off, b->st);
      if (s != GS_OK) break;
      // the solver's stream is idle (its setup waits for the device), so its
      // moments can be read from this one
      const double* M64 = nullptr;
      const float* M32 = nullptr;
      batch_moments(svs[i], l, &M64, &M32);
      const long long nt = kStencil * (long long)(L.nx + 1) * (L.ny + 1);
      const dim3 nb((unsigned)((nt + kBlock - 1) / kBlock));
      hipLaunchKernelGGL(k_stencil<float>, nb, dim3(kBlock), 0, b->st, L.nx, L.ny, (float)(0.5 / L.hx),
                         (float)(0.5 / L.hy), M32, b->Lbc + L.node_off, b->LS + kStencil * L.node_off);
      if (l == 0)
        hipLaunchKernelGGL(k_stencil<double>, nb, dim3(kBlock), 0, b->st, L.nx, L.ny, 0.5 / L.hx, 0.5 / L.hy, M64,
                           b->Lbc + L.node_off, b->FS + kStencil * I.node_off);
      if (hipGetLastError() != hipSuccess) s = GS_E_HIP;
    }
    if (s == GS_OK && I.nfc > 0) s = batch_copy_dense(svs[i], b->Kinv + I.kinv_off, b->freeidx + I.free_off, b->st);
    if (s == GS_OK && hipStreamSynchronize(b->st) != hipSuccess) s = GS_E_HIP;
    if (s != GS_OK) return fail(s);
    // the fine-level node flags equal level 0's
    const BLevel& L0 = b->hlev[I.lev0];
    if (hipMemcpyAsync(b->bc + I.node_off, b->Lbc + L0.node_off, (size_t)(I.nx + 1) * (I.ny + 1),
                       hipMemcpyDeviceToDevice, b->st) != hipSuccess)
      return fail(GS_E_HIP);
    gs_solver_destroy(svs[i]);
    svs[i] = nullptr;
    gs_problem_destroy(pbs[i]);
    pbs[i] = nullptr;
  }
  std::vector<int> ord(count);
  for (int i = 0; i < count; i++) ord[i] = i;
  std::stable_sort(ord.begin(), ord.end(), [&](int a, int c) {
    return (long long)b->hinst[a].nx * b->hinst[a].ny > (long long)b->hinst[c].nx * b->hinst[c].ny;
  });
  if (hipMemcpyAsync(b->inst, b->hinst.data(), sizeof(BInst) * count, hipMemcpyHostToDevice, b->st) ||
      hipMemcpyAsync(b->lev, b->hlev.data(), sizeof(BLevel) * b->hlev.size(), hipMemcpyHostToDevice, b->st) ||
      hipMemcpyAsync(b->order, ord.data(), sizeof(int) * count, hipMemcpyHostToDevice, b->st) ||
      hipStreamSynchronize(b->st))
    return fail(GS_E_HIP);
  *out = b;
  return GS_OK;
}

extern "C" int32_t gs_batch_set_tile(gs_batch* b, int32_t block, int32_t tx) {
  if (!b) return GS_E_INVALID;
  for (int k = 0; k < 6; k++)
    if (kTiles[k].bs == block && kTiles[k].tx == tx) {
      if (b->tile != k) free_graph(b);
      b->tile = k;
      return GS_OK;
    }
  return GS_E_INVALID;
}

static BArgs make_args(gs_batch* b, const gs_batch_params* p) {
  BArgs A{};
  A.inst = b->inst;
  A.lev = b->lev;
  A.LS = b->LS;
  A.FS = b->FS;
  A.Ldinv = b->Ldinv;
  A.Lbc = b->Lbc;
  A.Lb = b->Lb;
  A.Lx = b->Lx;
  A.Lr = b->Lr;
  A.Ld = b->Ld;
  A.Lx2 = b->Lx2;
  A.Kinv = b->Kinv;
  A.freeidx = b->freeidx;
  A.order = b->order;
  A.B = b->B;
  A.f = b->f;
  A.dinv = b->dinv;
  A.Qinv = b->Qinv;
  A.bc = b->bc;
  A.u = b->u;
  A.vstar = b->vstar;
  A.ft = b->ft;
  A.cr = b->cr;
  A.cp = b->cp;
  A.cAp = b->cAp;
  A.p = b->p;
  A.r = b->r;
  A.s = b->s;
  A.q = b->q;
  A.z = b->z;
  A.status = b->status;
  A.itime = b->itime;
  A.outer = b->outer;
  A.inner = b->inner;
  A.relres = b->relres;
  A.queue = b->queue;
  A.tol = p->tolerance;
  A.irt = (p->inner_rtol_factor > 0 ? p->inner_rtol_factor : 0.1) * p->tolerance;
  A.max_outer = p->max_iterations > 0 ? p->max_iterations : 1000;
  A.max_inner = p->max_inner > 0 ? p->max_inner : 20000;
  A.nu = p->mg_smooth > 0 ? p->mg_smooth : 2;
  A.relax = p->inner_relax_max > 0 ? p->inner_relax_max : 0.0;
  A.window = p->flexible_window > 0 ? std::min(p->flexible_window, kBatchMaxWin) : 8;
  A.fs = b->fs;
  A.fq = b->fq;
  return A;
}

// Direction rings of the relaxed loop (allocated on first use, before any
// graph capture).  A captured graph holds their addresses, so it goes with the
// rings it was captured with.
static int32_t ensure_rings(gs_batch* b, const gs_batch_params* p) {
  if (!(p->inner_relax_max > 0)) return GS_OK;
  const int m = p->flexible_window > 0 ? std::min(p->flexible_window, kBatchMaxWin) : 8;
  if (b->fs && b->fwin == m) return GS_OK;
  free_graph(b);
  if (b->fs) (void)hipFree(b->fs);
  if (b->fq) (void)hipFree(b->fq);
  b->fs = b->fq = nullptr;
  b->fwin = 0;
  BCK(balloc(&b->fs, (long long)m * b->elems));
  BCK(balloc(&b->fq, (long long)m * b->elems));
  b->fwin = m;
  return GS_OK;
}

static void launch_batch(gs_batch* b, const BArgs& A, int tile, hipStream_t st) {
  // one workgroup per instance, up to 2 per CU; the queue hands out instances
  const unsigned grid = (unsigned)std::min(b->B, 2 * b->ncu);
  hipLaunchKernelGGL(k_zero_queue, dim3(1), dim3(64), 0, st, b->queue);
  // the tile width only tells shapes of one block size apart: the stencil
  // applies walk the nodes in order whatever it is
  const int bs = kTiles[tile].bs;
  if (A.relax > 0) {
    switch (bs) {
      case 256: hipLaunchKernelGGL((k_batch_uzawa<256, true>), dim3(grid), dim3(256), 0, st, A); break;
      case 512: hipLaunchKernelGGL((k_batch_uzawa<512, true>), dim3(grid), dim3(512), 0, st, A); break;
      default: hipLaunchKernelGGL((k_batch_uzawa<1024, true>), dim3(grid), dim3(1024), 0, st, A); break;
    }
  } else {
    switch (bs) {
      case 256: hipLaunchKernelGGL((k_batch_uzawa<256, false>), dim3(grid), dim3(256), 0, st, A); break;
      case 512: hipLaunchKernelGGL((k_batch_uzawa<512, false>), dim3(grid), dim3(512), 0, st, A); break;
      default: hipLaunchKernelGGL((k_batch_uzawa<1024, false>), dim3(grid), dim3(1024), 0, st, A); break;
    }
  }
}

static bool same_params(const gs_batch_params& a, const gs_batch_params& c) {
  return a.tolerance == c.tolerance && a.max_iterations == c.max_iterations && a.max_inner == c.max_inner &&
         a.inner_rtol_factor == c.inner_rtol_factor && a.mg_smooth == c.mg_smooth &&
         a.inner_relax_max == c.inner_relax_max && a.flexible_window == c.flexible_window;
}

extern "C" int32_t gs_batch_solve(gs_batch* b, const gs_batch_params* p, gs_batch_result* results, double* seconds) {
  if (!b || !p || !(p->tolerance > 0)) return GS_E_INVALID;
  if (p->flexible_window < 0 || p->flexible_window > kBatchMaxWin) return GS_E_INVALID;
  {
    const int32_t s = ensure_rings(b, p);
    if (s != GS_OK) return s;
  }
  const BArgs A = make_args(b, p);
  if (p->use_graph) {
    if (!b->exec || b->gtile != b->tile || !same_params(b->gparams, *p)) {
      free_graph(b);
      BCK(hipStreamBeginCapture(b->st, hipStreamCaptureModeThreadLocal));
      launch_batch(b, A, b->tile, b->st);
      BCK(hipStreamEndCapture(b->st, &b->graph));
      BCK(hipGraphInstantiate(&b->exec, b->graph, nullptr, nullptr, 0));
      b->gparams = *p;
      b->gtile = b->tile;
    }
    BCK(hipEventRecord(b->e0, b->st));
    BCK(hipGraphLaunch(b->exec, b->st));
    BCK(hipEventRecord(b->e1, b->st));
  } else {
    BCK(hipEventRecord(b->e0, b->st));
    launch_batch(b, A, b->tile, b->st);
    BCK(hipGetLastError());
    BCK(hipEventRecord(b->e1, b->st));
  }
  BCK(hipEventSynchronize(b->e1));
  float ms = 0.f;
  BCK(hipEventElapsedTime(&ms, b->e0, b->e1));
  if (seconds) *seconds = ms * 1e-3;
  std::vector<int> st(b->B), ou(b->B);
  std::vector<long long> in(b->B);
  std::vector<double> rr(b->B);
  std::vector<unsigned long long> tk(b->B);
  BCK(hipMemcpy(st.data(), b->status, sizeof(int) * b->B, hipMemcpyDeviceToHost));
  BCK(hipMemcpy(tk.data(), b->itime, sizeof(unsigned long long) * b->B, hipMemcpyDeviceToHost));
  BCK(hipMemcpy(ou.data(), b->outer, sizeof(int) * b->B, hipMemcpyDeviceToHost));
  BCK(hipMemcpy(in.data(), b->inner, sizeof(long long) * b->B, hipMemcpyDeviceToHost));
  BCK(hipMemcpy(rr.data(), b->relres, sizeof(double) * b->B, hipMemcpyDeviceToHost));
  int32_t worst = GS_OK;
  for (int i = 0; i < b->B; i++) {
    if (results) results[i] = gs_batch_result{st[i], ou[i], (int64_t)in[i], rr[i], (double)tk[i] / (b->clock_khz * 1e3)};
    if (st[i] != GS_OK && worst == GS_OK) worst = st[i];
  }
  return worst;
}

extern "C" int32_t gs_batch_autotune(gs_batch* b, const gs_batch_params* p, int32_t* block, int32_t* tx, float* ms) {
  if (!b || !p) return GS_E_INVALID;
  if (p->flexible_window < 0 || p->flexible_window > kBatchMaxWin) return GS_E_INVALID;
  {
    const int32_t s = ensure_rings(b, p);
    if (s != GS_OK) return s;
  }
  gs_batch_params q = *p;
  q.use_graph = 0;
  if (q.max_iterations <= 0 || q.max_iterations > 3) q.max_iterations = 3;  // a few Uzawa iterations per instance
  const BArgs A = make_args(b, &q);
  int best = b->tile;
  float best_ms = 1e30f;
  for (int k = 0; k < 6; k++) {
    if (k > 0 && kTiles[k].bs == kTiles[k - 1].bs) {  // the same kernel
      if (ms) ms[k] = ms[k - 1];
      continue;
    }
    BCK(hipEventRecord(b->e0, b->st));
    launch_batch(b, A, k, b->st);
    BCK(hipGetLastError());
    BCK(hipEventRecord(b->e1, b->st));
    BCK(hipEventSynchronize(b->e1));
    float t = 0.f;
    BCK(hipEventElapsedTime(&t, b->e0, b->e1));
    if (ms) ms[k] = t;
    if (t < best_ms) {
      best_ms = t;
      best = k;
    }
  }
  if (b->tile != best) free_graph(b);
  b->tile = best;
  if (block) *block = kTiles[best].bs;
  if (tx) *tx = kTiles[best].tx;
  return GS_OK;
}

extern "C" int32_t gs_batch_solution(gs_batch* b, int32_t i, double* u, double* p) {
  if (!b || i < 0 || i >= b->B) return GS_E_INVALID;
  const BInst& I = b->hinst[i];
  BCK(hipStreamSynchronize(b->st));
  if (u)
    BCK(hipMemcpy(u, b->u + 2 * I.node_off, sizeof(double) * 2 * (I.nx + 1) * (I.ny + 1), hipMemcpyDeviceToHost));
  if (p) BCK(hipMemcpy(p, b->p + I.elem_off, sizeof(double) * I.nx * I.ny, hipMemcpyDeviceToHost));
  return GS_OK;
}
