// gs_dense.hip -- the dense coarsest operator of the multigrid: assembled
// from the element moments and inverted on the device.
//
// The inverse is the symmetric sweep, 64 rows at a time.  With P the panel of
// block column k (rows of other blocks), D = A_kk^-1 and T = P D:
//   A_ij <- A_ij - T_i P_j^T,  A_ik <- T_i,  A_kk <- -D
// after every block has been swept A holds -A^-1.  Only the lower triangle of
// blocks is kept up to date, so the whole inverse is n^3 flops, nearly all of
// them in k_sweep_update on v_mfma_f64_16x16x4.  Per 64-row step it is three
// dependent launches: at n = 5577 (the 12^3 level) 88 steps, where the update
// reads and writes the 125 MB lower triangle once per step and is bound by
// that.  Assembly and inverse there take about 11 ms where probing the
// operator from the host and a library Cholesky factor and inverse took
// 125 ms; at n = 1701 (8^3) under 2 ms against 1.3 s for a host inverse.
#include "gs_dense.h"
#include "gs_tile.h"

#include <math.h>

namespace gs {

namespace {

typedef double dvec2 __attribute__((ext_vector_type(2)));
typedef double dvec4 __attribute__((ext_vector_type(4)));
constexpr int NB = kDenseBlock;

__global__ void k_dense_clear(double* __restrict__ A, int nf, int ld) {
  const long long n2 = (long long)ld * ld / 2;
  dvec2* A2 = reinterpret_cast<dvec2*>(A);
  for (long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x; t < n2; t += (long long)gridDim.x * blockDim.x) {
    const long long r = 2 * t / ld, c = 2 * t - r * ld;
    dvec2 v;
    v.x = (r >= nf && c == r) ? 1.0 : 0.0;
    v.y = (r >= nf && c + 1 == r) ? 1.0 : 0.0;
    A2[t] = v;
  }
}

// D = A_kk^-1 by an unblocked sweep.  16 x 16 threads hold 4 x 4 entries each
// in registers; the pivot column goes through LDS (two buffers, so one
// barrier per pivot).  One workgroup on the critical path of every step: 64
// pivots of an LDS round trip and one division each.
__global__ __launch_bounds__(256) void k_sweep_diag(double* __restrict__ A, int ld, int k, double* __restrict__ D,
                                                    int* __restrict__ bad) {
  __shared__ double col[2][NB];
  const int ti = threadIdx.x >> 4, tj = threadIdx.x & 15;
  double* Ak = A + ((long long)k * NB) * ld + (long long)k * NB;
  double a[4][4];
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int r = 4 * ti + i, c = 4 * tj + j;
      a[i][j] = r >= c ? Ak[(long long)r * ld + c] : Ak[(long long)c * ld + r];
    }
  bool ok = true;
  for (int p4 = 0; p4 < 16; p4++) {
#pragma unroll
    for (int s = 0; s < 4; s++) {
      const int p = 4 * p4 + s;
      double* cb = col[s & 1];
      if (tj == p4)
#pragma unroll
        for (int i = 0; i < 4; i++) cb[4 * ti + i] = a[i][s];
      __syncthreads();
      const double d = cb[p];
      ok = ok && d > 0.0 && isfinite(d);
      const double rd = 1.0 / d;
      double ci[4], cj[4];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        ci[i] = cb[4 * ti + i];
        cj[i] = cb[4 * tj + i] * rd;
      }
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const bool pr = ti == p4 && i == s, pc = tj == p4 && j == s;
          if (pr && pc)
            a[i][j] = -rd;
          else if (pr)
            a[i][j] = cj[j];
          else if (pc)
            a[i][j] = ci[i] * rd;
          else
            a[i][j] -= ci[i] * cj[j];
        }
    }
  }
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int r = 4 * ti + i, c = 4 * tj + j;
      D[r * NB + c] = -a[i][j];
      Ak[(long long)r * ld + c] = a[i][j];
    }
  if (!ok && threadIdx.x == 0) *bad = 1;
}

// A 16-row operand block of v_mfma_f64_16x16x4: lane l holds, of row l % 16,
// the 16 consecutive K values 16 (l / 16) .. of the 64 (A and B share this
// order of K, so the product is the same), read as eight 16-byte loads.
__device__ __forceinline__ void load_op(const double* __restrict__ rows, long long ld, int lane, double (&v)[16]) {
  const dvec2* p = reinterpret_cast<const dvec2*>(rows + (long long)(lane & 15) * ld + 16 * (lane >> 4));
#pragma unroll
  for (int q = 0; q < 8; q++) {
    const dvec2 t = p[q];
    v[2 * q] = t.x;
    v[2 * q + 1] = t.y;
  }
}

// Panel of block column k: P_i = A_ik (from the lower triangle), T_i = P_i D.
// Writes P (ld x 64), -T (ld x 64) and the swept panel entries into A.
__global__ __launch_bounds__(256) void k_sweep_panel(double* __restrict__ A, int ld, int k,
                                                     const double* __restrict__ D, double* __restrict__ P,
                                                     double* __restrict__ Tn) {
  __shared__ __align__(16) double sp[NB][NB + 2];
  const int i = blockIdx.x + (blockIdx.x >= (unsigned)k ? 1 : 0);  // every block row but k
  if (i > k) {
    const double* src = A + (long long)i * NB * ld + (long long)k * NB;
    for (int t = threadIdx.x; t < NB * NB; t += 256) sp[t >> 6][t & 63] = src[(long long)(t >> 6) * ld + (t & 63)];
  } else {
    const double* src = A + (long long)k * NB * ld + (long long)i * NB;
    for (int t = threadIdx.x; t < NB * NB; t += 256) sp[t & 63][t >> 6] = src[(long long)(t >> 6) * ld + (t & 63)];
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  for (int t = threadIdx.x; t < NB * NB; t += 256) P[(long long)i * NB * NB + t] = sp[t >> 6][t & 63];
  // wave w: rows 16 w .. 16 w + 15, all 64 columns
  double av[16];
  load_op(&sp[16 * w][0], NB + 2, lane, av);
  dvec4 acc[4];
#pragma unroll
  for (int c = 0; c < 4; c++) {
    acc[c] = dvec4{0.0, 0.0, 0.0, 0.0};
    double bv[16];
    load_op(D + 16 * c * NB, NB, lane, bv);  // D is symmetric
#pragma unroll
    for (int s = 0; s < 16; s++) acc[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[s], bv[s], acc[c], 0, 0, 0);
  }
  __syncthreads();
#pragma unroll
  for (int c = 0; c < 4; c++)
#pragma unroll
    for (int q = 0; q < 4; q++) sp[16 * w + 4 * q + (lane >> 4)][16 * c + (lane & 15)] = acc[c][q];
  __syncthreads();
  for (int t = threadIdx.x; t < NB * NB; t += 256) Tn[(long long)i * NB * NB + t] = -sp[t >> 6][t & 63];
  if (i > k) {
    double* dst = A + (long long)i * NB * ld + (long long)k * NB;
    for (int t = threadIdx.x; t < NB * NB; t += 256) dst[(long long)(t >> 6) * ld + (t & 63)] = sp[t >> 6][t & 63];
  } else {
    double* dst = A + (long long)k * NB * ld + (long long)i * NB;
    for (int t = threadIdx.x; t < NB * NB; t += 256) dst[(long long)(t >> 6) * ld + (t & 63)] = sp[t & 63][t >> 6];
  }
}

// A_ij += (-T_i) P_j^T for the blocks i >= j, neither of them k: a workgroup
// per 64 x 64 block, a wave per 32 x 32 quadrant, operands straight from L2
// (the panels are 2.9 MB each at n = 5577) in 16-byte loads, no barriers.
__global__ __launch_bounds__(256) void k_sweep_update(double* __restrict__ A, int ld, int k, int nb,
                                                      const double* __restrict__ P, const double* __restrict__ Tn) {
  // block pair of this workgroup: t counts the lower triangle of the nb - 1
  // remaining block rows, row by row
  const long long t = blockIdx.x;
  int r = (int)((sqrt(8.0 * (double)t + 1.0) - 1.0) * 0.5);
  while ((long long)(r + 1) * (r + 2) / 2 <= t) r++;
  while ((long long)r * (r + 1) / 2 > t) r--;
  int c = (int)(t - (long long)r * (r + 1) / 2);
  const int i = r + (r >= k ? 1 : 0), j = c + (c >= k ? 1 : 0);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int r0 = 32 * (w >> 1), c0 = 32 * (w & 1);
  double* C = A + ((long long)i * NB + r0) * ld + (long long)j * NB + c0;
  dvec4 acc[2][2];
#pragma unroll
  for (int x = 0; x < 2; x++)
#pragma unroll
    for (int y = 0; y < 2; y++)
#pragma unroll
      for (int q = 0; q < 4; q++)
        acc[x][y][q] = C[(long long)(16 * x + 4 * q + (lane >> 4)) * ld + 16 * y + (lane & 15)];
  const double* Ti = Tn + ((long long)i * NB + r0) * NB;
  const double* Pj = P + ((long long)j * NB + c0) * NB;
  double av[2][16], bv[2][16];
#pragma unroll
  for (int x = 0; x < 2; x++) load_op(Ti + 16 * x * NB, NB, lane, av[x]);
#pragma unroll
  for (int y = 0; y < 2; y++) load_op(Pj + 16 * y * NB, NB, lane, bv[y]);
#pragma unroll
  for (int s = 0; s < 16; s++)
#pragma unroll
    for (int x = 0; x < 2; x++)
#pragma unroll
      for (int y = 0; y < 2; y++)
        acc[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[x][s], bv[y][s], acc[x][y], 0, 0, 0);
#pragma unroll
  for (int x = 0; x < 2; x++)
#pragma unroll
    for (int y = 0; y < 2; y++)
#pragma unroll
      for (int q = 0; q < 4; q++)
        C[(long long)(16 * x + 4 * q + (lane >> 4)) * ld + 16 * y + (lane & 15)] = acc[x][y][q];
}

// A <- -A from the lower triangle, both triangles, with an FP32 copy (Af null:
// without).
__global__ __launch_bounds__(256) void k_sweep_finish(double* __restrict__ A, float* __restrict__ Af, int ld) {
  __shared__ double sp[NB][NB + 1];
  const long long t = blockIdx.x;
  int r = (int)((sqrt(8.0 * (double)t + 1.0) - 1.0) * 0.5);
  while ((long long)(r + 1) * (r + 2) / 2 <= t) r++;
  while ((long long)r * (r + 1) / 2 > t) r--;
  const int i = r, j = (int)(t - (long long)r * (r + 1) / 2);
  const long long lo = (long long)i * NB * ld + (long long)j * NB, up = (long long)j * NB * ld + (long long)i * NB;
  for (int q = threadIdx.x; q < NB * NB; q += 256) sp[q >> 6][q & 63] = -A[lo + (long long)(q >> 6) * ld + (q & 63)];
  __syncthreads();
  for (int q = threadIdx.x; q < NB * NB; q += 256) {
    const int a = q >> 6, b = q & 63;
    const double v = i == j && a < b ? sp[b][a] : sp[a][b];
    A[lo + (long long)a * ld + b] = v;
    if (Af) Af[lo + (long long)a * ld + b] = (float)v;
    if (i != j) {
      A[up + (long long)a * ld + b] = sp[b][a];
      if (Af) Af[up + (long long)a * ld + b] = (float)sp[b][a];
    }
  }
}

}  // namespace

void launch_dense_assemble(const Geo& g, const double* Mom, const int* pos, int nf, int ld, double* A,
                           hipStream_t st) {
  const long long n2 = (long long)ld * ld / 2;
  long long gb = (n2 + kBlock - 1) / kBlock;
  if (gb > 8192) gb = 8192;
  hipLaunchKernelGGL(k_dense_clear, dim3((unsigned)gb), dim3(kBlock), 0, st, A, nf, ld);
  launch_dense_elements(g, Mom, pos, ld, A, st);
}

void launch_spd_inverse(double* A, float* Af, int ld, double* work, int* bad, hipStream_t st) {
  const int nb = ld / NB;
  double* P = work;
  double* Tn = P + (long long)ld * NB;
  double* D = Tn + (long long)ld * NB;
  const unsigned pairs = (unsigned)((long long)(nb - 1) * nb / 2);
  for (int k = 0; k < nb; k++) {
    hipLaunchKernelGGL(k_sweep_diag, dim3(1), dim3(256), 0, st, A, ld, k, D, bad);
    if (nb == 1) break;
    hipLaunchKernelGGL(k_sweep_panel, dim3(nb - 1), dim3(256), 0, st, A, ld, k, D, P, Tn);
    hipLaunchKernelGGL(k_sweep_update, dim3(pairs), dim3(256), 0, st, A, ld, k, nb, P, Tn);
  }
  hipLaunchKernelGGL(k_sweep_finish, dim3((unsigned)((long long)nb * (nb + 1) / 2)), dim3(256), 0, st, A, Af, ld);
}

}  // namespace gs
