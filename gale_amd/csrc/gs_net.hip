// gs_net.hip -- BF16 matrix-core kernels of the learned Schur-complement
// preconditioner network (forward, data gradient, weight gradient), its
// pooling / upsampling / loss kernels and the Adam optimiser.
//
// Convolutions are implicit GEMMs on the BF16 matrix cores: a wavefront
// computes 16 consecutive voxels (flat index over batch x grid) times all
// output channels; the K dimension is the flattened (tap, input channel)
// index kk = tap*Cin + ci, consumed KW at a time -- 32 with gfx950's
// v_mfma_f32_16x16x32_bf16 wherever Cin is a multiple of 8 (the forward
// passes), else 16 with v_mfma_f32_16x16x16_bf16.  Lane l holds the KW/4 K
// values KW/4 (l/16) .. of a step for row l%16 of A and column l%16 of B, and
// receives D[4(l/16)+i][l%16], i = 0..3 (a product over K does not depend on
// the order in which A and B share K).  Weights are pre-packed into exactly
// that per-lane B order, so a lane's B operand is one 8- or 16-byte load;
// with Cin a multiple of KW/4 a lane's A values are consecutive channels of
// one neighbour voxel (one load of the same width).
#include "gs_net.h"

#include <math.h>
#include <string.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../../include/gale_stokes.h"
#include "gs_reduce.h"

namespace gs {
namespace net {

typedef short s4 __attribute__((ext_vector_type(4)));
typedef short s8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf8v __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));

// One K step of the implicit GEMM (16 or 32 K values) on the matrix cores.
__device__ __forceinline__ f4 mfma_bf16(const s4& a, const s4& b, const f4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f4 mfma_bf16(const s8& a, const s8& b, const f4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8v, a), __builtin_bit_cast(bf8v, b), c, 0, 0,
                                                 0);
}
template <int KW>
struct KOp {
  typedef s4 type;
};
template <>
struct KOp<32> {
  typedef s8 type;
};

static LayerSpec make_layer(int l) {
  // encoder / bottom
  if (l < 2 * kLevels) {
    const int lev = l / 2;
    const bool a = (l % 2) == 0;
    if (a) {
      const int cin = lev == 0 ? 4 : kChan[lev - 1];
      return LayerSpec{cin, kChan[lev], lev, 1, lev == 0 ? 2 : cin};
    }
    const int cout = lev == kLevels - 1 ? kChan[kLevels - 2] : kChan[lev];
    return LayerSpec{kChan[lev], cout, lev, 1, kChan[lev]};
  }
  // decoder
  const int k = l - 2 * kLevels;
  const int lev = kLevels - 2 - k / 2;
  if ((k % 2) == 0) return LayerSpec{kChan[lev], kChan[lev], lev, 1, kChan[lev]};
  return lev == 0 ? LayerSpec{kChan[0], 1, 0, 0, kChan[0]} : LayerSpec{kChan[lev], kChan[lev - 1], lev, 1, kChan[lev]};
}

static const LayerSpec* build_spec() {
  static LayerSpec t[kLayers];
  for (int l = 0; l < kLayers; l++) t[l] = make_layer(l);
  return t;
}
const LayerSpec* const kSpec = build_spec();

long long weight_offset(int l) {
  long long o = 0;
  for (int i = 0; i < l; i++) o += 27LL * kSpec[i].cin * kSpec[i].cout + kSpec[i].cout;
  return o;
}
long long bias_offset(int l) { return weight_offset(l) + 27LL * kSpec[l].cin * kSpec[l].cout; }
long long num_params() { return weight_offset(kLayers); }

static inline int kchunks(int cin) { return (27 * cin + 15) / 16; }
static inline int kchunks32(int cin) { return (27 * cin + 31) / 32; }
static inline int ntiles(int cout) { return (cout + 15) / 16; }

#define NCK(x)                                                                                        \
  do {                                                                                                \
    hipError_t e_ = (x);                                                                              \
    if (e_ != hipSuccess) {                                                                           \
      std::fprintf(stderr, "gale_stokes(net): HIP error %s at %s:%d\n", hipGetErrorString(e_), __FILE__, \
                   __LINE__);                                                                         \
      return GS_E_HIP;                                                                                \
    }                                                                                                 \
  } while (0)

// ---------------------------------------------------------------------------
// BF16 helpers (round to nearest even; NaN kept quiet)
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint16_t f2bf(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return 0x7fc0;
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

__device__ __forceinline__ void vox_xyz(long long vox, long long V, int nx, int ny, long long* b, int* x, int* y,
                                        int* z) {
  const long long bb = vox / V;
  const long long v = vox - bb * V;
  *b = bb;
  *x = (int)(v % nx);
  const long long t = v / nx;
  *y = (int)(t % ny);
  *z = (int)(t / ny);
}

// ---------------------------------------------------------------------------
// Convolution (forward and data gradient share this kernel)
// ---------------------------------------------------------------------------
// out[vox][co] = act(bias[co] + sum_kk in[nbr(vox, tap(kk))][ci(kk)] * W[kk][co])
// Wp: packed [KC][NT][64 lanes] of KW/4 BF16.  Grid: ceil(BV/64) blocks x 256.
template <int CIN, int NT, bool OUT_F32, int KW>
__global__ __launch_bounds__(256) void k_conv(const uint16_t* __restrict__ in,
                                              const typename KOp<KW>::type* __restrict__ Wp,
                                              const float* __restrict__ bias, void* __restrict__ out,
                                              int cout_store, int nx, int ny, int nz, long long BV, int relu) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const long long v0 = ((long long)blockIdx.x * 4 + wave) * 16;
  if (v0 >= BV) return;
  const int row = lane & 15, kg = lane >> 4;
  const long long V = (long long)nx * ny * nz;
  const long long vox = v0 + row;
  const bool valid = vox < BV;
  long long b = 0;
  int x = 0, y = 0, z = 0;
  if (valid) vox_xyz(vox, V, nx, ny, &b, &x, &y, &z);
  const long long bbase = b * V;
  f4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; t++) acc[t] = f4{0.f, 0.f, 0.f, 0.f};
  typedef typename KOp<KW>::type AT;
  constexpr int KT = 27 * CIN;
  constexpr int KC = (KT + KW - 1) / KW;
  // K steps in groups of U: all operand loads of a group are issued before
  // its MFMAs, so a wave keeps U x (1 + NT) loads in flight instead of
  // waiting on one load per step.
  constexpr int U = KC < 9 ? KC : 9;
  for (int kc0 = 0; kc0 < KC; kc0 += U) {
    AT a[U];
    AT w[U][NT];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int kc = kc0 + u;
      const int kk = kc * KW + kg * (KW / 4);
      a[u] = AT{};
      if (valid && kc < KC && kk < KT) {
        const int tap = kk / CIN;
        const int ci = kk - tap * CIN;
        const int xx = x + tap % 3 - 1, yy = y + (tap / 3) % 3 - 1, zz = z + tap / 9 - 1;
        if (xx >= 0 && xx < nx && yy >= 0 && yy < ny && zz >= 0 && zz < nz) {
          const long long nb = bbase + xx + (long long)nx * (yy + (long long)ny * zz);
          a[u] = *reinterpret_cast<const AT*>(in + nb * CIN + ci);
        }
      }
#pragma unroll
      for (int t = 0; t < NT; t++) w[u][t] = kc < KC ? Wp[(kc * NT + t) * 64 + lane] : AT{};
    }
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int t = 0; t < NT; t++) acc[t] = mfma_bf16(a[u], w[u][t], acc[t]);
  }
#pragma unroll
  for (int t = 0; t < NT; t++) {
    const int co = t * 16 + row;
    if (co >= cout_store) continue;
    const float bv = bias ? bias[co] : 0.f;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const long long vo = v0 + kg * 4 + i;
      if (vo >= BV) continue;
      float val = acc[t][i] + bv;
      if (relu) val = fmaxf(val, 0.f);
      if (OUT_F32)
        reinterpret_cast<float*>(out)[vo * cout_store + co] = val;
      else
        reinterpret_cast<uint16_t*>(out)[vo * cout_store + co] = f2bf(val);
    }
  }
}

// Split-K form of k_conv for the small levels, where a wave per 16 voxels
// leaves most of the chip idle and each wave would walk all 27 x CIN / 16 K
// steps in sequence: S waves share one 16-voxel tile, wave w taking K steps
// in groups of four interleaved with the others, and their partial sums are
// added in wave order through LDS.
template <int CIN, int NT, bool OUT_F32, int S, int KW>
__global__ __launch_bounds__(64 * S) void k_conv_splitk(const uint16_t* __restrict__ in,
                                                        const typename KOp<KW>::type* __restrict__ Wp,
                                                        const float* __restrict__ bias, void* __restrict__ out,
                                                        int cout_store, int nx, int ny, int nz, long long BV,
                                                        int relu) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const long long v0 = (long long)blockIdx.x * 16;
  const int row = lane & 15, kg = lane >> 4;
  const long long V = (long long)nx * ny * nz;
  const long long vox = v0 + row;
  const bool valid = vox < BV;
  long long b = 0;
  int x = 0, y = 0, z = 0;
  if (valid) vox_xyz(vox, V, nx, ny, &b, &x, &y, &z);
  const long long bbase = b * V;
  f4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; t++) acc[t] = f4{0.f, 0.f, 0.f, 0.f};
  typedef typename KOp<KW>::type AT;
  constexpr int KT = 27 * CIN;
  constexpr int KC = (KT + KW - 1) / KW;
  constexpr int U = 4;
  for (int kc0 = w * U; kc0 < KC; kc0 += S * U) {
    AT a[U];
    AT wv[U][NT];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int kc = kc0 + u;
      const int kk = kc * KW + kg * (KW / 4);
      a[u] = AT{};
      if (valid && kc < KC && kk < KT) {
        const int tap = kk / CIN;
        const int ci = kk - tap * CIN;
        const int xx = x + tap % 3 - 1, yy = y + (tap / 3) % 3 - 1, zz = z + tap / 9 - 1;
        if (xx >= 0 && xx < nx && yy >= 0 && yy < ny && zz >= 0 && zz < nz) {
          const long long nb = bbase + xx + (long long)nx * (yy + (long long)ny * zz);
          a[u] = *reinterpret_cast<const AT*>(in + nb * CIN + ci);
        }
      }
#pragma unroll
      for (int t = 0; t < NT; t++) wv[u][t] = kc < KC ? Wp[(kc * NT + t) * 64 + lane] : AT{};
    }
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int t = 0; t < NT; t++) acc[t] = mfma_bf16(a[u], wv[u][t], acc[t]);
  }
  __shared__ f4 red[S][NT][64];
#pragma unroll
  for (int t = 0; t < NT; t++) red[w][t][lane] = acc[t];
  __syncthreads();
  if (w != 0) return;
#pragma unroll
  for (int t = 0; t < NT; t++) {
    f4 sum = red[0][t][lane];
    for (int ww = 1; ww < S; ww++) sum += red[ww][t][lane];
    const int co = t * 16 + row;
    if (co >= cout_store) continue;
    const float bv = bias ? bias[co] : 0.f;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const long long vo = v0 + kg * 4 + i;
      if (vo >= BV) continue;
      float val = sum[i] + bv;
      if (relu) val = fmaxf(val, 0.f);
      if (OUT_F32)
        reinterpret_cast<float*>(out)[vo * cout_store + co] = val;
      else
        reinterpret_cast<uint16_t*>(out)[vo * cout_store + co] = f2bf(val);
    }
  }
}

// LDS-tiled form of k_conv for the large levels (CIN a multiple of 4, of 8
// on the 32-wide step; nx, ny, nz multiples of 16, 4, 4).  A block computes a 16 x 4 x 4 voxel tile:
// it stages the 18 x 6 x 6 input box (zero outside the grid) in LDS once, and
// each wave takes the four x-rows of one z-slice, so every input voxel is
// read from memory once per tile instead of once per tap.  The K steps and
// their order per output are those of k_conv (identical results).
template <int CIN, int NT, bool OUT_F32, int KW>
__global__ __launch_bounds__(256) void k_conv_tiled(const uint16_t* __restrict__ in,
                                                    const typename KOp<KW>::type* __restrict__ Wp,
                                                    const float* __restrict__ bias, void* __restrict__ out,
                                                    int cout_store, int nx, int ny, int nz, int relu) {
  typedef typename KOp<KW>::type AT;
  constexpr int BX = 18, BY = 6, BZ = 6, NBOX = BX * BY * BZ;
  constexpr int KT = 27 * CIN;
  constexpr int KC = (KT + KW - 1) / KW;  // K steps (with KW = 32 and CIN = 16 a step spans two taps)
  constexpr int Q = CIN / 4;              // s4 chunks per voxel
  constexpr int STG = 4 * 4 * 16 * NT * 16 / 4;  // output staging (s4 units), reuses the box
  __shared__ __align__(16) s4 box[NBOX * Q > STG ? NBOX * Q : STG];
  const int tx = nx / 16, ty = ny / 4, tz = nz / 4;
  long long t = blockIdx.x;
  const int bx = (int)(t % tx);
  t /= tx;
  const int by = (int)(t % ty);
  t /= ty;
  const int bz = (int)(t % tz);
  const long long b = t / tz;
  const int x0 = bx * 16, y0 = by * 4, z0 = bz * 4;
  const long long bbase = b * (long long)nx * ny * nz;
  // A thread's pieces of the box are all requested before the first is
  // written to LDS, and the first weights before the barrier; the K loop is
  // unrolled, so that a step's place in the box costs at most three selects
  // instead of divisions.  16 to 16 channels at 96^3: 30.2 -> 25.4 us, the
  // network there 342 -> 315 us (57 MB in and out: 11 us at the copy rate).
  constexpr int PS = Q % 2 == 0 ? 8 : 4;  // channels of a piece: 16 bytes where a voxel holds a whole number of them
  typedef short piece_t __attribute__((ext_vector_type(PS)));
  constexpr int QP = CIN / PS, NP = (NBOX * QP + 255) / 256;
  const piece_t* inp = reinterpret_cast<const piece_t*>(in);
  piece_t* boxp = reinterpret_cast<piece_t*>(box);
  piece_t pv[NP];
  bool pin[NP];
#pragma unroll
  for (int i = 0; i < NP; i++) {
    const int q = threadIdx.x + 256 * i;
    const int c = q % QP, vx = q / QP;
    const int xx = vx % BX, yy = (vx / BX) % BY, zz = vx / (BX * BY);
    const int gx = x0 - 1 + xx, gy = y0 - 1 + yy, gz = z0 - 1 + zz;
    pin[i] = vx < NBOX && gx >= 0 && gx < nx && gy >= 0 && gy < ny && gz >= 0 && gz < nz;
    pv[i] = inp[pin[i] ? (bbase + gx + (long long)nx * (gy + (long long)ny * gz)) * QP + c : 0];
  }
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int row = lane & 15, kg = lane >> 4;
  // K steps in batches of U, the next batch's weights in flight
  constexpr int U = NT == 1 ? 9 : (NT == 2 ? 5 : 3), NBATCH = (KC + U - 1) / U;
  AT wv[2][U][NT];
  auto load_w = [&](int n) {
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int v = 0; v < NT; v++)
        if (n * U + u < KC) wv[n & 1][u][v] = Wp[((n * U + u) * NT + v) * 64 + lane];
  };
  load_w(0);
#pragma unroll
  for (int i = 0; i < NP; i++) {
    const int q = threadIdx.x + 256 * i;
    if (q < NBOX * QP) boxp[q] = pin[i] ? pv[i] : piece_t{};
  }
  __syncthreads();
  f4 acc[4][NT];
#pragma unroll
  for (int j = 0; j < 4; j++)
#pragma unroll
    for (int u = 0; u < NT; u++) acc[j][u] = f4{0.f, 0.f, 0.f, 0.f};
  constexpr bool kOneTap = CIN % KW == 0;  // a K step lies in one tap
  const s4* bw = box + (w * BY * BX + row) * Q + (kOneTap ? kg * (KW / 16) : 0);
#pragma unroll
  for (int n = 0; n < NBATCH; n++) {
    if (n + 1 < NBATCH) load_w(n + 1);
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int kc = n * U + u;
      if (kc >= KC) break;
      // this lane's first K index of the step is kc KW + kg KW / 4: its place
      // in the box is one of four constants (linear in kg within a tap)
      auto place = [&](int g) {
        const int kk = kc * KW + g * (KW / 4), tap = kk / CIN;
        return ((tap / 9 * BY + tap / 3 % 3) * BX + tap % 3) * Q + (kk - tap * CIN) / 4;
      };
      auto in_k = [&](int g) { return kc * KW + g * (KW / 4) < KT; };
      int o = place(0);
      bool ok = true;
#pragma unroll
      for (int g = 1; g < (kOneTap ? 1 : 4); g++) {
        if (in_k(g)) o = kg >= g ? place(g) : o;
        if (!in_k(g)) ok = ok && kg != g;
      }
#pragma unroll
      for (int j = 0; j < 4; j++) {
        AT a = *reinterpret_cast<const AT*>(bw + o + j * BX * Q);
        if (!ok) a = AT{};
#pragma unroll
        for (int v = 0; v < NT; v++) acc[j][v] = mfma_bf16(a, wv[n & 1][u][v], acc[j][v]);
      }
    }
  }
  if (!OUT_F32 && cout_store == NT * 16) {
    // BF16 output of every channel: the wave's 64 voxels x NT*16 channels
    // go through LDS (the box is free once every wave is past its K loop)
    // and leave as 16-byte stores of whole voxel rows, instead of one
    // 2-byte store per lane per voxel (same values, 10 % less time)
    __syncthreads();
    uint16_t* stg = reinterpret_cast<uint16_t*>(box) + w * (4 * 16 * NT * 16);
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
      for (int v = 0; v < NT; v++) {
        const int co = v * 16 + row;
        const float bv = bias ? bias[co] : 0.f;
#pragma unroll
        for (int i = 0; i < 4; i++) {
          float val = acc[j][v][i] + bv;
          if (relu) val = fmaxf(val, 0.f);
          stg[(j * 16 + kg * 4 + i) * (NT * 16) + co] = f2bf(val);
        }
      }
    __syncthreads();
    const s8* st8 = reinterpret_cast<const s8*>(stg);
    constexpr int CH8 = NT * 2;  // 16-byte pieces per voxel
    for (int c = lane; c < 4 * 16 * CH8; c += 64) {
      const int vx = c / CH8, part = c - vx * CH8;
      const int j = vx / 16, xx = vx - j * 16;
      const long long vo = bbase + (x0 + xx) + (long long)nx * ((y0 + j) + (long long)ny * (z0 + w));
      reinterpret_cast<s8*>(reinterpret_cast<uint16_t*>(out) + vo * cout_store)[part] = st8[c];
    }
    return;
  }
#pragma unroll
  for (int j = 0; j < 4; j++)
#pragma unroll
    for (int v = 0; v < NT; v++) {
      const int co = v * 16 + row;
      if (co >= cout_store) continue;
      const float bv = bias ? bias[co] : 0.f;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const long long vo = bbase + (x0 + kg * 4 + i) + (long long)nx * ((y0 + j) + (long long)ny * (z0 + w));
        float val = acc[j][v][i] + bv;
        if (relu) val = fmaxf(val, 0.f);
        if (OUT_F32)
          reinterpret_cast<float*>(out)[vo * cout_store + co] = val;
        else
          reinterpret_cast<uint16_t*>(out)[vo * cout_store + co] = f2bf(val);
      }
    }
}

// ---------------------------------------------------------------------------
// Weight gradient
// ---------------------------------------------------------------------------
// dW[tap][ci][co] = sum_vox X[vox + off(tap)][ci] G[vox][co] is a matrix
// product over voxels, so both operands are first laid out channel by channel
// (voxels contiguous) on the grid padded by one voxel per side and with zero
// halos: then a tap is a constant shift of the flat voxel index, no bounds are
// tested, and a lane's eight K values are one 16-byte load.  Halo terms are
// exact zeros (G is zero there).
//
// k_pad_t: out[c * stride + p] = in[vox(p)][c] for the C channels of a
// channels-last tensor with cs stored channels; zero on the halo, up to
// stride, and for `margin` entries after the last row (the shifted loads of
// the last row run over into them).  A block moves kPadVox voxels through
// LDS, a thread's pieces in flight together (in four rounds of 64 voxels, each
// waiting for its loads, the 36 calls of a backward pass took 10.9 us on
// average, and now 7.0).  With bpart, also the block's sum of every channel:
// the bias gradient as a by-product.
constexpr int kPadVox = 256;
inline unsigned pad_lds(int cs) { return kPadVox * (cs + 2) * sizeof(uint16_t); }
__global__ __launch_bounds__(256) void k_pad_t(const uint16_t* __restrict__ in, int cs, int C,
                                               uint16_t* __restrict__ out, long long stride, int margin, int nx,
                                               int ny, int nz, int B, float* __restrict__ bpart) {
  extern __shared__ __align__(16) uint16_t tile[];
  __shared__ long long src[kPadVox];
  __shared__ float bsum[kPadVox / 64][96];
  const int ld = cs + 2, C4 = cs / 4;
  const unsigned w = nx + 2, h = ny + 2, d = nz + 2, pv = w * h * d;
  if (blockIdx.x == gridDim.x - 1) {  // the margin after the last row
    for (int i = threadIdx.x; i < margin; i += 256) out[(long long)C * stride + i] = 0;
    return;
  }
  const long long p0 = (long long)blockIdx.x * kPadVox;
  {
    const long long p = p0 + threadIdx.x;
    const long long b = p / pv;
    const unsigned q = (unsigned)(p - b * pv);
    const int x = (int)(q % w) - 1, y = (int)((q / w) % h) - 1, z = (int)(q / (w * h)) - 1;
    const bool in_grid = b < B && x >= 0 && x < nx && y >= 0 && y < ny && z >= 0 && z < nz;
    src[threadIdx.x] = in_grid ? ((b * nz + z) * ny + y) * (long long)nx + x : -1;
  }
  __syncthreads();
  // kPadVox * C4 pieces are C4 a thread
  for (int i0 = 0; i0 < C4; i0 += 4) {
    s4 val[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      val[i] = s4{0, 0, 0, 0};
      if (i0 + i < C4) {
        const int q = (i0 + i) * 256 + threadIdx.x, v = q / C4, part = q - v * C4;
        const long long sv = src[v];
        if (sv >= 0) val[i] = reinterpret_cast<const s4*>(in + sv * cs)[part];
      }
    }
#pragma unroll
    for (int i = 0; i < 4; i++)
      if (i0 + i < C4) {
        const int q = (i0 + i) * 256 + threadIdx.x, v = q / C4, part = q - v * C4;
        // rows of an odd number of dwords: two dword writes
        unsigned* t = reinterpret_cast<unsigned*>(tile + v * ld + part * 4);
        const uint2 u = __builtin_bit_cast(uint2, val[i]);
        t[0] = u.x;
        t[1] = u.y;
      }
  }
  __syncthreads();
  // eight lanes write 64 voxels of a channel: a whole line
  for (int q = threadIdx.x; q < C * (kPadVox / 8); q += 256) {
    const int r = q >> 3, sub = r / C, c = r - sub * C, v0 = sub * 64 + (q & 7) * 8;
    s8 o;
    float bs = 0.f;
#pragma unroll
    for (int k = 0; k < 8; k++) {
      o[k] = (short)tile[(v0 + k) * ld + c];
      bs += bf2f((uint16_t)o[k]);
    }
    // stride is a multiple of 32, so whole 8-voxel pieces lie inside it
    if (p0 + v0 < stride) *reinterpret_cast<s8*>(out + (long long)c * stride + p0 + v0) = o;
    if (bpart) {  // C * 32 is a multiple of 32, so eight lanes of a sum are here together
#pragma unroll
      for (int m = 1; m < 8; m <<= 1) bs += __shfl_xor(bs, m, 64);
      if ((q & 7) == 0) bsum[sub][c] = bs;
    }
  }
  if (!bpart) return;
  __syncthreads();
  if ((int)threadIdx.x < C) {
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < kPadVox / 64; k++) s += bsum[k][threadIdx.x];
    bpart[(long long)blockIdx.x * C + threadIdx.x] = s;
  }
}

// gb[co] = sum over the blocks' partial sums, one block per channel.
__global__ void k_bgrad_reduce(const float* __restrict__ bpart, int n, int C, float* __restrict__ gb) {
  __shared__ float sh[kBlock / 64];
  const int co = blockIdx.x;
  float v = 0.f;
  for (int k = threadIdx.x; k < n; k += blockDim.x) v += bpart[(long long)k * C + co];
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    float t = 0.f;
    for (int k = 0; k < (int)(blockDim.x >> 6); k++) t += sh[k];
    gb[co] = t;
  }
}

// P[group][(tap * cin + ci)][co] over the group's share of the voxels: block
// (m tile, dy, dz) x group, its four waves a quarter of the group each, three
// taps (dx) x NT column tiles of 16x16 accumulators a wave.  Per 32-voxel K
// step a wave loads a row's eight values with the dwords before and after
// them and NT 16-byte pieces of G for 3 NT v_mfma_f32_16x16x32_bf16, the next
// step's in flight; the taps dx = -1, 1 are those values shifted by 16 bits.
// Loading each tap instead (16 bytes from an odd element) was what bounded
// the kernel: for eight 32^3 samples the 16-channel layers took 110 us and
// now take 38, the 32-channel ones 29 and 14.  Neither whole 128-byte lines
// per row nor keeping the nine blocks of a group on one XCD changed it.
typedef unsigned u4 __attribute__((ext_vector_type(4)));
typedef u4 u4u __attribute__((aligned(2)));  // a tap's shift leaves 4-byte alignment, 2-byte on a grid of odd width
typedef unsigned u1u __attribute__((aligned(2)));
template <int NT>
__global__ __launch_bounds__(256) void k_wgrad(const uint16_t* __restrict__ X, const uint16_t* __restrict__ G,
                                               long long stride, int cin, int cout, int w, int pl, long long kper,
                                               float* __restrict__ partial) {
  __shared__ f4 red[4][NT][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int mt = blockIdx.x / 9, yz = blockIdx.x - 9 * mt;
  const int row = lane & 15, kg = lane >> 4;
  const int off = (yz % 3 - 1) * w + (yz / 3 - 1) * pl;
  const long long k0 = ((long long)blockIdx.y * 4 + wave) * kper;
  const long long k1 = k0 + kper < stride ? k0 + kper : stride;
  const uint16_t* xa = X + (long long)(mt * 16 + row) * stride + 8 * kg + off;
  const uint16_t* gb = G + (long long)row * stride + 8 * kg;
  f4 acc[3][NT];
#pragma unroll
  for (int q = 0; q < 3; q++)
#pragma unroll
    for (int t = 0; t < NT; t++) acc[q][t] = f4{0.f, 0.f, 0.f, 0.f};
  // the eight values of the middle tap and the dwords before and after them
  u4 a;
  unsigned al, ar;
  s8 g[NT];
  auto load = [&](long long k) {
    a = *reinterpret_cast<const u4u*>(xa + k);
    al = *reinterpret_cast<const u1u*>(xa + k - 2);
    ar = *reinterpret_cast<const u1u*>(xa + k + 8);
#pragma unroll
    for (int t = 0; t < NT; t++) g[t] = *reinterpret_cast<const s8*>(gb + (long long)t * 16 * stride + k);
  };
  if (k0 < k1) load(k0);
  for (long long k = k0; k < k1; k += 32) {
    s8 ac[3], gc[NT];
    u4 lo, hi;  // the values shifted by one voxel either way
#pragma unroll
    for (int i = 0; i < 4; i++) {
      lo[i] = __builtin_amdgcn_alignbit(a[i], i ? a[i ? i - 1 : 0] : al, 16);
      hi[i] = __builtin_amdgcn_alignbit(i < 3 ? a[i < 3 ? i + 1 : 3] : ar, a[i], 16);
    }
    ac[0] = __builtin_bit_cast(s8, lo);
    ac[1] = __builtin_bit_cast(s8, a);
    ac[2] = __builtin_bit_cast(s8, hi);
#pragma unroll
    for (int t = 0; t < NT; t++) gc[t] = g[t];
    if (k + 32 < k1) load(k + 32);
#pragma unroll
    for (int q = 0; q < 3; q++)
#pragma unroll
      for (int t = 0; t < NT; t++) acc[q][t] = mfma_bf16(ac[q], gc[t], acc[q][t]);
  }
  float* P = partial + (long long)blockIdx.y * 27 * cin * cout;
#pragma unroll
  for (int q = 0; q < 3; q++) {
#pragma unroll
    for (int t = 0; t < NT; t++) red[wave][t][lane] = acc[q][t];
    __syncthreads();
    for (int e = threadIdx.x; e < NT * 64; e += 256) {
      const int t = e >> 6, l = e & 63;
      const f4 s = ((red[0][t][l] + red[1][t][l]) + red[2][t][l]) + red[3][t][l];
      const int co = t * 16 + (l & 15), tap = yz * 3 + q;
      if (co < cout)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const int ci = mt * 16 + 4 * (l >> 4) + i;
          if (ci < cin) P[((long long)tap * cin + ci) * cout + co] = s[i];
        }
    }
    __syncthreads();
  }
}

// grad W = sum over the groups (fixed order).
__global__ void k_wgrad_reduce(const float* __restrict__ partial, int ngroup, long long n, float* __restrict__ gw) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
    float s = 0.f;
#pragma unroll 8
    for (int c = 0; c < ngroup; c++) s += partial[(long long)c * n + i];
    gw[i] = s;
  }
}

// Weight packing.  Forward: B[kk][co] = W[kk][co].  Transposed (data
// gradient of a layer with cin -> cout): the convolution runs cout -> cin with
// B[kk'][c] where kk' = tap'*cout_in + co, B = W[(26 - tap')*cin + c][co].
__global__ void k_pack(const float* __restrict__ W, int cin, int cout, int transpose, int cin_g, int nt, int kc,
                       s4* __restrict__ out) {
  // cin_g: input channels of the packed GEMM; nt: its N tiles; kc: its K chunks
  const long long n = (long long)kc * nt * 64;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
    const int lane = (int)(i % 64);
    const long long r = i / 64;
    const int t = (int)(r % nt), c = (int)(r / nt);
    const int col = t * 16 + (lane & 15);
    s4 v = s4{0, 0, 0, 0};
    for (int j = 0; j < 4; j++) {
      const int kk = c * 16 + (lane >> 4) * 4 + j;
      if (kk >= 27 * cin_g) continue;
      const int tap = kk / cin_g, ci = kk - tap * cin_g;
      float w = 0.f;
      if (!transpose) {
        if (col < cout) w = W[(long long)kk * cout + col];
      } else {
        // ci indexes the forward layer's outputs, col its inputs
        if (ci < cout && col < cin) w = W[(long long)((26 - tap) * cin + col) * cout + ci];
      }
      v[j] = (short)f2bf(w);
    }
    out[i] = v;
  }
}

// Forward weights for the 32-wide K step: lane l of chunk c, tile t holds
// B[c*32 + 8(l/16) + j][t*16 + l%16], j = 0..7.  The 32-wide step halves the
// matrix-core instructions and operand loads (measured at 96^3: the 48^3
// convolutions 37.8 -> 22.6 us, the 96^3 ones 37.3 -> 36.1 us, the network
// 0.48 -> about 0.37 ms per application).  It regroups the FP32 partial sums,
// which flips some of the BF16 roundings of the activations between layers:
// on a 48^3 input the two widths differ by 3.5e-3 relative, as far as either
// is from the numpy oracle.  The learned solve's iteration count moves by up
// to 30 % either way with such changes, so the two widths were compared over
// ten 96^3 fields of the generator: 19.83 s (32) against 20.59 s (16) in
// total, 5 % less time per Uzawa iteration, faster on eight.  The 32-wide
// step is the default; GALE_LPC_K32=0 selects the 16-wide one.
__global__ void k_pack32(const float* __restrict__ W, int cin, int cout, int nt, int kc, s8* __restrict__ out) {
  const long long n = (long long)kc * nt * 64;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
    const int lane = (int)(i % 64);
    const long long r = i / 64;
    const int t = (int)(r % nt), c = (int)(r / nt);
    const int col = t * 16 + (lane & 15);
    s8 v = s8{};
    for (int j = 0; j < 8; j++) {
      const int kk = c * 32 + (lane >> 4) * 8 + j;
      if (kk < 27 * cin && col < cout) v[j] = (short)f2bf(W[(long long)kk * cout + col]);
    }
    out[i] = v;
  }
}

// ---------------------------------------------------------------------------
// elementwise kernels
// ---------------------------------------------------------------------------
__global__ void k_pack_input(const float* __restrict__ in2, uint16_t* __restrict__ x4, long long BV) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < BV; i += (long long)gridDim.x * blockDim.x) {
    x4[i * 4 + 0] = f2bf(in2[i * 2 + 0]);
    x4[i * 4 + 1] = f2bf(in2[i * 2 + 1]);
    x4[i * 4 + 2] = 0;
    x4[i * 4 + 3] = 0;
  }
}
__global__ void k_pack_gout(const float* __restrict__ g, uint16_t* __restrict__ g4, long long BV) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < BV; i += (long long)gridDim.x * blockDim.x) {
    g4[i * 4 + 0] = f2bf(g[i]);
    g4[i * 4 + 1] = 0;
    g4[i * 4 + 2] = 0;
    g4[i * 4 + 3] = 0;
  }
}

// 2x2x2 average pool: fine (nx,ny,nz) -> coarse (nx/2, ny/2, nz/2).
// 2x2x2 average pool; four channels (one 8-byte word) per thread, C % 4 == 0.
__global__ void k_pool(const uint16_t* __restrict__ in, uint16_t* __restrict__ out, int C, int nx, int ny, int nz,
                       long long Bc) {
  const int cx = nx / 2, cy = ny / 2, cz = nz / 2;
  const long long Vc = (long long)cx * cy * cz, Vf = (long long)nx * ny * nz;
  const int C4 = C / 4;
  const long long n = Bc * Vc * C4;
  const s4* in4 = reinterpret_cast<const s4*>(in);
  s4* out4 = reinterpret_cast<s4*>(out);
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
    const int c = (int)(i % C4);
    const long long vv = i / C4;
    long long b;
    int x, y, z;
    vox_xyz(vv, Vc, cx, cy, &b, &x, &y, &z);
    float s[4] = {0.f, 0.f, 0.f, 0.f};
    for (int a = 0; a < 8; a++) {
      const long long f = b * Vf + (2 * x + (a & 1)) + (long long)nx * ((2 * y + ((a >> 1) & 1)) +
                                                                       (long long)ny * (2 * z + ((a >> 2) & 1)));
      const s4 v = in4[f * C4 + c];
#pragma unroll
      for (int k = 0; k < 4; k++) s[k] += bf2f((uint16_t)v[k]);
    }
    s4 o;
#pragma unroll
    for (int k = 0; k < 4; k++) o[k] = (short)f2bf(s[k] * 0.125f);
    out4[i] = o;
  }
}

// out[fine] = up(coarse)[fine] + skip[fine]
__global__ void k_up_add(const uint16_t* __restrict__ coarse, const uint16_t* __restrict__ skip,
                         uint16_t* __restrict__ out, int C, int nx, int ny, int nz, long long BVf) {
  const long long Vf = (long long)nx * ny * nz;
  const int cx = nx / 2, cy = ny / 2, cz = nz / 2;
  const long long Vc = (long long)cx * cy * cz;
  const int C4 = C / 4;  // four channels (one 8-byte word) per thread, C % 4 == 0
  const long long n = BVf * C4;
  const s4* c4p = reinterpret_cast<const s4*>(coarse);
  const s4* s4p = reinterpret_cast<const s4*>(skip);
  s4* o4p = reinterpret_cast<s4*>(out);
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
    const int c = (int)(i % C4);
    const long long vv = i / C4;
    long long b;
    int x, y, z;
    vox_xyz(vv, Vf, nx, ny, &b, &x, &y, &z);
    const long long p = b * Vc + (x / 2) + (long long)cx * ((y / 2) + (long long)cy * (z / 2));
    (void)cz;
    const s4 cv = c4p[p * C4 + c], sv = s4p[i];
    s4 o;
#pragma unroll
    for (int k = 0; k < 4; k++) o[k] = (short)f2bf(bf2f((uint16_t)cv[k]) + bf2f((uint16_t)sv[k]));
    o4p[i] = o;
  }
}

// Backward of up+add for the coarse branch: gc[parent] = sum of the 8 children
// of gfine, masked by ReLU of the coarse activation (act > 0).
__global__ void k_up_bwd(const uint16_t* __restrict__ gf, const uint16_t* __restrict__ act_c,
                         uint16_t* __restrict__ gc, int C, int nx, int ny, int nz, long long Bc) {
  const int cx = nx / 2, cy = ny / 2, cz = nz / 2;
  const long long Vc = (long long)cx * cy * cz, Vf = (long long)nx * ny * nz;
  const long long n = Bc * Vc * C;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
    const int c = (int)(i % C);
    const long long vv = i / C;
    long long b;
    int x, y, z;
    vox_xyz(vv, Vc, cx, cy, &b, &x, &y, &z);
    float s = 0.f;
    for (int a = 0; a < 8; a++) {
      const long long f = b * Vf + (2 * x + (a & 1)) + (long long)nx * ((2 * y + ((a >> 1) & 1)) +
                                                                       (long long)ny * (2 * z + ((a >> 2) & 1)));
      s += bf2f(gf[f * C + c]);
    }
    gc[i] = bf2f(act_c[i]) > 0.f ? f2bf(s) : (uint16_t)0;
  }
}

// Gradient of an encoder activation that feeds both the pool and a skip:
// gfine = (gpool[parent] / 8 + gskip[fine]) masked by ReLU of act.
__global__ void k_pool_bwd(const uint16_t* __restrict__ gpool, const uint16_t* __restrict__ gskip,
                           const uint16_t* __restrict__ act, uint16_t* __restrict__ gf, int C, int nx, int ny, int nz,
                           long long BVf) {
  const long long Vf = (long long)nx * ny * nz;
  const int cx = nx / 2, cy = ny / 2;
  const long long Vc = (long long)cx * cy * (nz / 2);
  const long long n = BVf * C;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
    const int c = (int)(i % C);
    const long long vv = i / C;
    long long b;
    int x, y, z;
    vox_xyz(vv, Vf, nx, ny, &b, &x, &y, &z);
    const long long p = b * Vc + (x / 2) + (long long)cx * ((y / 2) + (long long)cy * (z / 2));
    const float s = bf2f(gpool[p * C + c]) * 0.125f + bf2f(gskip[i]);
    gf[i] = bf2f(act[i]) > 0.f ? f2bf(s) : (uint16_t)0;
  }
}

__global__ void k_relu_mask(uint16_t* __restrict__ g, const uint16_t* __restrict__ act, long long n) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    if (!(bf2f(act[i]) > 0.f)) g[i] = 0;
}

// ---------------------------------------------------------------------------
// loss
// ---------------------------------------------------------------------------
// per-sample partial sums of d = c - a (grid (nblk, B))
__global__ void k_seg_sum(const float* __restrict__ c, const float* __restrict__ a, long long V, int nblk,
                          double* __restrict__ partial) {
  __shared__ double sh[kBlock / 64];
  const int b = blockIdx.y;
  double s = 0.0;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < V; i += (long long)nblk * blockDim.x)
    s += (double)c[b * V + i] - (double)a[b * V + i];
  s = wave_sum(s);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int w = 0; w < (int)(blockDim.x >> 6); w++) t += sh[w];
    partial[b * nblk + blockIdx.x] = t;
  }
}
// gout = (2 w_b / B) (d - mean_b);  partial of sum (d - mean)^2
__global__ void k_loss_grad(const float* __restrict__ c, const float* __restrict__ a, const float* __restrict__ w,
                            const int* __restrict__ proj, const double* __restrict__ sums, long long V, int B,
                            int nblk, float* __restrict__ gout, double* __restrict__ partial) {
  __shared__ double sh[kBlock / 64];
  const int b = blockIdx.y;
  double tot = 0.0;
  for (int k = 0; k < nblk; k++) tot += sums[b * nblk + k];
  const double mean = proj[b] ? tot / (double)V : 0.0;
  const double scale = 2.0 * (double)w[b] / (double)B;
  double s = 0.0;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < V; i += (long long)nblk * blockDim.x) {
    const double d = (double)c[b * V + i] - (double)a[b * V + i] - mean;
    gout[b * V + i] = (float)(scale * d);
    s += d * d;
  }
  s = wave_sum(s);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int q = 0; q < (int)(blockDim.x >> 6); q++) t += sh[q];
    partial[b * nblk + blockIdx.x] = t;
  }
}

// ---------------------------------------------------------------------------
// optimiser
// ---------------------------------------------------------------------------
__global__ void k_sumsq_partial(const float* __restrict__ g, long long n, double* __restrict__ partial) {
  __shared__ double sh[kBlock / 64];
  double s = 0.0;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    s += (double)g[i] * (double)g[i];
  s = wave_sum(s);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int q = 0; q < (int)(blockDim.x >> 6); q++) t += sh[q];
    partial[blockIdx.x] = t;
  }
}
// clip factor from the per-block sums of squares: out[0] = min(1, clip / |g|), out[1] = |g|
__global__ void k_clip_factor(const double* __restrict__ partial, int nblk, float clip, double* __restrict__ out) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  double ss = 0.0;
  for (int k = 0; k < nblk; k++) ss += partial[k];
  const double gn = sqrt(ss);
  out[0] = (clip > 0.f && gn > clip) ? clip / gn : 1.0;
  out[1] = gn;
}
__global__ void k_adam(float* __restrict__ w, const float* __restrict__ g, float* __restrict__ m,
                       float* __restrict__ v, long long n, const double* __restrict__ clipf, float lr, float b1,
                       float b2, float eps, float bc1, float bc2) {
  const float sc = (float)clipf[0];
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
    const float gi = g[i] * sc;
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    w[i] -= lr * (mi / bc1) / (sqrtf(vi / bc2) + eps);
  }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
static inline unsigned gridn(long long n) {
  long long b = (n + kBlock - 1) / kBlock;
  if (b > 65535) b = 65535;
  if (b < 1) b = 1;
  return (unsigned)b;
}

static uint64_t splitmix(uint64_t* s) {
  uint64_t z = (*s += 0x9E3779B97F4A7C15ULL);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
  return z ^ (z >> 31);
}
static double unif(uint64_t* s) { return ((splitmix(s) >> 11) + 0.5) * (1.0 / 9007199254740992.0); }

int create(Net* n, uint64_t seed, hipStream_t st) {
  n->st = st;
  const long long np = num_params();
  NCK(hipMalloc(&n->w, sizeof(float) * np));
  NCK(hipMalloc(&n->g, sizeof(float) * np));
  NCK(hipMalloc(&n->m, sizeof(float) * np));
  NCK(hipMalloc(&n->v, sizeof(float) * np));
  NCK(hipMemset(n->g, 0, sizeof(float) * np));
  NCK(hipMemset(n->m, 0, sizeof(float) * np));
  NCK(hipMemset(n->v, 0, sizeof(float) * np));
  // He-normal initialisation (fan-in 27 * real input channels), zero biases;
  // the output layer starts small so that the untrained network is close to
  // the plain diagonal preconditioner.
  std::vector<float> h(np, 0.f);
  uint64_t s = seed * 0x2545F4914F6CDD1DULL + 1;
  for (int l = 0; l < kLayers; l++) {
    const LayerSpec& L = kSpec[l];
    double sd = std::sqrt(2.0 / (27.0 * L.cin_real));
    if (l == kLayers - 1) sd *= 0.01;
    const long long o = weight_offset(l);
    for (int kk = 0; kk < 27 * L.cin; kk++) {
      const int ci = kk % L.cin;
      for (int co = 0; co < L.cout; co++) {
        const double u1 = unif(&s), u2 = unif(&s);
        const double gsn = std::sqrt(-2.0 * std::log(u1)) * std::cos(6.283185307179586 * u2);
        h[o + (long long)kk * L.cout + co] = ci < L.cin_real ? (float)(sd * gsn) : 0.f;
      }
    }
  }
  NCK(hipMemcpy(n->w, h.data(), sizeof(float) * np, hipMemcpyHostToDevice));
  for (int l = 0; l < kLayers; l++) {
    const LayerSpec& L = kSpec[l];
    NCK(hipMalloc(&n->wp[l], sizeof(s4) * 64LL * kchunks(L.cin) * ntiles(L.cout)));
    // forward passes of layers with cin a multiple of 8 run on the 32-wide
    // step unless GALE_LPC_K32=0 (see the note at k_pack32)
    const char* k32 = std::getenv("GALE_LPC_K32");
    if (L.cin % 8 == 0 && !(k32 && k32[0] == '0'))
      NCK(hipMalloc(&n->wp32[l], sizeof(s8) * 64LL * kchunks32(L.cin) * ntiles(L.cout)));
    const int cin_t = L.cout < 4 ? 4 : L.cout;  // transposed GEMM input channels (gradient tensor)
    NCK(hipMalloc(&n->wt[l], sizeof(s4) * 64LL * kchunks(cin_t) * ntiles(L.cin)));
  }
  pack(n);
  NCK(hipStreamSynchronize(st));
  return GS_OK;
}

void pack(Net* n) {
  for (int l = 0; l < kLayers; l++) {
    const LayerSpec& L = kSpec[l];
    const float* W = n->w + weight_offset(l);
    const int kc = kchunks(L.cin), nt = ntiles(L.cout);
    hipLaunchKernelGGL(k_pack, dim3(gridn(64LL * kc * nt)), dim3(kBlock), 0, n->st, W, L.cin, L.cout, 0, L.cin, nt,
                       kc, (s4*)n->wp[l]);
    if (n->wp32[l])
      hipLaunchKernelGGL(k_pack32, dim3(gridn(64LL * kchunks32(L.cin) * nt)), dim3(kBlock), 0, n->st, W, L.cin,
                         L.cout, nt, kchunks32(L.cin), (s8*)n->wp32[l]);
    const int cin_t = L.cout < 4 ? 4 : L.cout;
    const int kct = kchunks(cin_t), ntt = ntiles(L.cin);
    hipLaunchKernelGGL(k_pack, dim3(gridn(64LL * kct * ntt)), dim3(kBlock), 0, n->st, W, L.cin, L.cout, 1, cin_t,
                       ntt, kct, (s4*)n->wt[l]);
  }
  n->packed = true;
}

static void free_work(Work& w) {
  auto f = [](void* p) {
    if (p) (void)hipFree(p);
  };
  f(w.x4);
  for (int l = 0; l < kLayers; l++) f(w.act[l]);
  for (int l = 0; l < kLevels; l++) {
    f(w.pool[l]);
    f(w.upadd[l]);
    f(w.gskip[l]);
  }
  f(w.out32);
  f(w.g4);
  f(w.ga);
  f(w.gb);
  f(w.gc);
  f(w.partial);
  f(w.bpart);
  f(w.xt);
  f(w.gt);
  f(w.dpartial);
  w = Work{};
}

void destroy(Net* n) {
  free_work(n->work);
  auto f = [](void* p) {
    if (p) (void)hipFree(p);
  };
  f(n->w);
  f(n->g);
  f(n->m);
  f(n->v);
  for (int l = 0; l < kLayers; l++) {
    f(n->wp[l]);
    f(n->wp32[l]);
    f(n->wt[l]);
  }
  *n = Net{};
}

// Weight-gradient layout of a layer: flat length of its padded grid (one row
// per channel), reach of a tap's shift, groups of voxels and K values a wave.
struct WgradPlan {
  long long stride, kper;
  int w, pl, ngroup, nblk;
};
static WgradPlan wgrad_plan(const Shape& sh, int l) {
  const LayerSpec& L = kSpec[l];
  const int nx = sh.nx >> L.level, ny = sh.ny >> L.level, nz = sh.nz >> L.level;
  WgradPlan p;
  p.w = nx + 2;
  p.pl = (nx + 2) * (ny + 2);
  p.stride = ((long long)sh.batch * p.pl * (nz + 2) + 31) / 32 * 32;
  const int mt = (L.cin + 15) / 16;
  // about a thousand blocks, but at least four K steps a wave and at most 64
  // partial sums to add
  long long g = 1024 / (9 * mt);
  if (g > 64) g = 64;
  if (g > p.stride / 512) g = p.stride / 512;
  if (g < 1) g = 1;
  p.kper = ((p.stride + 4 * g - 1) / (4 * g) + 31) / 32 * 32;
  p.ngroup = (int)((p.stride + 4 * p.kper - 1) / (4 * p.kper));
  p.nblk = (int)((p.stride + kPadVox - 1) / kPadVox);
  return p;
}
static inline int wgrad_margin(const WgradPlan& p) { return p.pl + p.w + 2 + 32; }

static int alloc_work(Net* n, const Shape& sh) {
  if (sh.nx % kGridMultiple || sh.ny % kGridMultiple || sh.nz % kGridMultiple || sh.nx < kGridMultiple ||
      sh.ny < kGridMultiple || sh.nz < kGridMultiple || sh.batch < 1)
    return GS_E_INVALID;
  free_work(n->work);
  Work& w = n->work;
  w.sh = sh;
  for (int l = 0; l < kLevels; l++)
    w.BV[l] = (long long)sh.batch * (sh.nx >> l) * (sh.ny >> l) * (sh.nz >> l);
  auto al = [](uint16_t** p, long long cnt) { return hipMalloc(p, sizeof(uint16_t) * (cnt > 0 ? cnt : 1)); };
  NCK(al(&w.x4, w.BV[0] * 4));
  long long gmax = w.BV[0] * 4;
  for (int l = 0; l < kLayers; l++) {
    const long long cnt = w.BV[kSpec[l].level] * kSpec[l].cout;
    if (l < kLayers - 1) NCK(al(&w.act[l], cnt));
    gmax = cnt > gmax ? cnt : gmax;
    const long long cin_cnt = w.BV[kSpec[l].level] * kSpec[l].cin;
    gmax = cin_cnt > gmax ? cin_cnt : gmax;
  }
  for (int l = 1; l < kLevels; l++) NCK(al(&w.pool[l], w.BV[l] * kChan[l - 1]));
  for (int l = 0; l < kLevels - 1; l++) {
    NCK(al(&w.upadd[l], w.BV[l] * kChan[l]));
    NCK(al(&w.gskip[l], w.BV[l] * kChan[l]));
  }
  NCK(hipMalloc(&w.out32, sizeof(float) * w.BV[0]));
  NCK(al(&w.g4, w.BV[0] * 4));
  NCK(al(&w.ga, gmax));
  NCK(al(&w.gb, gmax));
  NCK(al(&w.gc, gmax));
  long long pc = 0, xc = 0, gc = 0, bc = 0;
  w.tmargin = 0;
  for (int l = 0; l < kLayers; l++) {
    const LayerSpec& L = kSpec[l];
    const WgradPlan p = wgrad_plan(sh, l);
    const long long m = (wgrad_margin(p) + 31) / 32 * 32;
    w.tmargin = m > w.tmargin ? m : w.tmargin;
    pc = std::max(pc, (long long)p.ngroup * 27 * L.cin * L.cout);
    xc = std::max(xc, (L.cin + 15) / 16 * 16 * p.stride);
    gc = std::max(gc, (long long)ntiles(L.cout) * 16 * p.stride);
    bc = std::max(bc, (long long)p.nblk * L.cout);
  }
  // rows start tmargin entries in: the first row's shifted loads run below it
  // and the last row's beyond it, both over zeros
  NCK(al(&w.xt, xc + 2 * w.tmargin));
  NCK(al(&w.gt, gc + 2 * w.tmargin));
  NCK(hipMemset(w.xt, 0, sizeof(uint16_t) * (xc + 2 * w.tmargin)));
  NCK(hipMemset(w.gt, 0, sizeof(uint16_t) * (gc + 2 * w.tmargin)));
  NCK(hipMalloc(&w.partial, sizeof(float) * pc));
  NCK(hipMalloc(&w.bpart, sizeof(float) * bc));
  NCK(hipMalloc(&w.dpartial, sizeof(double) * 65536));
  return GS_OK;
}

// A shape that does not fit leaves nothing: with some of its buffers the next
// call of that shape would take it for allocated.
int ensure_work(Net* n, const Shape& sh) {
  if (n->work.sh == sh && n->work.x4) return GS_OK;
  const int e = alloc_work(n, sh);
  if (e == GS_E_HIP) {
    (void)hipGetLastError();
    free_work(n->work);
  }
  return e;
}

// dispatch of the templated convolution kernels
#define CONV_CASES(X) \
  X(4, 1) X(16, 1) X(16, 2) X(32, 1) X(32, 2) X(32, 3) X(48, 2) X(48, 3) X(48, 4) X(64, 3) X(64, 4) X(64, 6) X(96, 4)

#define CONV_TILED_CASES(X) X(4, 1) X(16, 1) X(16, 2) X(32, 1) X(32, 2) X(32, 3)

// KW: 16 or 32 K values per matrix-core step (32 needs cin a multiple of 8
// and weights packed for it).
template <int KW>
static int launch_conv_kw(int cin, int nt, bool f32, const uint16_t* in, const void* Wp, const float* bias,
                          void* out, int cout_store, int nx, int ny, int nz, long long BV, int relu, hipStream_t st) {
  typedef typename KOp<KW>::type AT;
  const AT* W = static_cast<const AT*>(Wp);
  if (nx % 16 == 0 && ny % 4 == 0 && nz % 4 == 0) {
    const long long V = (long long)nx * ny * nz;
    const dim3 tgrid((unsigned)(BV / V * (V / 256))), tblock(256);
#define X(C, N)                                                                                                  \
  if constexpr (KW == 16 || (C) % 8 == 0) {                                                                      \
    if (cin == C && nt == N) {                                                                                   \
      if (f32)                                                                                                   \
        hipLaunchKernelGGL((k_conv_tiled<C, N, true, KW>), tgrid, tblock, 0, st, in, W, bias, out, cout_store,   \
                           nx, ny, nz, relu);                                                                    \
      else                                                                                                       \
        hipLaunchKernelGGL((k_conv_tiled<C, N, false, KW>), tgrid, tblock, 0, st, in, W, bias, out, cout_store,  \
                           nx, ny, nz, relu);                                                                    \
      return GS_OK;                                                                                              \
    }                                                                                                            \
  }
    CONV_TILED_CASES(X)
#undef X
  }
  const long long tiles16 = (BV + 15) / 16;
  if (tiles16 < 4096) {  // small level: split K over 4 (or 8) waves per 16-voxel tile
    const dim3 sgrid((unsigned)tiles16);
#define X(C, N)                                                                                                  \
  if constexpr (KW == 16 || (C) % 8 == 0) {                                                                      \
    if (cin == C && nt == N) {                                                                                   \
      if (tiles16 < 512) {                                                                                       \
        if (f32)                                                                                                 \
          hipLaunchKernelGGL((k_conv_splitk<C, N, true, 8, KW>), sgrid, dim3(512), 0, st, in, W, bias, out,      \
                             cout_store, nx, ny, nz, BV, relu);                                                  \
        else                                                                                                     \
          hipLaunchKernelGGL((k_conv_splitk<C, N, false, 8, KW>), sgrid, dim3(512), 0, st, in, W, bias, out,     \
                             cout_store, nx, ny, nz, BV, relu);                                                  \
      } else {                                                                                                   \
        if (f32)                                                                                                 \
          hipLaunchKernelGGL((k_conv_splitk<C, N, true, 4, KW>), sgrid, dim3(256), 0, st, in, W, bias, out,      \
                             cout_store, nx, ny, nz, BV, relu);                                                  \
        else                                                                                                     \
          hipLaunchKernelGGL((k_conv_splitk<C, N, false, 4, KW>), sgrid, dim3(256), 0, st, in, W, bias, out,     \
                             cout_store, nx, ny, nz, BV, relu);                                                  \
      }                                                                                                          \
      return GS_OK;                                                                                              \
    }                                                                                                            \
  }
    CONV_CASES(X)
#undef X
  }
  const dim3 grid((unsigned)((BV + 63) / 64)), block(256);
#define X(C, N)                                                                                                  \
  if constexpr (KW == 16 || (C) % 8 == 0) {                                                                      \
    if (cin == C && nt == N) {                                                                                   \
      if (f32)                                                                                                   \
        hipLaunchKernelGGL((k_conv<C, N, true, KW>), grid, block, 0, st, in, W, bias, out, cout_store, nx, ny,   \
                           nz, BV, relu);                                                                        \
      else                                                                                                       \
        hipLaunchKernelGGL((k_conv<C, N, false, KW>), grid, block, 0, st, in, W, bias, out, cout_store, nx, ny,  \
                           nz, BV, relu);                                                                        \
      return GS_OK;                                                                                              \
    }                                                                                                            \
  }
  CONV_CASES(X)
#undef X
  std::fprintf(stderr, "gale_stokes(net): no convolution kernel for cin %d, %d tiles, K step %d\n", cin, nt, KW);
  return GS_E_INVALID;
}

static int launch_conv(int cin, int nt, bool f32, const uint16_t* in, const void* Wp, const float* bias, void* out,
                       int cout_store, int nx, int ny, int nz, long long BV, int relu, hipStream_t st, int kw = 16) {
  if (kw == 32)
    return launch_conv_kw<32>(cin, nt, f32, in, Wp, bias, out, cout_store, nx, ny, nz, BV, relu, st);
  return launch_conv_kw<16>(cin, nt, f32, in, Wp, bias, out, cout_store, nx, ny, nz, BV, relu, st);
}

// dW and db of layer l from its input x and the gradient g of its output
// (cg stored channels).
static int launch_wgrad(Net* n, int l, const uint16_t* x, const uint16_t* g, int cg, int nx, int ny, int nz) {
  Work& w = n->work;
  const LayerSpec& L = kSpec[l];
  hipStream_t st = n->st;
  const WgradPlan p = wgrad_plan(w.sh, l);
  const int margin = wgrad_margin(p), B = w.sh.batch;
  uint16_t *xt = w.xt + w.tmargin, *gt = w.gt + w.tmargin;
  hipLaunchKernelGGL(k_pad_t, dim3(p.nblk + 1), dim3(256), pad_lds(L.cin), st, x, L.cin, L.cin, xt, p.stride, margin, nx, ny, nz,
                     B, (float*)nullptr);
  hipLaunchKernelGGL(k_pad_t, dim3(p.nblk + 1), dim3(256), pad_lds(cg), st, g, cg, L.cout, gt, p.stride, margin, nx, ny, nz, B,
                     w.bpart);
  const dim3 grid((unsigned)((L.cin + 15) / 16 * 9), (unsigned)p.ngroup), block(256);
  switch (ntiles(L.cout)) {
#define X(N)                                                                                                      \
  case N:                                                                                                         \
    hipLaunchKernelGGL(k_wgrad<N>, grid, block, 0, st, xt, gt, p.stride, L.cin, L.cout, p.w, p.pl, p.kper,        \
                       w.partial);                                                                                \
    break;
    X(1) X(2) X(3) X(4) X(6)
#undef X
    default:
      std::fprintf(stderr, "gale_stokes(net): no weight-gradient kernel for %d outputs\n", L.cout);
      return GS_E_INVALID;
  }
  const long long nw = 27LL * L.cin * L.cout;
  hipLaunchKernelGGL(k_wgrad_reduce, dim3(gridn(nw)), dim3(kBlock), 0, st, w.partial, p.ngroup, nw,
                     n->g + weight_offset(l));
  hipLaunchKernelGGL(k_bgrad_reduce, dim3(L.cout), dim3(kBlock), 0, st, w.bpart, p.nblk, L.cout,
                     n->g + bias_offset(l));
  return GS_OK;
}

static int lvl_dims(const Shape& sh, int l, int* nx, int* ny, int* nz) {
  *nx = sh.nx >> l;
  *ny = sh.ny >> l;
  *nz = sh.nz >> l;
  return 0;
}

// forward of layer l from tensor `in` into act[l] (or out32 for the last)
static int fwd_layer(Net* n, int l, const uint16_t* in, void* out) {
  Work& w = n->work;
  const LayerSpec& L = kSpec[l];
  int nx, ny, nz;
  lvl_dims(w.sh, L.level, &nx, &ny, &nz);
  const bool last = (l == kLayers - 1);
  if (n->wp32[l])  // gfx950's 16x16x32 matrix-core step
    return launch_conv(L.cin, ntiles(L.cout), last, in, n->wp32[l], n->w + bias_offset(l), out, L.cout, nx, ny,
                       nz, w.BV[L.level], L.relu, n->st, 32);
  return launch_conv(L.cin, ntiles(L.cout), last, in, n->wp[l], n->w + bias_offset(l), out, L.cout, nx, ny, nz,
                     w.BV[L.level], L.relu, n->st);
}

int forward(Net* n, const Shape& sh, const float* in2, float* out) {
  int e = ensure_work(n, sh);
  if (e) return e;
  Work& w = n->work;
  hipStream_t st = n->st;
  hipLaunchKernelGGL(k_pack_input, dim3(gridn(w.BV[0])), dim3(kBlock), 0, st, in2, w.x4, w.BV[0]);
  int nx, ny, nz;
  // encoder and bottom level
  for (int l = 0; l < kLevels; l++) {
    const uint16_t* in = w.x4;
    if (l > 0) {
      lvl_dims(sh, l - 1, &nx, &ny, &nz);
      const int C = kChan[l - 1];
      hipLaunchKernelGGL(k_pool, dim3(gridn(w.BV[l] * C / 4)), dim3(kBlock), 0, st, w.act[enc_b(l - 1)], w.pool[l], C,
                         nx, ny, nz, (long long)sh.batch);
      in = w.pool[l];
    }
    if ((e = fwd_layer(n, enc_a(l), in, w.act[enc_a(l)]))) return e;
    if ((e = fwd_layer(n, enc_b(l), w.act[enc_a(l)], w.act[enc_b(l)]))) return e;
  }
  // decoder
  int cur = enc_b(kLevels - 1);
  for (int l = kLevels - 2; l >= 0; l--) {
    lvl_dims(sh, l, &nx, &ny, &nz);
    const int C = kChan[l];
    hipLaunchKernelGGL(k_up_add, dim3(gridn(w.BV[l] * C / 4)), dim3(kBlock), 0, st, w.act[cur], w.act[enc_b(l)],
                       w.upadd[l], C, nx, ny, nz, w.BV[l]);
    if ((e = fwd_layer(n, dec_a(l), w.upadd[l], w.act[dec_a(l)]))) return e;
    void* o = l > 0 ? (void*)w.act[dec_b(l)] : (void*)(out ? out : w.out32);
    if ((e = fwd_layer(n, dec_b(l), w.act[dec_a(l)], o))) return e;
    cur = dec_b(l);
  }
  return GS_OK;
}

// Gradients of layer l given g_pre (ReLU-masked gradient of its output,
// channels cg) and its input tensor x; writes dW, db, and (if gin) the
// gradient of its input (unmasked).
static int bwd_layer(Net* n, int l, const uint16_t* x, const uint16_t* gpre, int cg, uint16_t* gin) {
  Work& w = n->work;
  const LayerSpec& L = kSpec[l];
  int nx, ny, nz;
  lvl_dims(w.sh, L.level, &nx, &ny, &nz);
  const long long BV = w.BV[L.level];
  hipStream_t st = n->st;
  int e = launch_wgrad(n, l, x, gpre, cg, nx, ny, nz);
  if (e) return e;
  if (gin) {
    const int cin_t = L.cout < 4 ? 4 : L.cout;
    e = launch_conv(cin_t, ntiles(L.cin), false, gpre, n->wt[l], nullptr, gin, L.cin, nx, ny, nz, BV, 0, st);
    if (e) return e;
  }
  return GS_OK;
}

int backward(Net* n, const Shape& sh, const float* gout) {
  Work& w = n->work;
  if (!(w.sh == sh) || !w.x4) return GS_E_INVALID;
  hipStream_t st = n->st;
  int e, nx, ny, nz;
  uint16_t *A = w.ga, *B = w.gb, *C = w.gc;
  hipLaunchKernelGGL(k_pack_gout, dim3(gridn(w.BV[0])), dim3(kBlock), 0, st, gout, w.g4, w.BV[0]);
  // decoder, finest level first; B holds the ReLU-masked gradient of the
  // level's output (level 0: the packed dL/dc)
  for (int l = 0; l <= kLevels - 2; l++) {
    const int a = dec_a(l), b = dec_b(l);
    const int Cl = kChan[l];
    if ((e = bwd_layer(n, b, w.act[a], l == 0 ? w.g4 : B, l == 0 ? 4 : kSpec[b].cout, A))) return e;
    hipLaunchKernelGGL(k_relu_mask, dim3(gridn(w.BV[l] * Cl)), dim3(kBlock), 0, st, A, w.act[a], w.BV[l] * Cl);
    if ((e = bwd_layer(n, a, w.upadd[l], A, Cl, w.gskip[l]))) return e;
    // upadd[l] = up(src) + skip l
    const int src = l == kLevels - 2 ? enc_b(kLevels - 1) : dec_b(l + 1);
    lvl_dims(sh, l, &nx, &ny, &nz);
    hipLaunchKernelGGL(k_up_bwd, dim3(gridn(w.BV[l + 1] * Cl)), dim3(kBlock), 0, st, w.gskip[l], w.act[src], B, Cl,
                       nx, ny, nz, (long long)sh.batch);
  }
  // bottom level
  {
    const int L = kLevels - 1;
    if ((e = bwd_layer(n, enc_b(L), w.act[enc_a(L)], B, kChan[L - 1], A))) return e;
    hipLaunchKernelGGL(k_relu_mask, dim3(gridn(w.BV[L] * kChan[L])), dim3(kBlock), 0, st, A, w.act[enc_a(L)],
                       w.BV[L] * kChan[L]);
    if ((e = bwd_layer(n, enc_a(L), w.pool[L], A, kChan[L], C))) return e;  // C: gradient of pool[L]
  }
  // encoder, coarse to fine: act[enc_b(l)] feeds pool[l+1] and skip l
  for (int l = kLevels - 2; l >= 0; l--) {
    const int Cl = kChan[l];
    lvl_dims(sh, l, &nx, &ny, &nz);
    hipLaunchKernelGGL(k_pool_bwd, dim3(gridn(w.BV[l] * Cl)), dim3(kBlock), 0, st, C, w.gskip[l], w.act[enc_b(l)], B,
                       Cl, nx, ny, nz, w.BV[l]);
    if ((e = bwd_layer(n, enc_b(l), w.act[enc_a(l)], B, Cl, A))) return e;
    hipLaunchKernelGGL(k_relu_mask, dim3(gridn(w.BV[l] * Cl)), dim3(kBlock), 0, st, A, w.act[enc_a(l)], w.BV[l] * Cl);
    if ((e = bwd_layer(n, enc_a(l), l > 0 ? w.pool[l] : w.x4, A, Cl, l > 0 ? C : nullptr))) return e;
  }
  return GS_OK;
}

int adam_step(Net* n, float lr, float beta1, float beta2, float eps, float clip, double* gnorm_out) {
  const long long np = num_params();
  Work& w = n->work;
  if (!w.dpartial) return GS_E_INVALID;
  const int nb = 512;
  double* clipf = w.dpartial + nb;
  hipLaunchKernelGGL(k_sumsq_partial, dim3(nb), dim3(kBlock), 0, n->st, n->g, np, w.dpartial);
  hipLaunchKernelGGL(k_clip_factor, dim3(1), dim3(64), 0, n->st, w.dpartial, nb, clip, clipf);
  n->adam_t++;
  const float bc1 = 1.f - std::pow(beta1, (float)n->adam_t), bc2 = 1.f - std::pow(beta2, (float)n->adam_t);
  hipLaunchKernelGGL(k_adam, dim3(gridn(np)), dim3(kBlock), 0, n->st, n->w, n->g, n->m, n->v, np, clipf, lr, beta1,
                     beta2, eps, bc1, bc2);
  if (gnorm_out) {
    double h[2];
    NCK(hipMemcpyAsync(h, clipf, sizeof(h), hipMemcpyDeviceToHost, n->st));
    NCK(hipStreamSynchronize(n->st));
    *gnorm_out = h[1];
  }
  pack(n);
  return GS_OK;
}

int loss_grad(Net* n, const Shape& sh, const float* c, const float* a, const float* w, const int* proj, float* gout,
              double* loss) {
  Work& wk = n->work;
  if (!wk.dpartial) return GS_E_INVALID;
  const long long V = (long long)sh.nx * sh.ny * sh.nz;
  const int B = sh.batch;
  int nblk = (int)((V + kBlock - 1) / kBlock);
  if (nblk > 64) nblk = 64;
  if ((long long)B * nblk * 2 > 65536) return GS_E_INVALID;
  double* sums = wk.dpartial;
  double* sq = wk.dpartial + (long long)B * nblk;
  hipLaunchKernelGGL(k_seg_sum, dim3(nblk, B), dim3(kBlock), 0, n->st, c, a, V, nblk, sums);
  hipLaunchKernelGGL(k_loss_grad, dim3(nblk, B), dim3(kBlock), 0, n->st, c, a, w, proj, sums, V, B, nblk, gout, sq);
  if (loss) {
    std::vector<double> h((size_t)B * nblk);
    std::vector<float> hw(B);
    NCK(hipMemcpyAsync(h.data(), sq, sizeof(double) * B * nblk, hipMemcpyDeviceToHost, n->st));
    NCK(hipMemcpyAsync(hw.data(), w, sizeof(float) * B, hipMemcpyDeviceToHost, n->st));
    NCK(hipStreamSynchronize(n->st));
    double L = 0.0;
    for (int b = 0; b < B; b++) {
      double s = 0.0;
      for (int k = 0; k < nblk; k++) s += h[(size_t)b * nblk + k];
      L += hw[b] * s;
    }
    *loss = L / B;
  }
  return GS_OK;
}

// ---------------------------------------------------------------------------
// self test of the operand layout: D = A B for A[i][k] = (i + 2k) / 32,
// B[k][j] = (3k - j) / 32 (exact in BF16), one wavefront.
// ---------------------------------------------------------------------------
__global__ void k_mfma_selftest(float* __restrict__ out) {
  const int lane = threadIdx.x;
  if (lane >= 64) return;
  s4 a, b;
  for (int j = 0; j < 4; j++) {
    const int k = 4 * (lane >> 4) + j;
    a[j] = (short)f2bf((float)((lane & 15) + 2 * k) / 32.f);
    b[j] = (short)f2bf((float)(3 * k - (lane & 15)) / 32.f);
  }
  f4 acc = f4{0.f, 0.f, 0.f, 0.f};
  acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc, 0, 0, 0);
  for (int i = 0; i < 4; i++) out[(4 * (lane >> 4) + i) * 16 + (lane & 15)] = acc[i];
}

// The same for the 32-wide step (v_mfma_f32_16x16x32_bf16): lane l holds
// K = 8 (l / 16) + j, j = 0..7, of A's row l % 16 and B's column l % 16.
__global__ void k_mfma_selftest32(float* __restrict__ out) {
  const int lane = threadIdx.x;
  if (lane >= 64) return;
  s8 a, b;
  for (int j = 0; j < 8; j++) {
    const int k = 8 * (lane >> 4) + j;
    a[j] = (short)f2bf((float)((lane & 15) + 2 * k) / 32.f);
    b[j] = (short)f2bf((float)(3 * k - (lane & 15)) / 32.f);
  }
  f4 acc = f4{0.f, 0.f, 0.f, 0.f};
  acc = mfma_bf16(a, b, acc);
  for (int i = 0; i < 4; i++) out[(4 * (lane >> 4) + i) * 16 + (lane & 15)] = acc[i];
}

// Both step widths against the exact product (every value is exact in BF16
// and every partial sum in FP32); returns the larger error.
int selftest_mfma(float* max_err) {
  float* d = nullptr;
  NCK(hipMalloc(&d, sizeof(float) * 512));
  hipLaunchKernelGGL(k_mfma_selftest, dim3(1), dim3(64), 0, 0, d);
  hipLaunchKernelGGL(k_mfma_selftest32, dim3(1), dim3(64), 0, 0, d + 256);
  float h[512];
  NCK(hipMemcpy(h, d, sizeof(h), hipMemcpyDeviceToHost));
  NCK(hipFree(d));
  float e = 0.f;
  for (int kw = 16; kw <= 32; kw += 16)
    for (int i = 0; i < 16; i++)
      for (int j = 0; j < 16; j++) {
        double s = 0.0;
        for (int k = 0; k < kw; k++) s += ((i + 2.0 * k) / 32.0) * ((3.0 * k - j) / 32.0);
        e = std::fmax(e, (float)std::fabs(h[(kw == 32 ? 256 : 0) + i * 16 + j] - s));
      }
  *max_err = e;
  return GS_OK;
}

}  // namespace net
}  // namespace gs
