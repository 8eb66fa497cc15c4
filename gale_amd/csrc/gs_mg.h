// gs_mg.h -- launchers of the multigrid kernels (gs_mg.hip).
#pragma once

#include "gs_internal.h"
#include "gs_tile.h"

namespace gs {

void launch_moments_fine(const Geo& g, const double4* pk, const int* off, double* M, hipStream_t st);
void launch_moments_coarsen(const Geo& gc, const Geo& gf, const double* Mf, double* Mc, hipStream_t st);
void launch_d2f(const double* a, float* b, long long n, hipStream_t st);
// FP32 copy of a level's moments, layout-aware (gs_tile.h mom_index).
void launch_mom_d2f(const Geo& g, const double* a, float* b, hipStream_t st);
// Moment-form K apply (tiled, gs_tile.hip); Mom in the layout of gs_tile.h
// (mom_index: tile-major in 3D, SoA in 2D); halo
// needs tile_halo_size(g) values.
template <typename T>
void launch_mom_apply(const Geo& g, const T* x, T* y, const T* Mom, const uint8_t* bcflag, T* halo, hipStream_t st);
void launch_mom_diag(const Geo& g, const double* Mom, double* diag, hipStream_t st);
template <typename T>
void launch_restrict(const Geo& gc, const Geo& gf, const T* rf, T* bc, const uint8_t* bcflag_c, hipStream_t st);
template <typename T>
void launch_prolong_add(const Geo& gc, const Geo& gf, const T* xc, T* xf, const uint8_t* bcflag_f, hipStream_t st);
template <typename T>
void launch_cheb(const T* b, const T* Ax, const T* dinv, T* d, T* x, long long n, T alpha, T beta, int first,
                 hipStream_t st);
// Smoothing step or residual (TileEpi kinds 1 and 2, x null included) on an
// assembled level, one launch.
template <typename T>
void launch_stencil_epi(const Geo& g, const T* A, const T* x, const TileEpi<T>& ep, hipStream_t st);
// Dense coarsest solve x = Kinv b on the free dofs (nf at most
// kDenseWideMax, rows of ld values), zero on the others (pos < 0).  work: the
// inversion's scratch (ld^2 / 64 values at most are used).
constexpr int kDenseWideMax = 8192;
// From this size of the inverse on, half of it is read, in two launches.
// Measured, both launches against the one that reads all of it: n = 5577,
// FP64 (249 MB) 27.3 against 48.0 us, FP32 (124 MB) 18.7 against 23.1 us;
// n = 3267, FP64 (85 MB) 16.6 against 16.6 us; n = 1701, FP64 (23 MB) 10.1
// against 9.0 us, FP32 9.6 against 6.4 us.
constexpr long long kDenseSymBytes = 96LL << 20;
template <typename T>
void launch_dense_solve(const T* Kinv, const int* freeidx, const int* pos, int nf, int ld, double* work, const T* b,
                        T* x, long long n, hipStream_t st);
// Power iteration on D^-1 K (x, Ax, d: n values); st4 in the level's slots.
void launch_pow_init(double* x, const uint8_t* bc, long long n, double* st4, hipStream_t st);
void launch_pow_step(double* x, const double* Ax, const double* dinv, double* d, long long n, double* st4, Reducer rd,
                     hipStream_t st);

// Chebyshev-Jacobi smoothing damps the part [low, high] lambda_max of the
// spectrum of D^-1 K; lambda_max comes from 12 power iterations, which fall
// short of it.  With low = 0.1 the polynomial grows fast above the window, so
// an estimate 10 % short costs more than the wider window gains: inner
// iterations per Uzawa iteration with low 0.1 / 0.15 / 0.2 / 0.25 are 20.6 /
// 8.6 / 6.3 / 6.5 (Rayleigh-Taylor 64^3), 10.2 / - / 7.9 / - (48^3), 4.5 / 4.2
// / 3.8 / 3.9 (random viscosity 96^3), 9.0 / 8.4 / 8.2 / 8.3 (lithosphere
// 256 x 64); learned solves of ten 48^3 and ten 64^3 fields take 11.9 / 10.8 /
// 10.9 s in total.
constexpr double kChebLow = 0.2, kChebHigh = 1.1;

}  // namespace gs
