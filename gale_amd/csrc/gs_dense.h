// gs_dense.h -- assembly and inversion of the dense coarsest operator (gs_dense.hip).
#pragma once

#include "gs_internal.h"

namespace gs {

// Rows and columns of the dense operator are padded with the identity to a
// multiple of this block.
constexpr int kDenseBlock = 64;
inline int dense_ld(int nf) { return (nf + kDenseBlock - 1) / kDenseBlock * kDenseBlock; }

// Scratch of one inversion: two n x 64 panels, one 64 x 64 block.
inline long long dense_work_count(int ld) { return 2LL * ld * kDenseBlock + kDenseBlock * kDenseBlock; }

// A (ld x ld, row-major) = K of the level restricted to its free dofs, from
// the element moments; pos[dof] is the row of a free dof and -1 otherwise.
// Padding rows are the identity.
void launch_dense_assemble(const Geo& g, const double* Mom, const int* pos, int nf, int ld, double* A, hipStream_t st);

// A <- A^-1 (SPD, ld x ld, lower triangle read) with an FP32 copy in Af where
// that is not null.
// *bad is set to 1 when a pivot is not positive and is left alone otherwise.
void launch_spd_inverse(double* A, float* Af, int ld, double* work, int* bad, hipStream_t st);

}  // namespace gs
