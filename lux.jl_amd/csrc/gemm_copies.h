// K-major copies of bf16 operands (gemm_copies.hip)
#pragma once

#include <algorithm>

#include "common.h"

namespace luxhip {

// rows of K elements, k contiguous and rows ld apart, -> rows of Kp (a multiple of 64), zeros behind K
int kmajor_rows(hipStream_t s, const bf16_t* in, int64_t ld, int64_t rows, int64_t K, bf16_t* out, int64_t Kp);
// the same from a matrix whose rows are contiguous (k apart by ld)
int kmajor_transposed(hipStream_t s, const bf16_t* in, int64_t ld, int64_t rows, int64_t K, bf16_t* out, int64_t Kp);
// dz (may be null), its transpose dzT (may be null) and, if dbias != null, the bias gradient of a dense pullback; partial: ceil(N / 64) * M
// floats of scratch.  Where M or N is no multiple of 64, ldz and ldt are, and what lies behind the elements is cleared.
int dense_dz_kmajor(hipStream_t s, int act, int64_t M, int64_t N, const bf16_t* delta, const bf16_t* out, const bf16_t* pre, bf16_t* dz, int64_t ldz,
                    bf16_t* dzT, int64_t ldt, float* partial, bf16_t* dbias);
// elementwise.hip: dbias[m] = sum over slices of partial[slice][m]
int plane_finalize_dense_bf16(hipStream_t s, const float* partial, bf16_t* dbias, int64_t M, int64_t slices);

}  // namespace luxhip
