// Declarations shared by gemm.hip (dispatch) and gemm_inst_*.hip (kernel instantiations).
#pragma once

#include "common.h"
#include "gemm_core.h"

namespace luxhip {

template <typename T>
struct DenseArgs {
    Operand<T> A, B;
    int M, N, K;
    T* C;
    int64_t ldc;
    const T* bias;   // per m, may be null
    T* pre;          // same layout as C, may be null
    int act;
    int tiles_m, tiles_n;
    int c_vec = 0;   // C and pre allow 8-byte stores at every (m multiple of 4, n): aligned base, ldc a multiple of 4
    int tail = 0;    // this launch finishes the rows or columns of another one (profile name "...+tail")
    int c_f32 = 0;   // batched products of bf16 operands only: C points to fp32 values (same ldc and strides, in elements)
    // batched products only: the softmax rule as the epilogue (attention pullback).  ep_probs != null: with acc = the
    // cotangent of the weights, C = ep_scale * probs .* (acc - ep_d[column]); probs lies as C does (same ldc and
    // strides), ep_d holds one value per column of every product: product b's N values from ep_d + b * N on
    const T* ep_probs = nullptr;
    const float* ep_d = nullptr;
    float ep_scale = 0.0f;
    // batched products: the batch index runs over up to three nested dims (bdim[0] innermost); along
    // dim d the matrices of an operand lie stride[d] elements apart (0: one matrix shared by all)
    int batch = 1;
    int bdim[3] = {1, 1, 1};
    int64_t bsA[3] = {0, 0, 0}, bsB[3] = {0, 0, 0}, bsC[3] = {0, 0, 0};
    // batched products with a triangular operand or result (causal attention), see luxhip_batched_matmul_strided:
    // 0 none; 1 tiles of C with every m > n are left untouched; 2 op(B)[k, n] = 0 for k > n: the
    // contraction stops at the tile's last column; 3 op(B)[k, n] = 0 for k < n: it starts at the tile's first column
    int structure = 0;
};

// The 256 x 256 bf16 kernel (gemm_kk256.h) addresses the 256 rows of a tile, ld elements apart, in 31 bits of bytes
constexpr bool kk256_row_distance_ok(int64_t ld) { return 256 * ld * 2 < (int64_t(1) << 31); }

template <typename T, bool A_KMAJOR, bool B_KMAJOR>
int launch_layout(hipStream_t s, DenseArgs<T>& a);

template <typename T, bool A_KMAJOR, bool B_KMAJOR>
int launch_batched_layout(hipStream_t s, DenseArgs<T>& a);

// gemm_skinny.hip: at most 16 columns, A contiguous along m, B along k; false if the problem is another one
template <typename T>
bool launch_skinny(hipStream_t s, DenseArgs<T>& a, bool a_kmajor, bool b_kmajor, int* rc);
// gemm_split_*.hip: products with few tiles or ragged operands; false if the problem is not theirs
template <typename T>
bool launch_split(hipStream_t s, DenseArgs<T>& a, bool a_kmajor, bool b_kmajor, int* rc);
// two independent products in one launch: a with both operands contiguous along m / n, b with both along k
template <typename T>
bool launch_split_pair(hipStream_t s, DenseArgs<T>& a, DenseArgs<T>& b, int* rc);

// gemm_small.hip: fp32 products that are faster in tiles of 32; false if the problem is another one
bool launch_small(hipStream_t s, DenseArgs<float>& a, bool a_kmajor, bool b_kmajor, int* rc);
// the pullback of a small dense layer in one launch: dz = delta .* act'(y, pre), dW = dz x', dx = W' dz, dbias (may be null) = sum over n of dz;
// delta, y, pre: M x N without gaps.  false if the layer is another one
template <typename T>
bool launch_small_layer_bwd(hipStream_t s, int act, int64_t M, int64_t K, int64_t N, const T* delta, const T* y, const T* pre, const T* W, int64_t ldw,
                            const T* x, int64_t ldx, T* dW, T* dx, T* dbias, int* rc);

// gemm_split_batched_f32.hip: batched fp32 products that are faster there; false if the problem is another one
bool launch_split_batched(hipStream_t s, DenseArgs<float>& a, bool a_kmajor, bool b_kmajor, int* rc);

}  // namespace luxhip
