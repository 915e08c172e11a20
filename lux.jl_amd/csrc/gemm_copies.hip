// Copies of bf16 operands for the 256 x 256 kernel (gemm_kk256.h), which reads both of them along k: rows of whole steps (k padded
// with zeros to a multiple of 64) that start on 16 bytes.
//
// Bound by HBM: a copy reads and writes the operand once.  They pay where the product is large in the other dimension (the rule is
// beside its caller): the products of ragged tensors ran at 500 to 670 TFLOP/s on 128 x 128 tiles that load at any alignment, and run at 900 to
// 1050 on that kernel.  9403 x 10624 (200 MB): 81 us along k, 85 transposed (4.7 to 4.9 TB/s); layernorm, 3072 -> 9403 -> 3072 on 10624 tokens in training
// 5705 -> 3548 us, 1216 -> 3264 on 6845 761 -> 554.
#include "common.h"
#include "act_vec.h"
#include "gemm_copies.h"

namespace luxhip {

// in (rows of K elements, ld apart, at any alignment) -> out (rows of Kp, a multiple of 64, zeros behind K); one 16-byte chunk per
// thread and trip.
__global__ __launch_bounds__(256) void kmajor_rows_kernel(const bf16_t* __restrict__ in, bf16_t* __restrict__ out, int64_t ld, int K, FastDiv chunks,
                                                          uint32_t total) {
    constexpr int U = 4;
    for (uint32_t base = blockIdx.x * (256 * U); base < total; base += gridDim.x * (256 * U)) {
        raw16_t v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {                      // every load before the first store
            const uint32_t idx = min(base + u * 256 + threadIdx.x, total - 1), row = chunks.div(idx);
            const int k = (int)(idx - row * chunks.d) * 8;
            const bf16_t* p = in + (int64_t)row * ld;
            if (k + 8 <= K) {
                v[u] = *reinterpret_cast<const UnalignedVec<bf16_t>::type*>(p + k);
            } else {
                bf16_t e[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) e[i] = k + i < K ? p[k + i] : (bf16_t)0;
                v[u] = *reinterpret_cast<const raw16_t*>(e);
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t idx = base + u * 256 + threadIdx.x;
            if (idx < total) *reinterpret_cast<raw16_t*>(out + (size_t)idx * 8) = v[u];
        }
    }
}

int kmajor_rows(hipStream_t s, const bf16_t* in, int64_t ld, int64_t rows, int64_t K, bf16_t* out, int64_t Kp) {
    const int64_t total = rows * (Kp / 8);
    LUX_INVALID_IF(Kp % 64 != 0 || total >= (int64_t(1) << 31) - 2048, "kmajor_rows: rows of whole steps, fewer than 2^31 chunks");
    const int64_t cus = num_cus() > 0 ? num_cus() : 256;
    ProfScope ps("kmajor_rows_kernel", s);
    kmajor_rows_kernel<<<(unsigned)std::min<int64_t>(ceil_div(total, 1024), 16 * cus), 256, 0, s>>>(in, out, ld, (int)K, FastDiv((uint32_t)(Kp / 8)),
                                                                                                    (uint32_t)total);
    LUX_CHECK_LAUNCH();
    return LUXHIP_OK;
}

// The first pass of a dense pullback, over delta (M x N, m contiguous, columns ld apart): dz = delta .* act'(y, pre) along m
// (columns ldz apart), its transpose dzT along n (rows ldt apart; what the weight-gradient product reads) and the bias gradient's
// partial sums over the 64 columns of a tile.  dz, dzT and partial may be null; with the identity it is a transposing copy.  A 64 x 64 tile
// goes through LDS as fp32 (the sums add unrounded values): phase 1 reads 16-byte vectors along m, stores dz and fills the tile;
// phase 2 reads eight n of one m per thread (rows of 65 words: the 64 lanes of a wave hit 64 banks in both phases), stores 16
// bytes of dzT and adds its eight values; the eight threads of an m add theirs in a fixed order.
// RAGGED: any M, N and alignment of delta, out and pre; ldz and ldt are multiples of 64 then, and dz and dzT are written to the end of the
// tile, with zeros where there is no element.  Otherwise M and N are multiples of 64 and every pointer is 16-byte aligned.
template <int ACT, bool RAGGED>
__global__ __launch_bounds__(256) void dense_dz_kmajor_kernel(const bf16_t* __restrict__ delta, const bf16_t* __restrict__ out,
                                                              const bf16_t* __restrict__ pre, int64_t ld, bf16_t* dz, int64_t ldz,
                                                              bf16_t* __restrict__ dzT, int64_t ldt, float* __restrict__ partial, uint32_t M, uint32_t N) {
    constexpr int PITCH = 65;
    __shared__ float tile[64 * PITCH];
    const uint32_t m0 = blockIdx.x * 64, n0 = blockIdx.y * 64;
    float r[2][8];
#pragma unroll
    for (int it = 0; it < 2; ++it) {                 // loads first, then the stores
        const uint32_t idx = threadIdx.x + it * 256, n = n0 + (idx >> 3), m = m0 + (idx & 7) * 8;
        const size_t off = (size_t)n * ld + m;
        if constexpr (!RAGGED) {
            dx_vec<bf16_t, ACT, 8>(delta, out, pre, off, r[it]);
        } else if (n < N && m + 8 <= M) {
            dx_vec<bf16_t, ACT, 8, true>(delta, out, pre, off, r[it]);
        } else {
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                float v[1] = {0.0f};
                if (n < N && m + k < M) dx_vec<bf16_t, ACT, 1>(delta, out, pre, off + k, v);
                r[it][k] = v[0];
            }
        }
    }
#pragma unroll
    for (int it = 0; it < 2; ++it) {
        const uint32_t idx = threadIdx.x + it * 256, nl = idx >> 3, mv = idx & 7;
        if (dz != nullptr && (!RAGGED || n0 + nl < N)) store_vec<bf16_t, 8>(dz, (size_t)(n0 + nl) * ldz + m0 + mv * 8, r[it]);
#pragma unroll
        for (int k = 0; k < 8; ++k) tile[nl * PITCH + mv * 8 + k] = r[it][k];
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < 2; ++it) {
        const uint32_t idx = threadIdx.x + it * 256, ml = idx >> 3, nv = idx & 7;
        float v[8], sum = 0.0f;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            v[k] = tile[(nv * 8 + k) * PITCH + ml];
            sum += v[k];
        }
        const bool in = !RAGGED || m0 + ml < M;
        if (dzT != nullptr && in) store_vec<bf16_t, 8>(dzT, (size_t)(m0 + ml) * ldt + n0 + nv * 8, v);
        if (partial != nullptr) {
            // the eight threads of this m are neighbouring lanes: (((s0 + s1) + (s2 + s3)) + ((s4 + s5) + (s6 + s7)))
            sum += __shfl_xor(sum, 1);
            sum += __shfl_xor(sum, 2);
            sum += __shfl_xor(sum, 4);
            if (nv == 0 && in) partial[(size_t)blockIdx.y * M + m0 + ml] = sum;
        }
    }
}

int kmajor_transposed(hipStream_t s, const bf16_t* in, int64_t ld, int64_t rows, int64_t K, bf16_t* out, int64_t Kp) {
    LUX_INVALID_IF(Kp % 64 != 0 || K > Kp || ceil_div(K, 64) > 65535, "kmajor_transposed: rows of whole steps");
    const dim3 grid((unsigned)ceil_div(rows, 64), (unsigned)ceil_div(K, 64));
    ProfScope ps("kmajor_transposed_kernel", s);
    dense_dz_kmajor_kernel<LUXHIP_ACT_IDENTITY, true><<<grid, 256, 0, s>>>(in, nullptr, nullptr, ld, nullptr, 0, out, Kp, nullptr, (uint32_t)rows, (uint32_t)K);
    LUX_CHECK_LAUNCH();
    return LUXHIP_OK;
}

int dense_dz_kmajor(hipStream_t s, int act, int64_t M, int64_t N, const bf16_t* delta, const bf16_t* out, const bf16_t* pre, bf16_t* dz, int64_t ldz,
                    bf16_t* dzT, int64_t ldt, float* partial, bf16_t* dbias) {
    LUX_INVALID_IF(ceil_div(N, 64) > 65535, "dense_dz_kmajor: too many columns");
    const bool whole = M % 64 == 0 && N % 64 == 0 && aligned16(delta) && aligned16(out) && aligned16(pre);
    const dim3 grid((unsigned)ceil_div(M, 64), (unsigned)ceil_div(N, 64));
    float* const part = dbias != nullptr ? partial : nullptr;
#define LAUNCH_DZK(A)                                                                                                                    \
    do {                                                                                                                                 \
        if (whole) dense_dz_kmajor_kernel<A, false><<<grid, 256, 0, s>>>(delta, out, pre, M, dz, ldz, dzT, ldt, part, (uint32_t)M, (uint32_t)N); \
        else dense_dz_kmajor_kernel<A, true><<<grid, 256, 0, s>>>(delta, out, pre, M, dz, ldz, dzT, ldt, part, (uint32_t)M, (uint32_t)N);        \
    } while (0)
    {
        ProfScope ps("dense_dz_kmajor_kernel", s);
        LUX_DISPATCH_ACT(act, LAUNCH_DZK);
    }
#undef LAUNCH_DZK
    LUX_CHECK_LAUNCH();
    if (dbias != nullptr) return plane_finalize_dense_bf16(s, partial, dbias, M, ceil_div(N, 64));
    return LUXHIP_OK;
}

}  // namespace luxhip
