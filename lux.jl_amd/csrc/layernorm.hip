// layernorm forward and pullback over an (L, R) view: each of the R columns (L contiguous
// elements) is normalised on its own; gamma/beta (optional) are indexed by the position l.
//
//   forward : one wave (L small) or one workgroup per column keeps the column in registers:
//             mean, variance about the mean and the normalised output from one HBM read.
//   pullback: ln_bwd_dx_kernel, same ownership, delta and x in registers:
//               g = gamma*dy, dx = invstd*(g - mean(g) - xhat*mean(g*xhat))
//             ln_param_grad_kernel: dgamma[l] = sum_r dy*xhat, dbeta[l] = sum_r dy as a column
//             reduction (threads along l, coalesced; R split into slices, partials combined
//             in a fixed order by ln_param_finalize_kernel).
//             ln_bwd_fused_kernel: both in one pass for columns that one wavefront holds.
// Columns of any length are read and written in 16-byte vectors (RowVec in common.h); fp32 1023 x 6001 (24.6 MB a tensor):
// forward 13.9 -> 10.6 us, pullback 17.4 + 11.7 + 4.0 (dx, a second read for the parameters, their sum) -> 18.8 + 5.8 us.
#include <algorithm>

#include "common.h"

namespace luxhip {

constexpr int kLnCache = 8;   // vectors per thread kept in registers

// Vector q of a column of L elements (see RowVec in common.h for columns that are no multiple of a vector)
template <int VEC, bool RAGGED>
__device__ __forceinline__ uint32_t ln_off(uint32_t q, uint32_t L) {
    if constexpr (RAGGED) return min(q * VEC, L - VEC);
    else return q * VEC;
}
template <int VEC, bool RAGGED>
__device__ __forceinline__ uint32_t ln_skip(uint32_t q, uint32_t L) {
    if constexpr (RAGGED) return q * VEC + VEC > L ? q * VEC + VEC - L : 0u;
    else return 0u;
}

// Sum over the threads that share a column: the wave (WAVE) or the workgroup.
template <bool WAVE>
__device__ __forceinline__ float col_sum(float v, float* sm) {
    if constexpr (WAVE) return wave_sum(v);
    else return block_sum(v, sm);
}

// ------------------------------------------------------------------------------- forward
// CACHE: vectors per thread kept in registers; 0: the column is read from memory again
template <typename T, int ACT, int VEC, bool WAVE, int CACHE, bool RAGGED>
__global__ __launch_bounds__(WAVE ? 256 : 1024) void ln_fwd_kernel(const T* __restrict__ x, const T* __restrict__ gamma, const T* __restrict__ beta, T* y,
                              float* save_mean, float* save_invstd, uint32_t L, uint32_t nvec, uint32_t R, float inv_L, float eps) {
    constexpr bool CACHED = CACHE > 0;
    __shared__ float sm[16];
    const uint32_t tpc = WAVE ? 64u : blockDim.x;                       // threads per column
    const uint32_t t = WAVE ? (threadIdx.x & 63u) : threadIdx.x;
    const uint32_t r = WAVE ? blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6) : blockIdx.x;
    if (r >= R) return;                                                 // whole waves / workgroups only
    const size_t base = (size_t)r * L;
    using K = Kept<T, VEC>;
    typename K::type kv[CACHED ? CACHE : 1];   // cached: the column; loads past its end re-read the last vector
    float v[1][VEC];
    auto counts = [&](uint32_t q, int e) { return !RAGGED || (uint32_t)e >= ln_skip<VEC, RAGGED>(q, L); };
    float sum = 0.0f;
    if constexpr (CACHED) {
#pragma unroll
        for (int u = 0; u < CACHE; ++u) kv[u] = kept_load<T, VEC, RAGGED>(x, base + ln_off<VEC, RAGGED>(min(u * tpc + t, nvec - 1), L));
#pragma unroll
        for (int u = 0; u < CACHE; ++u) {
            const uint32_t q = u * tpc + t;
            if (q < nvec) {
                K::get(kv[u], v[0]);
#pragma unroll
                for (int e = 0; e < VEC; ++e) sum += counts(q, e) ? v[0][e] : 0.0f;
            }
        }
    } else {
        for (uint32_t q = t; q < nvec; q += tpc) {
            row_load<T, VEC, RAGGED>(x, base + ln_off<VEC, RAGGED>(q, L), v[0]);
#pragma unroll
            for (int e = 0; e < VEC; ++e) sum += counts(q, e) ? v[0][e] : 0.0f;
        }
    }
    const float mean = col_sum<WAVE>(sum, sm) * inv_L;
    float dev = 0.0f;
    if constexpr (CACHED) {
#pragma unroll
        for (int u = 0; u < CACHE; ++u) {
            const uint32_t q = u * tpc + t;
            if (q < nvec) {
                K::get(kv[u], v[0]);
#pragma unroll
                for (int e = 0; e < VEC; ++e) dev = counts(q, e) ? fmaf(v[0][e] - mean, v[0][e] - mean, dev) : dev;
            }
        }
    } else {
        for (uint32_t q = t; q < nvec; q += tpc) {
            row_load<T, VEC, RAGGED>(x, base + ln_off<VEC, RAGGED>(q, L), v[0]);
#pragma unroll
            for (int e = 0; e < VEC; ++e) dev = counts(q, e) ? fmaf(v[0][e] - mean, v[0][e] - mean, dev) : dev;
        }
    }
    const float var = col_sum<WAVE>(dev, sm) * inv_L;
    const float invstd = 1.0f / sqrtf(var + eps);
    if (t == 0) {
        if (save_mean) save_mean[r] = mean;
        if (save_invstd) save_invstd[r] = invstd;
    }
    auto emit = [&](uint32_t q, const float (&xv)[VEC]) {
        float gm[VEC], bt[VEC], o[VEC];
        if (gamma) {
            row_load<T, VEC, RAGGED>(gamma, ln_off<VEC, RAGGED>(q, L), gm);
            row_load<T, VEC, RAGGED>(beta, ln_off<VEC, RAGGED>(q, L), bt);
        }
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
            const float sc = (gamma ? gm[e] : 1.0f) * invstd;
            const float sh = fmaf(-mean, sc, gamma ? bt[e] : 0.0f);
            o[e] = Act<ACT>::f(fmaf(xv[e], sc, sh));
        }
        row_store<T, VEC, RAGGED>(y, base + ln_off<VEC, RAGGED>(q, L), o, ln_skip<VEC, RAGGED>(q, L));
    };
    if constexpr (CACHED) {
#pragma unroll
        for (int u = 0; u < CACHE; ++u) {
            const uint32_t q = u * tpc + t;
            if (q < nvec) {
                K::get(kv[u], v[0]);
                emit(q, v[0]);
            }
        }
    } else {
        for (uint32_t q = t; q < nvec; q += tpc) {
            row_load<T, VEC, RAGGED>(x, base + ln_off<VEC, RAGGED>(q, L), v[0]);
            emit(q, v[0]);
        }
    }
}

// ------------------------------------------------------------------------------- pullback: dx
// dy for one vector, given the column statistics and the affine parameters at its positions.
template <typename T, int ACT, int VEC, bool RAGGED>
__device__ __forceinline__ void ln_dy(const T* gamma, const T* beta, uint32_t off, float mean, float invstd,
                                      const float (&dv)[VEC], const float (&xv)[VEC], float (&dy)[VEC],
                                      float (&gm)[VEC]) {
    float bt[VEC];
    if (gamma) {
        row_load<T, VEC, RAGGED>(gamma, off, gm);
        if constexpr (ACT != LUXHIP_ACT_IDENTITY) row_load<T, VEC, RAGGED>(beta, off, bt);
    } else {
#pragma unroll
        for (int e = 0; e < VEC; ++e) { gm[e] = 1.0f; bt[e] = 0.0f; }
    }
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
        dy[e] = dv[e];
        if constexpr (ACT != LUXHIP_ACT_IDENTITY) {
            const float sc = gm[e] * invstd;
            const float pre = fmaf(xv[e], sc, fmaf(-mean, sc, bt[e]));
            dy[e] *= Act<ACT>::d(Act<ACT>::f(pre), pre);
        }
    }
}

// the same with the parameters already in registers
template <int ACT, int VEC>
__device__ __forceinline__ void ln_dy_regs(const float (&gm)[VEC], const float (&bt)[VEC], float mean, float invstd,
                                           const float (&dv)[VEC], const float (&xv)[VEC], float (&dy)[VEC]) {
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
        dy[e] = dv[e];
        if constexpr (ACT != LUXHIP_ACT_IDENTITY) {
            const float sc = gm[e] * invstd;
            const float pre = fmaf(xv[e], sc, fmaf(-mean, sc, bt[e]));
            dy[e] *= Act<ACT>::d(Act<ACT>::f(pre), pre);
        }
    }
}

template <typename T, int ACT, int VEC, bool WAVE, int CACHE, bool RAGGED>
__global__ __launch_bounds__(WAVE ? 256 : 1024) void ln_bwd_dx_kernel(const T* __restrict__ delta, const T* __restrict__ x, const T* __restrict__ gamma,
                                 const T* __restrict__ beta, const float* __restrict__ save_mean,
                                 const float* __restrict__ save_invstd, T* dx, uint32_t L, uint32_t nvec, uint32_t R, float inv_L) {
    constexpr bool CACHED = CACHE > 0;
    __shared__ float sm[16];
    const uint32_t tpc = WAVE ? 64u : blockDim.x;
    const uint32_t t = WAVE ? (threadIdx.x & 63u) : threadIdx.x;
    const uint32_t r = WAVE ? blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6) : blockIdx.x;
    if (r >= R) return;
    const size_t base = (size_t)r * L;
    const float mean = save_mean[r], invstd = save_invstd[r];
    using K = Kept<T, VEC>;
    typename K::type kd[CACHED ? CACHE : 1], kv[CACHED ? CACHE : 1];
    float d[1][VEC], v[1][VEC];
    float s1 = 0.0f, s2 = 0.0f;
    auto accumulate = [&](uint32_t q, const float (&dv)[VEC], const float (&xv)[VEC]) {
        float dy[VEC], gm[VEC];
        ln_dy<T, ACT, VEC, RAGGED>(gamma, beta, ln_off<VEC, RAGGED>(q, L), mean, invstd, dv, xv, dy, gm);
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
            if (RAGGED && (uint32_t)e < ln_skip<VEC, RAGGED>(q, L)) continue;
            const float g = gm[e] * dy[e];
            s1 += g;
            s2 = fmaf(g, (xv[e] - mean) * invstd, s2);
        }
    };
    if constexpr (CACHED) {
#pragma unroll
        for (int u = 0; u < CACHE; ++u) {
            const size_t off = base + ln_off<VEC, RAGGED>(min(u * tpc + t, nvec - 1), L);   // past the end: re-read the last vector
            kd[u] = kept_load<T, VEC, RAGGED>(delta, off);
            kv[u] = kept_load<T, VEC, RAGGED>(x, off);
        }
#pragma unroll
        for (int u = 0; u < CACHE; ++u) {
            const uint32_t q = u * tpc + t;
            if (q < nvec) {
                K::get(kd[u], d[0]);
                K::get(kv[u], v[0]);
                accumulate(q, d[0], v[0]);
            }
        }
    } else {
        for (uint32_t q = t; q < nvec; q += tpc) {
            row_load<T, VEC, RAGGED>(delta, base + ln_off<VEC, RAGGED>(q, L), d[0]);
            row_load<T, VEC, RAGGED>(x, base + ln_off<VEC, RAGGED>(q, L), v[0]);
            accumulate(q, d[0], v[0]);
        }
    }
    s1 = col_sum<WAVE>(s1, sm) * inv_L;
    s2 = col_sum<WAVE>(s2, sm) * inv_L;
    auto emit = [&](uint32_t q, const float (&dv)[VEC], const float (&xv)[VEC]) {
        float dy[VEC], gm[VEC], o[VEC];
        ln_dy<T, ACT, VEC, RAGGED>(gamma, beta, ln_off<VEC, RAGGED>(q, L), mean, invstd, dv, xv, dy, gm);
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
            const float xh = (xv[e] - mean) * invstd;
            o[e] = invstd * (gm[e] * dy[e] - s1 - xh * s2);
        }
        row_store<T, VEC, RAGGED>(dx, base + ln_off<VEC, RAGGED>(q, L), o, ln_skip<VEC, RAGGED>(q, L));
    };
    if constexpr (CACHED) {
#pragma unroll
        for (int u = 0; u < CACHE; ++u) {
            const uint32_t q = u * tpc + t;
            if (q < nvec) {
                K::get(kd[u], d[0]);
                K::get(kv[u], v[0]);
                emit(q, d[0], v[0]);
            }
        }
    } else {
        for (uint32_t q = t; q < nvec; q += tpc) {
            row_load<T, VEC, RAGGED>(delta, base + ln_off<VEC, RAGGED>(q, L), d[0]);
            row_load<T, VEC, RAGGED>(x, base + ln_off<VEC, RAGGED>(q, L), v[0]);
            emit(q, d[0], v[0]);
        }
    }
}

// ------------------------------------------------------------------------------- pullback: dx, dgamma, dbeta in one pass
// Columns of up to 64 * kLnCache vectors with affine parameters.  Two wavefronts share a column
// (half of its vectors each, so that the per-position sums fit the register file next to the
// column itself); a pair walks over columns r = pair, pair + P, ... (P pairs in the grid) with
// delta and x of the current column in registers, as ln_bwd_dx_kernel does, and keeps dy * xhat
// and dy of its positions l summed over its columns.  The two pairs of a workgroup add their sums
// in pair order through LDS; row `blockIdx.x` of pg / pb receives the result and
// ln_param_finalize_kernel adds the rows in order.  delta and x are read once.
constexpr int kLnFusedCache = kLnCache / 2;
template <typename T, int ACT, int VEC, int CACHE, bool RAGGED>
__global__ __launch_bounds__(256) void ln_bwd_fused_kernel(const T* __restrict__ delta, const T* __restrict__ x,
                                                           const T* __restrict__ gamma, const T* __restrict__ beta,
                                                           const float* __restrict__ save_mean,
                                                           const float* __restrict__ save_invstd, T* dx, float* pg, float* pb,
                                                           uint32_t L, uint32_t nvec, uint32_t R, float inv_L) {
    __shared__ float red[2][2][128 * VEC];
    __shared__ float colsum[2][2][2];                  // [pair][wave of the pair][s1, s2]
    const uint32_t w = threadIdx.x >> 6, pair = w >> 1, half = w & 1u;
    const uint32_t t = half * 64u + (threadIdx.x & 63u);          // 0..127 inside the pair
    const uint32_t pairs = gridDim.x * 2u;
    using K = Kept<T, VEC>;
    float ag[CACHE][VEC], ab[CACHE][VEC];
#pragma unroll
    for (int u = 0; u < CACHE; ++u)
#pragma unroll
        for (int e = 0; e < VEC; ++e) { ag[u][e] = 0.0f; ab[u][e] = 0.0f; }
    // The affine parameters at this thread's positions are the same for every column: read once and kept as they lie
    // in memory.  (Read inside the second pass they would sit between the dx stores, and a wave's memory operations
    // complete in the order of their issue: every such load would wait for the store before it.)
    typename K::type kgm[CACHE], kbt[CACHE];
    const bool affine = gamma != nullptr;
    if (affine) {
#pragma unroll
        for (int u = 0; u < CACHE; ++u) {
            const size_t off = ln_off<VEC, RAGGED>(min(u * 128u + t, nvec - 1), L);
            kgm[u] = kept_load<T, VEC, RAGGED>(gamma, off);
            if constexpr (ACT != LUXHIP_ACT_IDENTITY) kbt[u] = kept_load<T, VEC, RAGGED>(beta, off);
        }
    }
    auto params = [&](int u, float (&gm)[VEC], float (&bt)[VEC]) {
        if (affine) {
            K::get(kgm[u], gm);
            if constexpr (ACT != LUXHIP_ACT_IDENTITY) K::get(kbt[u], bt);
        } else {
#pragma unroll
            for (int e = 0; e < VEC; ++e) { gm[e] = 1.0f; bt[e] = 0.0f; }
        }
    };
    const uint32_t rounds = (R + pairs - 1) / pairs;              // the same for every wavefront: barriers inside
    for (uint32_t it = 0; it < rounds; ++it) {
        const uint32_t r = it * pairs + blockIdx.x * 2u + pair;
        const bool live = r < R;                                  // uniform per wavefront
        const uint32_t rc = live ? r : R - 1;
        const size_t base = (size_t)rc * L;
        const float mean = save_mean[rc], invstd = save_invstd[rc];
        typename K::type kd[CACHE], kv[CACHE];
#pragma unroll
        for (int u = 0; u < CACHE; ++u) {
            const size_t off = base + ln_off<VEC, RAGGED>(min(u * 128u + t, nvec - 1), L);   // past the end: the last vector again
            kd[u] = kept_load<T, VEC, RAGGED>(delta, off);
            kv[u] = kept_load<T, VEC, RAGGED>(x, off);
        }
        float s1 = 0.0f, s2 = 0.0f;
#pragma unroll
        for (int u = 0; u < CACHE; ++u) {
            const uint32_t q = u * 128u + t;
            if (q < nvec && live) {
                float d[VEC], v[VEC], dy[VEC], gm[VEC], bt[VEC];
                K::get(kd[u], d);
                K::get(kv[u], v);
                params(u, gm, bt);
                ln_dy_regs<ACT, VEC>(gm, bt, mean, invstd, d, v, dy);
#pragma unroll
                for (int e = 0; e < VEC; ++e) {
                    if (RAGGED && (uint32_t)e < ln_skip<VEC, RAGGED>(q, L)) continue;
                    const float xh = (v[e] - mean) * invstd;
                    const float g = gm[e] * dy[e];
                    s1 += g;
                    s2 = fmaf(g, xh, s2);
                    ag[u][e] = fmaf(dy[e], xh, ag[u][e]);
                    ab[u][e] += dy[e];
                }
            }
        }
        s1 = wave_sum(s1);
        s2 = wave_sum(s2);
        if ((threadIdx.x & 63u) == 0) { colsum[pair][half][0] = s1; colsum[pair][half][1] = s2; }
        __syncthreads();
        s1 = (colsum[pair][0][0] + colsum[pair][1][0]) * inv_L;
        s2 = (colsum[pair][0][1] + colsum[pair][1][1]) * inv_L;
        __syncthreads();                                          // colsum is rewritten in the next round
#pragma unroll
        for (int u = 0; u < CACHE; ++u) {
            const uint32_t q = u * 128u + t;
            if (q < nvec && live) {
                float d[VEC], v[VEC], dy[VEC], gm[VEC], bt[VEC], o[VEC];
                K::get(kd[u], d);
                K::get(kv[u], v);
                params(u, gm, bt);
                ln_dy_regs<ACT, VEC>(gm, bt, mean, invstd, d, v, dy);
#pragma unroll
                for (int e = 0; e < VEC; ++e) {
                    const float xh = (v[e] - mean) * invstd;
                    o[e] = invstd * (gm[e] * dy[e] - s1 - xh * s2);
                }
                row_store<T, VEC, RAGGED>(dx, base + ln_off<VEC, RAGGED>(q, L), o, ln_skip<VEC, RAGGED>(q, L));
            }
        }
    }
    // sums of the two pairs, in pair order, one cached vector at a time
    const size_t row = (size_t)blockIdx.x * L;
#pragma unroll
    for (int u = 0; u < CACHE; ++u) {
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
            red[0][pair][t * VEC + e] = ag[u][e];
            red[1][pair][t * VEC + e] = ab[u][e];
        }
        __syncthreads();
        for (uint32_t i = threadIdx.x; i < 128u * VEC; i += 256u) {
            const uint32_t q = u * 128u + i / VEC, e = i % VEC;
            const uint32_t l = ln_off<VEC, RAGGED>(q, L) + e;
            if (q < nvec && e >= ln_skip<VEC, RAGGED>(q, L)) {
                pg[row + l] = red[0][0][i] + red[0][1][i];
                pb[row + l] = red[1][0][i] + red[1][1][i];
            }
        }
        __syncthreads();
    }
}

// ------------------------------------------------------------------------------- pullback: dgamma, dbeta
// grid (ceil(nvec / 64), S): a thread owns one vector of positions l and walks over the
// columns of slice s; partial sums go to pg/pb[s][l].
template <typename T, int ACT, int VEC, bool RAGGED>
__global__ __launch_bounds__(64) void ln_param_grad_kernel(const T* __restrict__ delta, const T* __restrict__ x,
                                                           const T* __restrict__ gamma, const T* __restrict__ beta,
                                                           const float* __restrict__ save_mean,
                                                           const float* __restrict__ save_invstd, float* pg, float* pb,
                                                           uint32_t L, uint32_t nvec, uint32_t R, uint32_t cols_per_slice) {
    const uint32_t q = blockIdx.x * 64 + threadIdx.x;
    if (q >= nvec) return;
    const uint32_t l0 = ln_off<VEC, RAGGED>(q, L);
    const uint32_t r0 = blockIdx.y * cols_per_slice, r1 = min(r0 + cols_per_slice, R);
    float gm[VEC], bt[VEC], ag[VEC], ab[VEC];
    if (gamma) {
        row_load<T, VEC, RAGGED>(gamma, l0, gm);
        row_load<T, VEC, RAGGED>(beta, l0, bt);
    }
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
        ag[e] = 0.0f; ab[e] = 0.0f;
        if (!gamma) { gm[e] = 1.0f; bt[e] = 0.0f; }
    }
    const size_t stride = L;
#pragma unroll 4
    for (uint32_t r = r0; r < r1; ++r) {
        float dv[VEC], xv[VEC];
        row_load<T, VEC, RAGGED>(delta, r * stride + l0, dv);
        row_load<T, VEC, RAGGED>(x, r * stride + l0, xv);
        const float mean = save_mean[r], invstd = save_invstd[r];
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
            float dy = dv[e];
            if constexpr (ACT != LUXHIP_ACT_IDENTITY) {
                const float sc = gm[e] * invstd;
                const float pre = fmaf(xv[e], sc, fmaf(-mean, sc, bt[e]));
                dy *= Act<ACT>::d(Act<ACT>::f(pre), pre);
            }
            ag[e] = fmaf(dy, (xv[e] - mean) * invstd, ag[e]);
            ab[e] += dy;
        }
    }
    const size_t o = (size_t)blockIdx.y * stride + l0;
#pragma unroll
    for (int e = 0; e < VEC; ++e)
        if (!RAGGED || (uint32_t)e >= ln_skip<VEC, RAGGED>(q, L)) { pg[o + e] = ag[e]; pb[o + e] = ab[e]; }
}

// dgamma[l] = sum_s pg[s][l], dbeta likewise.  Workgroup of LW positions x (1024 / LW) slice groups: group g adds slices g, g + G, ...,
// U of each sum in flight whether or not there are as many, and the G group sums are added in group order.  Bound by the latency of the trips:
// the last few slices of a thread took one each (249 slices of 1862 positions: pass 20.2 -> 19.2 us).  16 positions a workgroup or eight loads in
// flight gain nothing with 768 slices and lose with 4096 positions (69.1 -> 72.1 and 69.5).  LW = 32: 128-byte row segments, and
// L / 32 workgroups fill the device for L of a few thousand.
constexpr int kLnFinalizeWidth = 32;
template <typename T>
__global__ __launch_bounds__(1024) void ln_param_finalize_kernel(const float* __restrict__ pg, const float* __restrict__ pb,
                                                                 T* dgamma, T* dbeta, uint32_t L, uint32_t S) {
    constexpr int LW = kLnFinalizeWidth, G = 1024 / LW, U = 4;
    __shared__ float sg[G][LW], sb[G][LW];
    const uint32_t lx = threadIdx.x % LW, grp = threadIdx.x / LW;
    const uint32_t l = blockIdx.x * LW + lx, lc = min(l, L - 1);
    float tg = 0.0f, tb = 0.0f;
    for (uint32_t s = grp; s < S; s += U * G) {
        float vg[U], vb[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {                // past the end: the last slice again, not added
            const size_t at = (size_t)min(s + u * G, S - 1) * L + lc;
            vg[u] = pg[at];
            vb[u] = pb[at];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (s + u * G < S) {
                tg += vg[u];
                tb += vb[u];
            }
        }
    }
    sg[grp][lx] = tg;
    sb[grp][lx] = tb;
    __syncthreads();
    if (grp == 0 && l < L) {
        tg = 0.0f; tb = 0.0f;
#pragma unroll
        for (int g = 0; g < G; ++g) { tg += sg[g][lx]; tb += sb[g][lx]; }
        if (dgamma) st(dgamma + l, tg);
        if (dbeta) st(dbeta + l, tb);
    }
}

// ------------------------------------------------------------------------------- host side
struct LnPlan {
    bool vec, ragged, wave, cached;
    uint32_t nvec;
    unsigned threads, blocks;
};

// Ragged columns (RowVec in common.h) go element by element where vectors would leave most of a wave idle.  Measured, us,
// elements against vectors, 2^24 elements: one pass forward (bf16 also pays for rows at odd addresses) fp32 99 42 / 47, 198
// 28 / 26, 295 24 / 24 (gelu 26 / 29), 390 24 / 22; bf16 98 44 / 73, 258 25 / 24 (gelu 28 / 31), 390 21 / 18, 511 18 / 20.
template <typename T>
static bool ln_ragged_vectors(int64_t L, int64_t nvec) {
    return L > 64 * kLnCache || (nvec * 20 >= 13 * 64 * ceil_div(nvec, 64) && (L * (int64_t)sizeof(T)) % 4 == 0);
}
// The pullback that makes all gradients in one pass has two waves per column: fp32 99 93 / 160, 198 76 / 87, 258 75 / 65;
// bf16 198 65 / 84 (gelu 85 / 135), 390 55 / 49 (72 / 76), 450 54 / 43.  Up to 2048 columns it takes what the two kernels
// and the launch between them do (bf16 257 x 512 8.3 / 7.1, x 2048 9.2 / 11.9), except that long bf16 columns which are too
// many for one each and too few for several lose to the sum of the partial gradients (2293 x 2048 with gelu 24.9 / 32.7,
// x 512 11.6 / 14.6, x 4096 41.9 / 39.1).
template <typename T>
static bool ln_ragged_fused(int64_t L, int64_t R, int64_t nvec) {
    if (sizeof(T) == 2 && L > 2048 && R >= 768 && R < 3072) return false;
    return R <= 2048 || nvec >= (sizeof(T) == 2 ? 52 : 60);
}

// elements: ragged columns one element at a time
template <typename T>
static LnPlan ln_plan(int64_t L, int64_t R, bool ragged, bool elements) {
    constexpr int V = Vec<T>::N;
    LnPlan p;
    p.vec = L >= V && !(ragged && elements);
    p.ragged = p.vec && ragged;
    p.nvec = (uint32_t)ceil_div(L, p.vec ? V : 1);
    p.wave = p.nvec <= 64u * kLnCache;
    if (p.wave) {
        p.cached = true;
        p.threads = 256;                                   // 4 columns per workgroup
        p.blocks = (unsigned)ceil_div(R, 4);
    } else {
        int64_t t = 256;
        while (t < 1024 && t * kLnCache < p.nvec) t <<= 1;
        p.threads = (unsigned)t;
        p.cached = (int64_t)p.nvec <= t * kLnCache;
        p.blocks = (unsigned)R;
    }
    return p;
}

static int ln_check(int dtype, int act, int64_t L, int64_t R) {
    LUX_UNSUPPORTED_IF(dtype != LUXHIP_F32 && dtype != LUXHIP_BF16, "unsupported dtype %d", dtype);
    LUX_UNSUPPORTED_IF(act < 0 || act >= LUXHIP_ACT_COUNT, "unsupported activation id %d", act);
    LUX_INVALID_IF(L < 0 || R < 0, "negative dimension");
    if (L > 0 && R > 0) {
        const long double tot = (long double)L * (long double)R;
        LUX_UNSUPPORTED_IF(tot >= 2147483648.0L, "tensors of 2^31 or more elements are not supported");
    }
    return LUXHIP_OK;
}

// Columns that a wave holds take the variant with as many registers as the column needs (a wave of 256 vectors that is built
// for 512 loads its last vector four times over)
#define LN_ONE(KERNEL, A, VV, WV, CA, RA, ...) launch_exact(ps, KERNEL<T, A, VV, WV, CA, RA>, dim3(p.blocks), dim3(p.threads), 0, s, __VA_ARGS__)
#define LN_RAGGED(KERNEL, A, WV, CA, ...)                                                               \
    do {                                                                                                \
        if (p.ragged) LN_ONE(KERNEL, A, V, WV, CA, true, __VA_ARGS__);                                  \
        else LN_ONE(KERNEL, A, V, WV, CA, false, __VA_ARGS__);                                          \
    } while (0)
#define LN_VARIANTS(KERNEL, A, ...)                                                                     \
    do {                                                                                                \
        if (p.vec && p.wave && p.nvec <= 64u * 4) LN_RAGGED(KERNEL, A, true, 4, __VA_ARGS__);           \
        else if (p.vec && p.wave) LN_RAGGED(KERNEL, A, true, kLnCache, __VA_ARGS__);                    \
        else if (p.vec && p.cached) LN_RAGGED(KERNEL, A, false, kLnCache, __VA_ARGS__);                 \
        else if (p.vec) LN_RAGGED(KERNEL, A, false, 0, __VA_ARGS__);                                    \
        else LN_ONE(KERNEL, A, 1, true, kLnCache, false, __VA_ARGS__);       /* element by element */    \
    } while (0)

template <typename T>
static int ln_fwd_impl(hipStream_t s, int act, int64_t L, int64_t R, const T* x, const T* gamma, const T* beta, float eps,
                       T* y, float* save_mean, float* save_invstd) {
    constexpr int V = Vec<T>::N;
    const bool ptr_ok = aligned16(x) && aligned16(y) && (gamma == nullptr || (aligned16(gamma) && aligned16(beta)));
    const bool ragged = !(ptr_ok && L % V == 0);
    LnPlan p = ln_plan<T>(L, R, ragged, !ln_ragged_vectors<T>(L, ceil_div(L, V)));
    const float inv_L = 1.0f / (float)L;
    ProfScope ps("ln_fwd_kernel", s, true);
#define LN_FWD(A) LN_VARIANTS(ln_fwd_kernel, A, x, gamma, beta, y, save_mean, save_invstd, (uint32_t)L, p.nvec, (uint32_t)R, inv_L, eps)
    LUX_DISPATCH_ACT(act, LN_FWD);
#undef LN_FWD
    LUX_CHECK_LAUNCH();
    return LUXHIP_OK;
}

template <typename T>
static int ln_bwd_impl(hipStream_t s, int act, int64_t L, int64_t R, const T* delta, const T* x, const T* gamma,
                       const T* beta, const float* save_mean, const float* save_invstd, T* dx, T* dgamma, T* dbeta) {
    constexpr int V = Vec<T>::N;
    const bool ptr_ok = aligned16(x) && aligned16(delta) && aligned16(dx) &&
                        (gamma == nullptr || (aligned16(gamma) && aligned16(beta)));
    const bool ragged = !(ptr_ok && L % V == 0), params = gamma != nullptr && (dgamma != nullptr || dbeta != nullptr);
    const int64_t nvec = ceil_div(L, V);
    const bool one_pass = L >= V && nvec <= 64 * kLnCache && params && R >= 64 && (!ragged || ln_ragged_fused<T>(L, R, nvec));
    LnPlan p = ln_plan<T>(L, R, ragged, !one_pass && (params && R >= 64 ? nvec <= 64 * kLnCache : !ln_ragged_vectors<T>(L, nvec)));
    const float inv_L = 1.0f / (float)L;
    if (one_pass) {
        // one pass over delta and x: dx and the per-position sums of every workgroup
        const int64_t blocks = std::min<int64_t>(ceil_div(R, 2), 3 * (int64_t)(num_cus() > 0 ? num_cus() : 256));
        Workspace ws;
        int rc = get_workspace(s, (size_t)2 * blocks * L * sizeof(float), &ws);
        if (rc != LUXHIP_OK) return rc;
        float* pg = reinterpret_cast<float*>(ws.data);
        float* pb = pg + (size_t)blocks * L;
        {
            ProfScope ps("ln_bwd_fused_kernel", s, true);
#define LN_FUSED_V(A, CA, RA) launch_exact(ps, ln_bwd_fused_kernel<T, A, V, CA, RA>, dim3((unsigned)blocks), dim3(256), 0, s, delta, x, gamma, beta, save_mean, save_invstd, dx, pg, pb, (uint32_t)L, p.nvec, (uint32_t)R, inv_L)
#define LN_FUSED(A)                                                                       \
    do {                                                                                  \
        if (p.nvec <= 128u * 2 && p.ragged) LN_FUSED_V(A, 2, true);                       \
        else if (p.nvec <= 128u * 2) LN_FUSED_V(A, 2, false);                             \
        else if (p.ragged) LN_FUSED_V(A, kLnFusedCache, true);                            \
        else LN_FUSED_V(A, kLnFusedCache, false);                                         \
    } while (0)
            LUX_DISPATCH_ACT(act, LN_FUSED);
#undef LN_FUSED
#undef LN_FUSED_V
        }
        LUX_CHECK_LAUNCH();
        ProfScope ps2("ln_param_finalize_kernel", s);
        ln_param_finalize_kernel<T><<<(unsigned)ceil_div(L, kLnFinalizeWidth), 1024, 0, s>>>(pg, pb, dgamma, dbeta, (uint32_t)L, (uint32_t)blocks);
        LUX_CHECK_LAUNCH();
        return LUXHIP_OK;
    }
    {
        ProfScope ps("ln_bwd_dx_kernel", s, true);
#define LN_BWD(A)                                                                                                         \
    do {                                                                                                                  \
        if (!p.vec && !p.wave) LN_ONE(ln_bwd_dx_kernel, A, 1, false, kLnCache, false, delta, x, gamma, beta, save_mean, save_invstd, dx, (uint32_t)L, p.nvec, (uint32_t)R, inv_L); \
        else LN_VARIANTS(ln_bwd_dx_kernel, A, delta, x, gamma, beta, save_mean, save_invstd, dx, (uint32_t)L, p.nvec, (uint32_t)R, inv_L);                       \
    } while (0)
        LUX_DISPATCH_ACT(act, LN_BWD);
#undef LN_BWD
    }
    LUX_CHECK_LAUNCH();
    if (gamma != nullptr && (dgamma != nullptr || dbeta != nullptr)) {
        const int64_t gx = ceil_div(p.nvec, 64);
        int64_t S = std::max<int64_t>(1, std::min<int64_t>(ceil_div(R, 16), ceil_div(2048, gx)));
        const uint32_t cols = (uint32_t)ceil_div(R, S);
        S = ceil_div(R, cols);
        LUX_UNSUPPORTED_IF(S > 65535, "layernorm_bwd: column split too large");
        Workspace ws;
        int rc = get_workspace(s, (size_t)2 * S * L * sizeof(float), &ws);
        if (rc != LUXHIP_OK) return rc;
        float* pg = reinterpret_cast<float*>(ws.data);
        float* pb = pg + (size_t)S * L;
        dim3 grid((unsigned)gx, (unsigned)S);
        {
            ProfScope ps("ln_param_grad_kernel", s);
#define LN_PG(A)                                                                                                           \
    do {                                                                                                                   \
        if (p.ragged) ln_param_grad_kernel<T, A, V, true><<<grid, 64, 0, s>>>(delta, x, gamma, beta, save_mean, save_invstd, pg, pb, (uint32_t)L, p.nvec, (uint32_t)R, cols); \
        else if (p.vec) ln_param_grad_kernel<T, A, V, false><<<grid, 64, 0, s>>>(delta, x, gamma, beta, save_mean, save_invstd, pg, pb, (uint32_t)L, p.nvec, (uint32_t)R, cols); \
        else ln_param_grad_kernel<T, A, 1, false><<<grid, 64, 0, s>>>(delta, x, gamma, beta, save_mean, save_invstd, pg, pb, (uint32_t)L, p.nvec, (uint32_t)R, cols);       \
    } while (0)
            LUX_DISPATCH_ACT(act, LN_PG);
#undef LN_PG
        }
        LUX_CHECK_LAUNCH();
        ProfScope ps2("ln_param_finalize_kernel", s);
        ln_param_finalize_kernel<T><<<(unsigned)ceil_div(L, kLnFinalizeWidth), 1024, 0, s>>>(pg, pb, dgamma, dbeta, (uint32_t)L, (uint32_t)S);
        LUX_CHECK_LAUNCH();
    }
    return LUXHIP_OK;
}

}  // namespace luxhip

using namespace luxhip;

extern "C" {

int luxhip_layernorm_fwd(luxhip_stream_t s, int dtype, int act, int64_t L, int64_t R, const void* x, const void* gamma,
                         const void* beta, double eps, void* y, float* save_mean, float* save_invstd) {
    LUX_REQUIRE_INIT();
    int rc = ln_check(dtype, act, L, R);
    if (rc != LUXHIP_OK) return rc;
    LUX_INVALID_IF((gamma == nullptr) != (beta == nullptr), "layernorm_fwd: gamma and beta must be given together");
    if (L * R == 0) return LUXHIP_OK;
    LUX_INVALID_IF(x == nullptr || y == nullptr, "layernorm_fwd: x and y must not be NULL");
    if (dtype == LUXHIP_F32)
        return ln_fwd_impl<float>((hipStream_t)s, act, L, R, (const float*)x, (const float*)gamma, (const float*)beta,
                                  (float)eps, (float*)y, save_mean, save_invstd);
    return ln_fwd_impl<bf16_t>((hipStream_t)s, act, L, R, (const bf16_t*)x, (const bf16_t*)gamma, (const bf16_t*)beta,
                               (float)eps, (bf16_t*)y, save_mean, save_invstd);
}

int luxhip_layernorm_bwd(luxhip_stream_t s, int dtype, int act, int64_t L, int64_t R, const void* delta, const void* x,
                         const void* gamma, const void* beta, const float* save_mean, const float* save_invstd, void* dx,
                         void* dgamma, void* dbeta) {
    LUX_REQUIRE_INIT();
    int rc = ln_check(dtype, act, L, R);
    if (rc != LUXHIP_OK) return rc;
    LUX_INVALID_IF((gamma == nullptr) != (beta == nullptr), "layernorm_bwd: gamma and beta must be given together");
    if (L * R == 0) {
        if (L > 0 && dgamma) { rc = luxhip_fill_zero(dgamma, (size_t)L * (dtype == LUXHIP_F32 ? 4 : 2), s); if (rc) return rc; }
        if (L > 0 && dbeta) { rc = luxhip_fill_zero(dbeta, (size_t)L * (dtype == LUXHIP_F32 ? 4 : 2), s); if (rc) return rc; }
        return LUXHIP_OK;
    }
    LUX_INVALID_IF(delta == nullptr || x == nullptr || dx == nullptr || save_mean == nullptr || save_invstd == nullptr,
                   "layernorm_bwd: delta, x, dx, save_mean and save_invstd must not be NULL");
    if (dtype == LUXHIP_F32)
        return ln_bwd_impl<float>((hipStream_t)s, act, L, R, (const float*)delta, (const float*)x, (const float*)gamma,
                                  (const float*)beta, save_mean, save_invstd, (float*)dx, (float*)dgamma, (float*)dbeta);
    return ln_bwd_impl<bf16_t>((hipStream_t)s, act, L, R, (const bf16_t*)delta, (const bf16_t*)x, (const bf16_t*)gamma,
                               (const bf16_t*)beta, save_mean, save_invstd, (bf16_t*)dx, (bf16_t*)dgamma, (bf16_t*)dbeta);
}

}  // extern "C"
