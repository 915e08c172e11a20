// bias_activation forward / pullback: HBM-bound streaming kernels.
//
// Tensor view: (I, C, N) column-major; element (i, c, n) lives at (n*C + c)*I + i.
// Two reduction layouts for dbias[c] = sum_{i,n} dx[i,c,n]:
//   "channel": workgroup (s, c) streams a slice of channel c's I*N elements (rows of I
//              contiguous elements) -- used when rows are long enough to coalesce;
//   "plane":   the I*C elements of one n are contiguous; a thread owns VEC consecutive plane
//              positions and walks over n -- used when I is small (dense layers: I == 1).
// Reductions are deterministic: per-workgroup partials are combined in a fixed order by a
// small finalize kernel.
#include <algorithm>

#include "common.h"
#include "act_vec.h"

namespace luxhip {

constexpr int kThreads = 256;
constexpr int kUnroll = 4;  // 16-byte vectors per thread; all of a thread's loads are issued before the first use

// ------------------------------------------------------------------------------- forward
// RAGGED: rows of I elements that are no multiple of a vector, or pointers that are not aligned to one (RowVec, common.h): every access stays
// one 16-byte instruction, where an element per thread took eight of two bytes.
// Bound by HBM: the pullback of 70 x 70 x 117 x 39 in bf16 70.9 -> 25.0 us (134 MB), fp32 51 x 51 x 128 x 40 with tanh 29.8 -> 27.4.
template <typename T, int ACT, int VEC, bool HAS_BIAS, bool WRITE_PRE, bool RAGGED>
__global__ __launch_bounds__(kThreads) void bias_act_fwd_kernel(const T* __restrict__ x, const T* __restrict__ bias,
                                                                T* y, T* pre, uint32_t total_vec, uint32_t I, uint32_t vpr, FastDiv rowdiv,
                                                                FastDiv cdiv, uint32_t C) {
    // rowdiv divides a vector index by vpr, the number of vectors per row
    for (uint32_t base = blockIdx.x * (kThreads * kUnroll); base < total_vec; base += gridDim.x * (kThreads * kUnroll)) {
        float v[kUnroll][VEC];
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
            const uint32_t idx = base + u * kThreads + threadIdx.x;
            const RowVec<VEC, RAGGED> rv(min(idx, total_vec - 1), I, vpr, rowdiv);      // past the end: last vector again (ignored below)
            row_load<T, VEC, RAGGED>(x, rv.off, v[u]);
        }
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
            const uint32_t idx = base + u * kThreads + threadIdx.x;
            if (idx < total_vec) {
                const RowVec<VEC, RAGGED> rv(idx, I, vpr, rowdiv);
                float b = 0.0f;
                if constexpr (HAS_BIAS) b = ld(bias + (rv.row - cdiv.div(rv.row) * C));
                float p[VEC], o[VEC];
#pragma unroll
                for (int k = 0; k < VEC; ++k) {
                    p[k] = v[u][k] + b;
                    o[k] = Act<ACT>::f(p[k]);
                }
                if constexpr (WRITE_PRE) row_store<T, VEC, RAGGED>(pre, rv.off, p, rv.skip);
                row_store<T, VEC, RAGGED>(y, rv.off, o, rv.skip);
            }
        }
    }
}

// Plane layout with the bias varying inside a vector (I < VEC, e.g. dense layers where
// I == 1): element e of the flat tensor belongs to channel (e / I) % C.
template <typename T, int ACT, int VEC, bool WRITE_PRE>
__global__ __launch_bounds__(kThreads) void bias_act_fwd_smallI_kernel(const T* __restrict__ x,
                                                                       const T* __restrict__ bias, T* y, T* pre,
                                                                       uint32_t total_vec, FastDiv idiv, FastDiv cdiv,
                                                                       uint32_t C) {
    for (uint32_t base = blockIdx.x * (kThreads * kUnroll); base < total_vec; base += gridDim.x * (kThreads * kUnroll)) {
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
            uint32_t idx = base + u * kThreads + threadIdx.x;
            if (idx < total_vec) {
                float v[VEC], p[VEC], o[VEC];
                Vec<T>::load(x + (size_t)idx * VEC, v);
#pragma unroll
                for (int k = 0; k < VEC; ++k) {
                    uint32_t row = idiv.div(idx * VEC + k);
                    uint32_t c = row - cdiv.div(row) * C;
                    p[k] = v[k] + ld(bias + c);
                    o[k] = Act<ACT>::f(p[k]);
                }
                if constexpr (WRITE_PRE) Vec<T>::store(pre + (size_t)idx * VEC, p);
                Vec<T>::store(y + (size_t)idx * VEC, o);
            }
        }
    }
}

// ------------------------------------------------------------------------------- pullback
// dx only (no bias gradient): flat streaming.
template <typename T, int ACT, int VEC>
__global__ __launch_bounds__(kThreads) void act_bwd_kernel(const T* __restrict__ delta, const T* __restrict__ out,
                                                           const T* __restrict__ pre, T* dx, uint32_t total_vec) {
    for (uint32_t base = blockIdx.x * (kThreads * kUnroll); base < total_vec; base += gridDim.x * (kThreads * kUnroll)) {
        float r[kUnroll][VEC];
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
            const uint32_t li = min(base + u * kThreads + threadIdx.x, total_vec - 1);   // past the end: ignored below
            dx_vec<T, ACT, VEC>(delta, out, pre, (size_t)li * VEC, r[u]);
        }
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
            const uint32_t idx = base + u * kThreads + threadIdx.x;
            if (idx < total_vec) store_vec<T, VEC>(dx, (size_t)idx * VEC, r[u]);
        }
    }
}

constexpr int kChanVecs = 4;   // vectors per thread of the channel-layout pullback

// "channel" layout: grid (S, C).  Workgroup (s, c) handles vectors [s*chunk, (s+1)*chunk) of
// the nq = I*N/VEC vectors of channel c and publishes its partial sum; the workgroup of a
// channel that arrives last adds the S partials in index order (same result on every run).
// FROM_X: `pre` is the operator's input, and the bias is added again (bit for bit what a stored pre-activation holds).  32 x 32 x 64 x 128 in fp32: the
// forward pass writes a tensor less, 16.4 -> 11.2 us.
template <typename T, int ACT, int VEC, bool RAGGED, bool FROM_X>
__global__ __launch_bounds__(kThreads) void bias_act_bwd_channel_kernel(const T* __restrict__ delta,
                                                                        const T* __restrict__ out,
                                                                        const T* __restrict__ pre, const T* __restrict__ bias, T* dx, T* dbias,
                                                                        float* partial, uint32_t* counters,
                                                                        uint32_t cstride, uint32_t nq,
                                                                        uint32_t chunk, FastDiv rowdiv,
                                                                        uint32_t vec_per_row, uint32_t I, uint32_t C) {
    __shared__ float smem[kThreads / 64];
    __shared__ uint32_t last_flag;
    const uint32_t c = blockIdx.y, s = blockIdx.x, S = gridDim.x;
    const uint32_t q0 = s * chunk;
    const uint32_t q1 = min(q0 + chunk, nq);
    float acc = 0.0f;
    std::conditional_t<FROM_X, PlusBias<T, 1>, Stored> pre_of;
    if constexpr (FROM_X) pre_of.b[0] = ld(bias + c);
    // Up to kChanVecs vectors per thread (the usual split): all loads in flight together, and the
    // partial sum is handed over before dx is stored, so the hand-off does not wait for the stores.
    const bool single = chunk <= kThreads * kChanVecs;
    float r0[kChanVecs][VEC];
    size_t off0[kChanVecs];
    uint32_t skip0[kChanVecs];
    bool have0[kChanVecs];
    // vector q of the channel: its offset and the elements that the vector before it holds too
    auto locate = [&](uint32_t q, size_t& off, uint32_t& skip) {
        const uint32_t n = rowdiv.div(q);
        if constexpr (RAGGED) {
            const uint32_t start = (q - n * vec_per_row) * VEC;
            skip = start + VEC > I ? start + VEC - I : 0u;
            off = ((size_t)n * C + c) * I + (start - skip);
        } else {
            skip = 0;
            off = ((size_t)q + (size_t)vec_per_row * ((size_t)n * (C - 1) + c)) * VEC;
        }
    };
    if (single) {
        // all loads of the thread are issued before the first use
#pragma unroll
        for (int u = 0; u < kChanVecs; ++u) {
            const uint32_t q = q0 + u * kThreads + threadIdx.x;
            have0[u] = q < q1;
            const uint32_t qq = have0[u] ? q : q1 - 1;            // past the end: last vector again (ignored)
            locate(qq, off0[u], skip0[u]);
        }
#pragma unroll
        for (int u = 0; u < kChanVecs; ++u) dx_vec<T, ACT, VEC, RAGGED>(delta, out, pre, off0[u], r0[u], pre_of);
#pragma unroll
        for (int u = 0; u < kChanVecs; ++u)
            if (have0[u]) {
#pragma unroll
                for (int k = 0; k < VEC; ++k)
                    if (!RAGGED || (uint32_t)k >= skip0[u]) acc += r0[u][k];
            }
    } else {
        for (uint32_t q = q0 + threadIdx.x; q < q1; q += kThreads) {
            size_t off;
            uint32_t skip;
            locate(q, off, skip);
            float r[VEC];
            dx_vec<T, ACT, VEC, RAGGED>(delta, out, pre, off, r, pre_of);
            if (dx) row_store<T, VEC, RAGGED>(dx, off, r, skip);
#pragma unroll
            for (int k = 0; k < VEC; ++k)
                if (!RAGGED || (uint32_t)k >= skip) acc += r[k];
        }
    }
    acc = block_sum(acc, smem);
    if (threadIdx.x == 0) {
        publish(partial + (size_t)c * S + s, acc);
        publish_done();
    }
    const bool last = arrive_last(counters + (size_t)c * cstride, S, &last_flag);
    if (single && dx) {
#pragma unroll
        for (int u = 0; u < kChanVecs; ++u)
            if (have0[u]) row_store<T, VEC, RAGGED>(dx, off0[u], r0[u], skip0[u]);
    }
    if (!last) return;
    if (threadIdx.x < 64) {
        float t = 0.0f;
        for (uint32_t i = threadIdx.x; i < S; i += 64) t += fetch(partial + (size_t)c * S + i);
        t = wave_sum(t);
        if (threadIdx.x == 0) st(dbias + c, t);
    }
}

// "plane" layout: P = I*C contiguous elements per n.  grid (ceil(P/(T*VEC)), S); a thread
// owns VEC consecutive plane positions and sums over the n of its slice.
template <typename T, int ACT, int VEC, bool FROM_X>
__global__ __launch_bounds__(kThreads) void bias_act_bwd_plane_kernel(const T* __restrict__ delta,
                                                                      const T* __restrict__ out,
                                                                      const T* __restrict__ pre, const T* __restrict__ bias, T* dx, float* partial,
                                                                      uint32_t P, uint32_t N, uint32_t n_per_slice, uint32_t I) {
    const uint32_t p = (blockIdx.x * kThreads + threadIdx.x) * VEC;
    if (p >= P) return;
    const uint32_t n0 = blockIdx.y * n_per_slice, n1 = min(n0 + n_per_slice, N);
    float acc[VEC];
#pragma unroll
    for (int k = 0; k < VEC; ++k) acc[k] = 0.0f;
    std::conditional_t<FROM_X, PlusBias<T, VEC>, Stored> pre_of;
    if constexpr (FROM_X) {
#pragma unroll
        for (int k = 0; k < VEC; ++k) pre_of.b[k] = ld(bias + (p + k) / I);
    }
    // Four n at a time, their loads before the first store: a load behind a store waits for it (a wave's memory
    // operations complete in the order of their issue), so one n per trip pays a store and a load latency per n.
    constexpr uint32_t U = 4;
    uint32_t n = n0;
    for (; n + U <= n1; n += U) {
        float r[U][VEC];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) dx_vec<T, ACT, VEC, false>(delta, out, pre, (size_t)(n + u) * P + p, r[u], pre_of);
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            if (dx) store_vec<T, VEC>(dx, (size_t)(n + u) * P + p, r[u]);
#pragma unroll
            for (int k = 0; k < VEC; ++k) acc[k] += r[u][k];
        }
    }
    for (; n < n1; ++n) {
        const size_t off = (size_t)n * P + p;
        float r[VEC];
        dx_vec<T, ACT, VEC, false>(delta, out, pre, off, r, pre_of);
        if (dx) store_vec<T, VEC>(dx, off, r);
#pragma unroll
        for (int k = 0; k < VEC; ++k) acc[k] += r[k];
    }
#pragma unroll
    for (int k = 0; k < VEC; ++k) partial[(size_t)blockIdx.y * P + p + k] = acc[k];
}

// dbias[c] = sum_s sum_{i<I} partial[s][c*I + i]; one wave per channel.
template <typename T>
__global__ __launch_bounds__(64) void plane_finalize_kernel(const float* __restrict__ partial, T* dbias, uint32_t P,
                                                            uint32_t I, uint32_t S) {
    const uint32_t c = blockIdx.x;
    float acc = 0.0f;
    const uint32_t cnt = S * I;
    for (uint32_t t = threadIdx.x; t < cnt; t += 64) {
        const uint32_t s = t / I, i = t - s * I;
        acc += partial[(size_t)s * P + (size_t)c * I + i];
    }
    acc = wave_sum(acc);
    if (threadIdx.x == 0) st(dbias + c, acc);
}

// I == 1 (dense layout): dbias[c] = sum_s partial[s][c] with threads along c.  Workgroup of COLS channels x 1024 / COLS slice groups: group g
// adds slices g, g + groups, ..., eight loads in flight; the group sums are added in order.  Bound by the latency of the trips: 16 channels give four times the
// workgroups of a quarter of the trips where 64 leave most of the chip idle (1184 channels, 2000 slices 36.1 -> 4.8 us).
template <typename T, int COLS>
__global__ __launch_bounds__(1024) void plane_finalize_dense_kernel(const float* __restrict__ partial, T* dbias, uint32_t C,
                                                                    uint32_t S) {
    constexpr uint32_t GROUPS = 1024 / COLS, U = 8;
    __shared__ float sg[GROUPS][COLS];
    const uint32_t cx = threadIdx.x % COLS, grp = threadIdx.x / COLS;
    const uint32_t c = blockIdx.x * COLS + cx;
    float t = 0.0f;
    if (c < C) {
        uint32_t s = grp;
        for (; s + (U - 1) * GROUPS < S; s += U * GROUPS) {
            float v[U];
#pragma unroll
            for (uint32_t u = 0; u < U; ++u) v[u] = partial[(size_t)(s + u * GROUPS) * C + c];
#pragma unroll
            for (uint32_t u = 0; u < U; ++u) t += v[u];
        }
#pragma unroll 4
        for (; s < S; s += GROUPS) t += partial[(size_t)s * C + c];
    }
    sg[grp][cx] = t;
    __syncthreads();
    if (grp == 0 && c < C) {
        t = 0.0f;
#pragma unroll
        for (uint32_t g = 0; g < GROUPS; ++g) t += sg[g][cx];
        st(dbias + c, t);
    }
}
template <typename T>
static void launch_plane_finalize_dense(hipStream_t s, const float* partial, T* dbias, int64_t C, int64_t S) {
    const int64_t cus = num_cus() > 0 ? num_cus() : 256;
    if (S > 128 && ceil_div(C, 64) < cus) plane_finalize_dense_kernel<T, 16><<<(unsigned)ceil_div(C, 16), 1024, 0, s>>>(partial, dbias, (uint32_t)C, (uint32_t)S);
    else plane_finalize_dense_kernel<T, 64><<<(unsigned)ceil_div(C, 64), 1024, 0, s>>>(partial, dbias, (uint32_t)C, (uint32_t)S);
}

static inline unsigned grid_for(uint32_t total_vec) {
    return (unsigned)ceil_div(total_vec, kThreads * kUnroll);
}

template <typename T>
static int bias_act_fwd_impl(hipStream_t s, int act, int64_t I, int64_t C, int64_t N, const T* x, const T* bias, T* y,
                             T* pre) {
    constexpr int V = Vec<T>::N;
    const int64_t total = I * C * N;
    const bool ptr_ok = aligned16(x) && aligned16(y) && (pre == nullptr || aligned16(pre));
    const FastDiv cdiv((uint32_t)C);
    // rows: without a bias the tensor is one of them; rows below a vector go element by element
    const int64_t len = bias ? I : total, rows = bias ? C * N : 1;
#define LAUNCH_FWD_AS(A, VV, R)                                                                                    \
    do {                                                                                                           \
        const uint32_t vpr = (uint32_t)ceil_div(len, VV), tv = (uint32_t)(vpr * rows);                             \
        const FastDiv rowdiv(vpr);                                                                                 \
        const dim3 grid(grid_for(tv));                                                                             \
        if (bias && pre)                                                                                           \
            launch_exact(ps, bias_act_fwd_kernel<T, A, VV, true, true, R>, grid, dim3(kThreads), 0, s, x, bias, y, pre, tv, (uint32_t)len, vpr, rowdiv, cdiv, (uint32_t)C); \
        else if (bias)                                                                                             \
            launch_exact(ps, bias_act_fwd_kernel<T, A, VV, true, false, R>, grid, dim3(kThreads), 0, s, x, bias, y, pre, tv, (uint32_t)len, vpr, rowdiv, cdiv, (uint32_t)C); \
        else if (pre)                                                                                              \
            launch_exact(ps, bias_act_fwd_kernel<T, A, VV, false, true, R>, grid, dim3(kThreads), 0, s, x, bias, y, pre, tv, (uint32_t)len, vpr, rowdiv, cdiv, (uint32_t)C); \
        else                                                                                                       \
            launch_exact(ps, bias_act_fwd_kernel<T, A, VV, false, false, R>, grid, dim3(kThreads), 0, s, x, bias, y, pre, tv, (uint32_t)len, vpr, rowdiv, cdiv, (uint32_t)C); \
    } while (0)
#define LAUNCH_FWD(A)                                                                                              \
    do {                                                                                                           \
        if (ptr_ok && len % V == 0) {                                                                              \
            LAUNCH_FWD_AS(A, V, false);                                                                            \
        } else if (ptr_ok && bias && I < 4 * V && total % V == 0) {                                                \
            const uint32_t tv = (uint32_t)(total / V);                                                             \
            const FastDiv idiv((uint32_t)I);                                                                       \
            if (pre)                                                                                               \
                bias_act_fwd_smallI_kernel<T, A, V, true><<<grid_for(tv), kThreads, 0, s>>>(x, bias, y, pre, tv, idiv, cdiv, (uint32_t)C); \
            else                                                                                                   \
                bias_act_fwd_smallI_kernel<T, A, V, false><<<grid_for(tv), kThreads, 0, s>>>(x, bias, y, pre, tv, idiv, cdiv, (uint32_t)C); \
        } else if (len >= V) {                                                                                     \
            LAUNCH_FWD_AS(A, V, true);                                                                             \
        } else {                                                                                                   \
            LAUNCH_FWD_AS(A, 1, false);                                                                            \
        }                                                                                                          \
    } while (0)
    {
        ProfScope ps("bias_act_fwd_kernel", s, true);
        LUX_DISPATCH_ACT(act, LAUNCH_FWD);
    }
#undef LAUNCH_FWD_AS
#undef LAUNCH_FWD
    LUX_CHECK_LAUNCH();
    return LUXHIP_OK;
}

// Where the pullback's scratch memory (partial sums, arrival counters) comes from: the stream's
// workspace, which may allocate, or a fixed block handed in by the entry point that allocates nothing.
struct FixedScratch {
    float* partial;
    size_t partial_bytes;
    uint32_t* counters;      // kWorkspaceCounters words, zero
};
static int bwd_scratch(hipStream_t s, const FixedScratch* fixed, size_t bytes, float** partial, uint32_t** counters) {
    if (fixed != nullptr) {
        LUX_INVALID_IF(bytes > fixed->partial_bytes,
                       "bias_activation_bwd_noalloc: this shape needs %zu bytes of scratch memory, the fixed block has %zu", bytes,
                       fixed->partial_bytes);
        *partial = fixed->partial;
        *counters = fixed->counters;
        return LUXHIP_OK;
    }
    Workspace ws;
    int rc = get_workspace(s, bytes, &ws);
    if (rc != LUXHIP_OK) return rc;
    *partial = reinterpret_cast<float*>(ws.data);
    *counters = ws.counters;
    return LUXHIP_OK;
}

template <typename T>
static int bias_act_bwd_impl(hipStream_t s, int act, int64_t I, int64_t C, int64_t N, const T* delta, const T* out,
                             const T* pre, const T* bias, T* dx, T* dbias, const FixedScratch* fixed = nullptr) {
    constexpr int V = Vec<T>::N;
    const int64_t total = I * C * N;
    const bool ptr_ok = aligned16(delta) && aligned16(dx) && (out == nullptr || aligned16(out)) &&
                        (pre == nullptr || aligned16(pre));
    if (dbias == nullptr) {
#define LAUNCH_ACT_BWD(A)                                                                                   \
    do {                                                                                                    \
        if (ptr_ok && total % V == 0) {                                                                     \
            const uint32_t tv = (uint32_t)(total / V);                                                      \
            act_bwd_kernel<T, A, V><<<grid_for(tv), kThreads, 0, s>>>(delta, out, pre, dx, tv);             \
        } else {                                                                                            \
            act_bwd_kernel<T, A, 1><<<grid_for((uint32_t)total), kThreads, 0, s>>>(delta, out, pre, dx, (uint32_t)total); \
        }                                                                                                   \
    } while (0)
        {
            ProfScope ps("act_bwd_kernel", s);
            LUX_DISPATCH_ACT(act, LAUNCH_ACT_BWD);
        }
#undef LAUNCH_ACT_BWD
        LUX_CHECK_LAUNCH();
        return LUXHIP_OK;
    }

    const bool channel_layout = I >= 64 && C <= 65535;
    if (channel_layout) {
        const bool whole = ptr_ok && I % V == 0;
        const uint32_t vpr = (uint32_t)ceil_div(I, V), nq = (uint32_t)(vpr * N);
        int64_t S = ceil_div(nq, kThreads * kChanVecs);
        const int64_t smax = std::min<int64_t>(kThreads, std::max<int64_t>(1, 16384 / C));
        if (S > smax) S = smax;
        if (S < 1) S = 1;
        const uint32_t chunk = (uint32_t)ceil_div(nq, S);
        S = ceil_div(nq, chunk);
        float* partial = nullptr;
        uint32_t* counters = nullptr;
        int rc = bwd_scratch(s, fixed, (size_t)C * S * sizeof(float), &partial, &counters);
        if (rc != LUXHIP_OK) return rc;
        const FastDiv rowdiv(vpr);
        dim3 grid((unsigned)S, (unsigned)C);
#define LAUNCH_CH_AS(A, R, X)                                                                                      \
    launch_exact(ps, bias_act_bwd_channel_kernel<T, A, V, R, X>, dim3(grid), dim3(kThreads), 0, s, delta, out, pre, bias, dx, dbias, partial, counters, counter_stride(C), nq, chunk, rowdiv, vpr, (uint32_t)I, (uint32_t)C)
#define LAUNCH_CH(A)                                                                                               \
    do {                                                                                                           \
        if (bias != nullptr && Act<A>::needs_pre) {                                                                \
            if (whole) LAUNCH_CH_AS(A, false, Act<A>::needs_pre);                                                  \
            else LAUNCH_CH_AS(A, true, Act<A>::needs_pre);                                                         \
        } else if (whole) {                                                                                        \
            LAUNCH_CH_AS(A, false, false);                                                                         \
        } else {                                                                                                   \
            LAUNCH_CH_AS(A, true, false);                                                                          \
        }                                                                                                          \
    } while (0)
        {
            ProfScope ps("bias_act_bwd_channel_kernel", s, true);
            LUX_DISPATCH_ACT(act, LAUNCH_CH);
        }
#undef LAUNCH_CH
#undef LAUNCH_CH_AS
        LUX_CHECK_LAUNCH();
        return LUXHIP_OK;
    }

    // plane layout
    const int64_t P = I * C;
    const bool vec = ptr_ok && P % V == 0;
    const int vv = vec ? V : 1;
    const int64_t gx = ceil_div(P, (int64_t)kThreads * vv);
    int64_t S = std::max<int64_t>(1, std::min<int64_t>(ceil_div(N, 8), ceil_div(2048, gx)));
    const uint32_t n_per_slice = (uint32_t)ceil_div(N, S);
    S = ceil_div(N, n_per_slice);
    LUX_UNSUPPORTED_IF(S > 65535, "bias_activation_bwd: batch split too large");
    float* partial = nullptr;
    uint32_t* counters_unused = nullptr;
    int rc = bwd_scratch(s, fixed, (size_t)P * S * sizeof(float), &partial, &counters_unused);
    if (rc != LUXHIP_OK) return rc;
    dim3 grid((unsigned)gx, (unsigned)S);
#define LAUNCH_PL_AS(A, VV, X)                                                                                     \
    bias_act_bwd_plane_kernel<T, A, VV, X><<<grid, kThreads, 0, s>>>(delta, out, pre, bias, dx, partial, (uint32_t)P, (uint32_t)N, n_per_slice, (uint32_t)I)
#define LAUNCH_PL(A)                                                                                               \
    do {                                                                                                           \
        if (bias != nullptr && Act<A>::needs_pre) {                                                                \
            if (vec) LAUNCH_PL_AS(A, V, Act<A>::needs_pre);                                                        \
            else LAUNCH_PL_AS(A, 1, Act<A>::needs_pre);                                                            \
        } else if (vec) {                                                                                          \
            LAUNCH_PL_AS(A, V, false);                                                                             \
        } else {                                                                                                   \
            LAUNCH_PL_AS(A, 1, false);                                                                             \
        }                                                                                                          \
    } while (0)
    {
        ProfScope ps("bias_act_bwd_plane_kernel", s);
        LUX_DISPATCH_ACT(act, LAUNCH_PL);
    }
#undef LAUNCH_PL
#undef LAUNCH_PL_AS
    LUX_CHECK_LAUNCH();
    ProfScope ps2("plane_finalize_kernel", s);
    if (I == 1) launch_plane_finalize_dense<T>(s, partial, dbias, C, S);
    else plane_finalize_kernel<T><<<(unsigned)C, 64, 0, s>>>(partial, dbias, (uint32_t)P, (uint32_t)I, (uint32_t)S);
    LUX_CHECK_LAUNCH();
    return LUXHIP_OK;
}

static int check_common(int dtype, int act, int64_t I, int64_t C, int64_t N) {
    LUX_UNSUPPORTED_IF(dtype != LUXHIP_F32 && dtype != LUXHIP_BF16, "unsupported dtype %d", dtype);
    LUX_UNSUPPORTED_IF(act < 0 || act >= LUXHIP_ACT_COUNT, "unsupported activation id %d", act);
    LUX_INVALID_IF(I < 0 || C < 0 || N < 0, "negative dimension (%lld, %lld, %lld)", (long long)I, (long long)C, (long long)N);
    // 31-bit element indexing inside the kernels
    if (I > 0 && C > 0 && N > 0) {
        const long double tot = (long double)I * (long double)C * (long double)N;
        LUX_UNSUPPORTED_IF(tot >= 2147483648.0L, "tensors of 2^31 or more elements are not supported");
    }
    return LUXHIP_OK;
}

int plane_finalize_dense_bf16(hipStream_t s, const float* partial, bf16_t* dbias, int64_t M, int64_t slices) {
    ProfScope ps("plane_finalize_kernel", s);
    launch_plane_finalize_dense<bf16_t>(s, partial, dbias, M, slices);
    LUX_CHECK_LAUNCH();
    return LUXHIP_OK;
}

// Shared with the dense and convolution pullbacks: dx may be NULL (bias gradient only).
int bias_act_bwd_dispatch(hipStream_t s, int dtype, int act, int64_t I, int64_t C, int64_t N, const void* delta,
                          const void* out, const void* pre, void* dx, void* dbias) {
    int rc = check_common(dtype, act, I, C, N);
    if (rc != LUXHIP_OK) return rc;
    if (I * C * N == 0) {
        if (dbias != nullptr && C > 0) return luxhip_fill_zero(dbias, (size_t)C * (dtype == LUXHIP_F32 ? 4 : 2), s);
        return LUXHIP_OK;
    }
    if (dx == nullptr && dbias == nullptr) return LUXHIP_OK;
    if (dtype == LUXHIP_F32)
        return bias_act_bwd_impl<float>(s, act, I, C, N, (const float*)delta, (const float*)out, (const float*)pre,
                                        nullptr, (float*)dx, (float*)dbias);
    return bias_act_bwd_impl<bf16_t>(s, act, I, C, N, (const bf16_t*)delta, (const bf16_t*)out, (const bf16_t*)pre,
                                     nullptr, (bf16_t*)dx, (bf16_t*)dbias);
}


// Storage conversion fp32 <-> bf16 (round to nearest even), for operands of mixed storage types that
// are promoted before a fused operator and for taking their gradients back.
template <typename TI, typename TO>
__global__ __launch_bounds__(256) void convert_kernel(const TI* __restrict__ in, TO* __restrict__ out, size_t n) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) st(out + i, ld(in + i));
}
// Eight elements per thread with 16-byte accesses on both sides (n a multiple of 8, both pointers 16-byte aligned).
template <typename T, int K>
__device__ __forceinline__ void load8(const T* p, float (&v)[8]) {
    if constexpr (sizeof(T) == 2) {
        Vec<bf16_t>::load(reinterpret_cast<const bf16_t*>(p), v);
    } else {
        float a[4], b[4];
        Vec<float>::load(reinterpret_cast<const float*>(p), a);
        Vec<float>::load(reinterpret_cast<const float*>(p) + 4, b);
#pragma unroll
        for (int i = 0; i < 4; ++i) { v[i] = a[i]; v[4 + i] = b[i]; }
    }
}
template <typename T>
__device__ __forceinline__ void store8(T* p, const float (&v)[8]) {
    if constexpr (sizeof(T) == 2) {
        Vec<bf16_t>::store(reinterpret_cast<bf16_t*>(p), v);
    } else {
        const float a[4] = {v[0], v[1], v[2], v[3]}, b[4] = {v[4], v[5], v[6], v[7]};
        Vec<float>::store(reinterpret_cast<float*>(p), a);
        Vec<float>::store(reinterpret_cast<float*>(p) + 4, b);
    }
}
template <typename TI, typename TO>
__global__ __launch_bounds__(256) void convert_vec_kernel(const TI* __restrict__ in, TO* __restrict__ out, size_t nvec) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < nvec; i += (size_t)gridDim.x * 256) {
        float v[8];
        load8<TI, 8>(in + i * 8, v);
        store8<TO>(out + i * 8, v);
    }
}

// ------------------------------------------------------------------------------- scratch of the entry point that allocates nothing
// luxhip_bias_activation_bwd_noalloc keeps its partial sums and arrival counters in this array instead
// of the stream's workspace.  Every device the library runs on holds its own copy for the life of the
// process.  In host code the array's name is only a handle for hipGetSymbolAddress: the device
// address it returns (kept per device in g_noalloc_ptr) is what kernels and fills receive.
constexpr size_t kNoAllocCounterBytes = kWorkspaceCounters * sizeof(uint32_t);    // 256 KiB
constexpr size_t kNoAllocPartialBytes = size_t(2) << 20;                          // 2 MiB of partial sums
constexpr int kNoAllocMaxDevices = 64;
static __device__ __align__(256) unsigned char scratch[kNoAllocCounterBytes + kNoAllocPartialBytes];
static unsigned char* g_noalloc_ptr[kNoAllocMaxDevices] = {};

// Called by luxhip_init with `device` current.
int noalloc_setup(int device) {
    LUX_INVALID_IF(device < 0 || device >= kNoAllocMaxDevices, "device %d beyond the %d the library keeps scratch blocks for", device,
                   kNoAllocMaxDevices);
    if (g_noalloc_ptr[device] != nullptr) return LUXHIP_OK;
    unsigned char* ptr = nullptr;
    LUX_CHECK_HIP(hipGetSymbolAddress((void**)&ptr, HIP_SYMBOL(scratch)));
    LUX_INVALID_IF(ptr == nullptr, "hipGetSymbolAddress returned no address for the scratch block");
    g_noalloc_ptr[device] = ptr;
    return LUXHIP_OK;
}

__global__ void fill_zero_words_kernel(uint32_t* p, size_t nwords) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < nwords) p[i] = 0u;
}

}  // namespace luxhip

using namespace luxhip;

extern "C" {

int luxhip_bias_activation_fwd(luxhip_stream_t s, int dtype, int act, int64_t I, int64_t C, int64_t N, const void* x,
                               const void* bias, void* y, void* pre) {
    LUX_REQUIRE_INIT();
    int rc = check_common(dtype, act, I, C, N);
    if (rc != LUXHIP_OK) return rc;
    if (I * C * N == 0) return LUXHIP_OK;
    LUX_INVALID_IF(x == nullptr || y == nullptr, "bias_activation_fwd: x and y must not be NULL");
    if (dtype == LUXHIP_F32)
        return bias_act_fwd_impl<float>((hipStream_t)s, act, I, C, N, (const float*)x, (const float*)bias, (float*)y, (float*)pre);
    return bias_act_fwd_impl<bf16_t>((hipStream_t)s, act, I, C, N, (const bf16_t*)x, (const bf16_t*)bias, (bf16_t*)y, (bf16_t*)pre);
}

int luxhip_bias_activation_bwd(luxhip_stream_t s, int dtype, int act, int64_t I, int64_t C, int64_t N,
                               const void* delta, const void* out, const void* pre, void* dx, void* dbias) {
    LUX_REQUIRE_INIT();
    int rc = check_common(dtype, act, I, C, N);
    if (rc != LUXHIP_OK) return rc;
    if (I * C * N == 0) {
        if (dbias != nullptr && C > 0) return luxhip_fill_zero(dbias, (size_t)C * (dtype == LUXHIP_F32 ? 4 : 2), s);
        return LUXHIP_OK;
    }
    LUX_INVALID_IF(delta == nullptr || dx == nullptr, "bias_activation_bwd: delta and dx must not be NULL");
    LUX_INVALID_IF(act != LUXHIP_ACT_IDENTITY && !act_needs_pre(act) && out == nullptr,
                   "bias_activation_bwd: activation %d needs `out`", act);
    LUX_INVALID_IF(act_needs_pre(act) && pre == nullptr, "bias_activation_bwd: activation %d needs `pre`", act);
    if (dtype == LUXHIP_F32)
        return bias_act_bwd_impl<float>((hipStream_t)s, act, I, C, N, (const float*)delta, (const float*)out,
                                        (const float*)pre, nullptr, (float*)dx, (float*)dbias);
    return bias_act_bwd_impl<bf16_t>((hipStream_t)s, act, I, C, N, (const bf16_t*)delta, (const bf16_t*)out,
                                     (const bf16_t*)pre, nullptr, (bf16_t*)dx, (bf16_t*)dbias);
}

int luxhip_bias_activation_bwd_from_x(luxhip_stream_t s, int dtype, int act, int64_t I, int64_t C, int64_t N, const void* delta, const void* out,
                                      const void* x, const void* bias, void* dx, void* dbias) {
    LUX_REQUIRE_INIT();
    LUX_INVALID_IF(bias != nullptr && dbias == nullptr, "bias_activation_bwd_from_x: dbias must not be NULL where there is a bias");
    if (bias == nullptr || !act_needs_pre(act)) return luxhip_bias_activation_bwd(s, dtype, act, I, C, N, delta, out, x, dx, dbias);
    int rc = check_common(dtype, act, I, C, N);
    if (rc != LUXHIP_OK) return rc;
    if (I * C * N == 0) return C > 0 ? luxhip_fill_zero(dbias, (size_t)C * (dtype == LUXHIP_F32 ? 4 : 2), s) : LUXHIP_OK;
    LUX_INVALID_IF(delta == nullptr || dx == nullptr || x == nullptr, "bias_activation_bwd_from_x: delta, x and dx must not be NULL");
    if (dtype == LUXHIP_F32)
        return bias_act_bwd_impl<float>((hipStream_t)s, act, I, C, N, (const float*)delta, (const float*)out, (const float*)x, (const float*)bias,
                                        (float*)dx, (float*)dbias);
    return bias_act_bwd_impl<bf16_t>((hipStream_t)s, act, I, C, N, (const bf16_t*)delta, (const bf16_t*)out, (const bf16_t*)x, (const bf16_t*)bias,
                                     (bf16_t*)dx, (bf16_t*)dbias);
}
int luxhip_bias_activation_bwd_noalloc(luxhip_stream_t s, int dtype, int act, int64_t I, int64_t C, int64_t N,
                                       const void* delta, const void* out, const void* pre, void* dx, void* dbias) {
    LUX_REQUIRE_INIT();
    int rc = check_common(dtype, act, I, C, N);
    if (rc != LUXHIP_OK) return rc;
    int device = -1;
    LUX_CHECK_HIP(hipGetDevice(&device));
    unsigned char* const block = (device >= 0 && device < kNoAllocMaxDevices) ? g_noalloc_ptr[device] : nullptr;
    LUX_INVALID_IF(block == nullptr, "bias_activation_bwd_noalloc: no scratch block on device %d (luxhip_init sets it up)", device);
    if (I * C * N == 0) {
        if (dbias != nullptr && C > 0) return luxhip_fill_zero(dbias, (size_t)C * (dtype == LUXHIP_F32 ? 4 : 2), s);
        return LUXHIP_OK;
    }
    LUX_INVALID_IF(delta == nullptr || dx == nullptr, "bias_activation_bwd_noalloc: delta and dx must not be NULL");
    LUX_INVALID_IF(act != LUXHIP_ACT_IDENTITY && !act_needs_pre(act) && out == nullptr,
                   "bias_activation_bwd_noalloc: activation %d needs `out`", act);
    LUX_INVALID_IF(act_needs_pre(act) && pre == nullptr, "bias_activation_bwd_noalloc: activation %d needs `pre`", act);
    FixedScratch fx;
    fx.counters = reinterpret_cast<uint32_t*>(block);
    fx.partial = reinterpret_cast<float*>(block + kNoAllocCounterBytes);
    fx.partial_bytes = kNoAllocPartialBytes;
    if (dbias != nullptr) {
        // the block keeps what the last call left: the arrival counters this call uses start at zero (a fill
        // kernel, which a recording stream can hold, unlike a memset node)
        const size_t words = std::min<size_t>((size_t)C * counter_stride(C), kWorkspaceCounters);
        fill_zero_words_kernel<<<dim3((unsigned)ceil_div((int64_t)words, 256)), dim3(256), 0, (hipStream_t)s>>>(fx.counters, words);
        LUX_CHECK_LAUNCH();
    }
    if (dtype == LUXHIP_F32)
        return bias_act_bwd_impl<float>((hipStream_t)s, act, I, C, N, (const float*)delta, (const float*)out, (const float*)pre,
                                        nullptr, (float*)dx, (float*)dbias, &fx);
    return bias_act_bwd_impl<bf16_t>((hipStream_t)s, act, I, C, N, (const bf16_t*)delta, (const bf16_t*)out, (const bf16_t*)pre,
                                     nullptr, (bf16_t*)dx, (bf16_t*)dbias, &fx);
}

int luxhip_convert(luxhip_stream_t s, int dtype_in, int dtype_out, int64_t n, const void* in, void* out) {
    LUX_REQUIRE_INIT();
    LUX_UNSUPPORTED_IF((dtype_in != LUXHIP_F32 && dtype_in != LUXHIP_BF16) || (dtype_out != LUXHIP_F32 && dtype_out != LUXHIP_BF16),
                       "convert: unsupported dtype %d -> %d", dtype_in, dtype_out);
    LUX_INVALID_IF(n < 0, "convert: negative length");
    if (n == 0) return LUXHIP_OK;
    LUX_INVALID_IF(in == nullptr || out == nullptr, "convert: in and out must not be NULL");
    const unsigned blocks = (unsigned)std::min<int64_t>((n + 255) / 256, 65535 * 8);
    const hipStream_t st_ = (hipStream_t)s;
    ProfScope ps("convert_kernel", st_);
    if (dtype_in == dtype_out)
        return luxhip_memcpy_d2d(out, in, (size_t)n * (dtype_in == LUXHIP_F32 ? 4 : 2), s);
    if (n % 8 == 0 && aligned16(in) && aligned16(out)) {
        const unsigned vblocks = (unsigned)std::min<int64_t>((n / 8 + 255) / 256, 65535 * 8);
        if (dtype_in == LUXHIP_BF16)
            convert_vec_kernel<bf16_t, float><<<vblocks, 256, 0, st_>>>((const bf16_t*)in, (float*)out, (size_t)(n / 8));
        else
            convert_vec_kernel<float, bf16_t><<<vblocks, 256, 0, st_>>>((const float*)in, (bf16_t*)out, (size_t)(n / 8));
    } else if (dtype_in == LUXHIP_BF16)
        convert_kernel<bf16_t, float><<<blocks, 256, 0, st_>>>((const bf16_t*)in, (float*)out, (size_t)n);
    else
        convert_kernel<float, bf16_t><<<blocks, 256, 0, st_>>>((const float*)in, (bf16_t*)out, (size_t)n);
    LUX_CHECK_LAUNCH();
    return LUXHIP_OK;
}

}  // extern "C"
