// y (M x N) = act.(W (M x K) * x (K x N) .+ bias) for a few columns (N <= 16): serving a handful of tokens.
//
// Bound by reading W once (rows of W contiguous along m).  A wave covers 128 (bf16) or 64 (fp32) consecutive m with its
// sixteen lanes of a quarter, 16 bytes each, and takes 32 (16) k at a time, 8 (4) rows per quarter: eight (four) loads of
// 1 KiB, all of them cache lines that are used whole.  The matrix instructions take any assignment of rows to lanes as
// long as both operands agree, so the loaded registers are A fragments as they come in fp32, and after an in-lane 8 x 8
// transpose of 16-bit values (one v_perm_b32 per dword) in bf16: no LDS, no barrier in the loop.  The sixteen columns of
// the instruction hold the N columns of x (the others repeat the last one and are not stored).  The next 32 k are
// requested before the current ones are used.
//
// Eight waves of a workgroup split its k range and add up in LDS; `slices` workgroups share a block of m, hand their sums
// over through device memory, and the last one to arrive adds them in slice order.
#include <algorithm>

#include "common.h"
#include "gemm_core.h"
#include "gemm_dense_decl.h"

namespace luxhip {
namespace skinny {

constexpr int WAVES = 8, THREADS = WAVES * 64, NMAX = 16;
typedef float f32x4_v __attribute__((ext_vector_type(4)));
template <typename T>
struct Elem {
    static constexpr int V = 16 / (int)sizeof(T);   // elements per 16 bytes: m per lane, and k per quarter and step
};

template <typename T>
struct Args {
    const T *W, *x, *bias;
    T *y, *pre;
    int64_t ldw, ldx, ldy;
    int M, N, K, act, slices, kwave;            // kwave: k per wave, a multiple of 4 V
    float* partial;                             // [block of m][slice][N][16 V]
    uint32_t* counters;
};

template <typename T>
__global__ __launch_bounds__(THREADS) void skinny_gemm_kernel(Args<T> a) {
    constexpr int V = Elem<T>::V, MT = 16 * V, KSTEP = 4 * V;
    using vec = typename UnalignedVec<T>::type;
    __shared__ float sums[WAVES][NMAX * MT];
    __shared__ uint32_t flag;
    const int block = blockIdx.x / a.slices, slice = blockIdx.x - block * a.slices;
    const int m0 = min(block * MT, a.M - MT);
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63, lm = l & 15, lq = l >> 4;
    const int kbeg = (slice * WAVES + w) * a.kwave, kend = min(kbeg + a.kwave, a.K);
    f32x4_v acc[V];
#pragma unroll
    for (int i = 0; i < V; ++i) acc[i] = f32x4_v{0.0f, 0.0f, 0.0f, 0.0f};
    const T* wp = a.W + m0 + lm * V;
    const T* xp = a.x + (int64_t)min(lm, a.N - 1) * a.ldx;
    u32x4_v rw[2][V], rx[2];
    auto fetch_step = [&](int k, u32x4_v (&dw)[V], u32x4_v& dx) {
        const int kl = k + lq * V;
        if (k + KSTEP <= a.K) {                                 // uniform
#pragma unroll
            for (int j = 0; j < V; ++j) dw[j] = *reinterpret_cast<const vec*>(wp + (int64_t)(kl + j) * a.ldw);
            dx = *reinterpret_cast<const vec*>(xp + kl);
        } else {                                                // past the end of K both operands are zero
            T e[V];
#pragma unroll
            for (int j = 0; j < V; ++j) {
                dw[j] = u32x4_v{0u, 0u, 0u, 0u};
                e[j] = T(0);
                if (kl + j < a.K) {
                    dw[j] = *reinterpret_cast<const vec*>(wp + (int64_t)(kl + j) * a.ldw);
                    e[j] = xp[kl + j];
                }
            }
            dx = *reinterpret_cast<const u32x4_v*>(e);
        }
    };
    auto multiply = [&](const u32x4_v (&dw)[V], const u32x4_v& dx) {
        if constexpr (sizeof(T) == 4) {
#pragma unroll
            for (int j = 0; j < V; ++j)
#pragma unroll
                for (int i = 0; i < V; ++i)
                    acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(dw[j][i]), __uint_as_float(dx[j]), acc[i], 0, 0, 0);
        } else {
            const bf16x8_v b = __builtin_bit_cast(bf16x8_v, dx);
#pragma unroll
            for (int i = 0; i < V; ++i) {                       // row i of the lane's eight: element i of each of the eight loads
                u32x4_v f;
#pragma unroll
                for (int p = 0; p < 4; ++p)
                    f[p] = __builtin_amdgcn_perm(dw[2 * p + 1][i / 2], dw[2 * p][i / 2], (i & 1) ? 0x07060302u : 0x05040100u);
                acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_v, f), b, acc[i], 0, 0, 0);
            }
        }
    };
    if (kbeg < kend) {
        fetch_step(kbeg, rw[0], rx[0]);
        int k = kbeg;
        for (; k + 2 * KSTEP <= kend; k += 2 * KSTEP) {
            fetch_step(k + KSTEP, rw[1], rx[1]);
            multiply(rw[0], rx[0]);
            if (k + 2 * KSTEP < kend) fetch_step(k + 2 * KSTEP, rw[0], rx[0]);
            multiply(rw[1], rx[1]);
        }
        if (k < kend) {
            const bool more = k + KSTEP < kend;
            if (more) fetch_step(k + KSTEP, rw[1], rx[1]);
            multiply(rw[0], rx[0]);
            if (more) multiply(rw[1], rx[1]);
        }
    }
    // acc[i][r] of lane l: m = m0 + (4 (l / 16) + r) V + i, n = l % 16
    if (lm < a.N) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int i = 0; i < V; ++i) sums[w][lm * MT + (4 * lq + r) * V + i] = acc[i][r];
    }
    __syncthreads();
    const int total = a.N * MT;
    float v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int e = threadIdx.x + u * THREADS;
        v[u] = 0.0f;
        if (e < total)
#pragma unroll
            for (int q = 0; q < WAVES; ++q) v[u] += sums[q][e];
    }
    if (a.slices > 1) {
        float* mine = a.partial + ((size_t)block * a.slices + slice) * (NMAX * MT);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int e = threadIdx.x + u * THREADS;
            if (e < total) publish(mine + e, v[u]);
        }
        publish_done();
        if (!arrive_last(a.counters + block, (uint32_t)a.slices, &flag)) return;
        const float* all = a.partial + (size_t)block * a.slices * (NMAX * MT);
        // the values of a thread (as many as any has, in the workgroup) and four slices on their way together, without conditions between
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = 0.0f;
        auto add = [&](auto COUNT) {
            constexpr int count = decltype(COUNT)::value;
#pragma unroll 4
            for (int q = 0; q < a.slices; ++q)
#pragma unroll
                for (int u = 0; u < count; ++u)
                    v[u] += fetch(all + (size_t)q * (NMAX * MT) + min((int)threadIdx.x + u * THREADS, total - 1));
        };
        if (w * 64 < total) switch ((total - 1) / THREADS) {        // waves without a value have none to ask for
            case 0: add(std::integral_constant<int, 1>{}); break;
            case 1: add(std::integral_constant<int, 2>{}); break;
            case 2: add(std::integral_constant<int, 3>{}); break;
            default: add(std::integral_constant<int, 4>{}); break;
        }
    }
    // the bias of all values together, and one activation's code for them in one piece
    auto each = [&](auto&& f) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int e = threadIdx.x + u * THREADS, n = e / MT, m = m0 + e % MT;
            if (e < total) f(u, (int64_t)n * a.ldy + m);
        }
    };
    if (a.bias) {
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] += ld(a.bias + m0 + (threadIdx.x + u * THREADS) % MT);
    }
    if (a.pre) each([&](int u, int64_t off) { st(a.pre + off, v[u]); });
    act_vec(a.act, v);
    each([&](int u, int64_t off) { st(a.y + off, v[u]); });
}

template <typename T>
int launch(hipStream_t s, const DenseArgs<T>& d) {
    constexpr int V = Elem<T>::V, MT = 16 * V, KSTEP = 4 * V;
    Args<T> a;
    a.W = d.A.p; a.x = d.B.p; a.bias = d.bias; a.y = d.C; a.pre = d.pre;
    a.ldw = d.A.sk; a.ldx = d.B.sr; a.ldy = d.ldc;
    a.M = d.M; a.N = d.N; a.K = d.K; a.act = d.act;
    const int64_t cus = num_cus() > 0 ? num_cus() : 256, blocks = ceil_div(d.M, MT);
    // At most one workgroup (eight waves with sixteen loads in flight each) per compute unit: a second one gains nothing
    // (11008 x 4096: 18.6 us against 20.4 with two in bf16, 29.7 against 38.2 in fp32).  Below that a workgroup's step of k costs what its 64 (32)
    // KiB take at the 35 bytes per ns that a compute unit loads, the hand-off 3.2 us and 0.2 for each slice's partial sums, apart from their bytes
    // (us, at least two steps a wave before / now: bf16 1355 -> 3753, 2 columns 8.5 / 6.9, 4096 -> 4096, 16 columns 13.7 / 12.1, 12000 -> 704, 6 columns 9.5 / 8.6;
    // fp32 700 -> 2000, 16 columns 7.6 / 6.8; 4096 -> 11008, 3 columns 18.1 / 18.1; 598 -> 1028, 15 columns stays whole: 6.8, in three slices 7.3).
    const double step_us = sizeof(T) == 2 ? 1.9 : 0.95, slice_us = 0.2 + (double)d.N * MT * 4.0 / 35e3;
    int64_t slices = 1;
    double t_best = 1e30;
    for (int64_t sl = 1; sl <= std::max<int64_t>(1, cus / blocks) && sl <= ceil_div(d.K, KSTEP * WAVES); ++sl) {
        const double t = (double)ceil_div(d.K, sl * KSTEP * WAVES) * step_us + (sl > 1 ? 3.2 + (double)sl * slice_us : 0.0);
        if (t < t_best) { t_best = t; slices = sl; }
    }
    if (blocks > (int64_t)kWorkspaceCounters) slices = 1;
    if (slices > 1 && !workspace_holds(s, (size_t)blocks * slices * NMAX * MT * sizeof(float))) slices = 1;
    a.kwave = (int)(ceil_div(ceil_div(d.K, slices * WAVES), KSTEP) * KSTEP);
    a.slices = (int)ceil_div(d.K, (int64_t)a.kwave * WAVES);
    a.partial = nullptr; a.counters = nullptr;
    if (a.slices > 1) {
        Workspace ws;
        const int rc = get_workspace(s, (size_t)blocks * a.slices * NMAX * MT * sizeof(float), &ws);
        if (rc != LUXHIP_OK) return rc;
        a.partial = reinterpret_cast<float*>(ws.data);
        a.counters = ws.counters;
    }
    ProfScope ps(sizeof(T) == 2 ? (a.slices > 1 ? "skinny_gemm_kernel<bf16>+slices" : "skinny_gemm_kernel<bf16>")
                                : (a.slices > 1 ? "skinny_gemm_kernel<f32>+slices" : "skinny_gemm_kernel<f32>"), s);
    skinny_gemm_kernel<T><<<dim3((unsigned)(blocks * a.slices)), dim3(THREADS), 0, s>>>(a);
    LUX_CHECK_LAUNCH();
    return LUXHIP_OK;
}

}  // namespace skinny

// Rows enough for several workgroups per compute unit fill the chip in tiles of 64 columns too, and what those pad costs less
// than the sums over eight waves do here: bf16 keeps to one workgroup per compute unit (one column, tiles against this
// kernel, us: 300000 x 128 18.8 / 24.1, 100000 x 1024 34.4 / 39.6, 30000 x 2048 26.0 / 25.4; 16 columns: 1000000 x 32
// 48.7 / 118.9), fp32, whose matrix rate is a sixteenth, to two where the k of its waves is mostly padding (one column:
// 100000 x 100 18.8 / 25.1, x 128 20.9 / 18.9; 30000 x 256 14.0 / 8.5; nine columns: 300000 x 512 186.2 / 147.0).
// With less than a step of k fp32 keeps to one as well (30000 x 8 4.0 / 5.8, 10000 x 8 4.2 / 3.6).
template <typename T>
static bool skinny_pays(int64_t M, int64_t K) {
    constexpr int V = skinny::Elem<T>::V, MT = 16 * V, KSTEP = 4 * V;
    const int64_t cus = num_cus() > 0 ? num_cus() : 256, blocks = ceil_div(M, MT);
    if (blocks <= (sizeof(T) == 2 || K < KSTEP ? cus : 2 * cus)) return true;
    const int64_t kpad = ceil_div(ceil_div(K, skinny::WAVES), KSTEP) * KSTEP * skinny::WAVES;
    return sizeof(T) == 4 && 7 * K > 4 * kpad + 380;
}

template <typename T>
bool launch_skinny(hipStream_t s, DenseArgs<T>& d, bool ak, bool bk, int* rc) {
    if (ceil_div(d.M, 16 * skinny::Elem<T>::V) * skinny::THREADS >= kMostThreads) return false;      // the tiled kernels are persistent
    if (ak || !bk || d.N > skinny::NMAX || d.N < 1 || d.M < 16 * skinny::Elem<T>::V || d.K < 1 || !skinny_pays<T>(d.M, d.K)) return false;
    *rc = skinny::launch<T>(s, d);
    return true;
}
template bool launch_skinny<float>(hipStream_t, DenseArgs<float>&, bool, bool, int*);
template bool launch_skinny<bf16_t>(hipStream_t, DenseArgs<bf16_t>&, bool, bool, int*);

}  // namespace luxhip
