// Choice of tile and slices for gemm_split.h, and the launch.
#pragma once

#include "gemm_split.h"

namespace luxhip {
namespace split {

struct Choice { int w, slices; };

// Time of a product in microseconds with tiles of 64 w and `slices` slices: one k of a tile costs `alone` ns when the
// workgroup has its compute unit to itself (the latency of a stage) and `shared` ns of the compute unit's time when it is
// full; a hand-off costs a round trip, a trip per slice for the workgroup that adds them, and the partial sums' bytes.
// The constants are fitted to sweeps over tile, slices and sizes from 256 x 64 x 128 to 3651 x 2048 x 1350, in fp32 on the fp32
// instruction: w = 2 computes in three bf16 parts since and is faster than these say (2048^3 0.71 of the time).
template <typename T>
double estimate(int w, int slices, int64_t M, int64_t N, int64_t K) {
    const int64_t cus = num_cus() > 0 ? num_cus() : 256;
    const double alone = sizeof(T) == 2 ? (w == 2 ? 19e-3 : 7e-3) : (w == 2 ? 73e-3 : 24e-3);
    const double shared = sizeof(T) == 2 ? (w == 2 ? 12.5e-3 : 5.5e-3) : (w == 2 ? 70e-3 : 19e-3);
    const double kslice = (double)ceil_div(K, slices);
    const int64_t tiles = ceil_div(M, 64 * w) * ceil_div(N, 64 * w), blocks = tiles * slices;
    double t = std::max(kslice * alone, (double)ceil_div(blocks, cus) * kslice * shared);
    if (slices > 1) t += 1.5 + 0.5 * w * w * slices + blocks * (64.0 * 64.0 * 8.0 * w * w) / 5e6;
    return t;
}
template <typename T>
Choice choose(int64_t M, int64_t N, int64_t K) {
    Choice best{1, 1};
    double t_best = 1e30;
    const int64_t most = std::min<int64_t>(16, std::max<int64_t>(1, K / (2 * GemmTraits<T>::BK)));
    for (int w = 1; w <= (M >= 128 && N >= 128 ? 2 : 1); ++w) {
        const int64_t tiles = ceil_div(M, 64 * w) * ceil_div(N, 64 * w);
        for (int sl = 1; sl <= most; ++sl) {
            if (sl > 1 && tiles > (int64_t)kWorkspaceCounters) break;
            const double t = estimate<T>(w, sl, M, N, K);
            if (t < t_best) { t_best = t; best = Choice{w, sl}; }
        }
    }
    return best;
}

// Tiles, slices and the workspace of one product; `front`: bytes of the workspace in use before it, moved on past what
// the product uses.  Counters from `first_counter` on.
template <typename T, int W>
Plan make_plan(DenseArgs<T>& a, int slices, size_t* front) {
    constexpr int BK = GemmTraits<T>::BK;
    a.tiles_m = (int)ceil_div(a.M, 64 * W);
    a.tiles_n = (int)ceil_div(a.N, 64 * W);
    Plan p{1, a.K, nullptr, nullptr};
    if (slices > 1) {
        p.kslice = (int)(ceil_div(ceil_div(a.K, slices), BK) * BK);
        p.slices = (int)ceil_div(a.K, p.kslice);
    }
    if (p.slices > 1) {
        p.partial = reinterpret_cast<float*>(*front);        // the offset for now
        *front += (size_t)a.tiles_m * a.tiles_n * p.slices * (64 * W) * (64 * W) * sizeof(float);
    }
    return p;
}
inline void place(Plan& p, const Workspace& ws, int first_counter) {
    if (p.slices == 1) return;
    p.partial = reinterpret_cast<float*>(ws.data + reinterpret_cast<size_t>(p.partial));
    p.counters = ws.counters + first_counter;
}

template <typename T, int W, bool AK, bool BKM>
int launch_cfg(hipStream_t s, DenseArgs<T>& a, int slices) {
    using B = Body<T, W, AK, BKM>;
    size_t bytes = 0;
    Plan p = make_plan<T, W>(a, slices, &bytes);
    if (p.slices > 1 && !workspace_holds(s, bytes)) p = make_plan<T, W>(a, 1, &bytes);
    if (p.slices > 1) {
        Workspace ws;
        const int rc = get_workspace(s, bytes, &ws);
        if (rc != LUXHIP_OK) return rc;
        place(p, ws, 0);
    }
    ProfScope ps(sizeof(T) == 2 ? "split_gemm_kernel<bf16>" : "split_gemm_kernel<f32>", s);
    ps.in_parts(split_f32<T, W, W>());
    split_gemm_kernel<T, W, AK, BKM><<<dim3((unsigned)(a.tiles_m * a.tiles_n * p.slices)), dim3(THREADS), B::LDS_BYTES, s>>>(a, p);
    LUX_CHECK_LAUNCH();
    return LUXHIP_OK;
}

template <typename T, int W>
int launch_layouts(hipStream_t s, DenseArgs<T>& a, bool ak, bool bk, int slices) {
    if (ak && bk) return launch_cfg<T, W, true, true>(s, a, slices);
    if (ak) return launch_cfg<T, W, true, false>(s, a, slices);
    if (bk) return launch_cfg<T, W, false, true>(s, a, slices);
    return launch_cfg<T, W, false, false>(s, a, slices);
}
// fp32 tiles of 128 have an object of their own: four kernels of half a megabyte, whose length otherwise moves those of the smaller
// tiles about in memory (517 x 301 x 1023: 16.5 or 17.6 us for the same instructions)
extern template int launch_layouts<float, 2>(hipStream_t, DenseArgs<float>&, bool, bool, int);

}  // namespace split

// The kernels of gemm_split.h take the problem, and are faster on it than the big-tile kernels: those keep whole aligned
// 128 x 128 tiles that nearly fill the chip.  With 160 and more of the 256 compute units in use they are ahead in bf16
// (us, big tiles against these: 1920 x 2048 x 2048 27.4 / 36.3, 1280 x 2048 x 4096 46.9 / 62.0), with 128 they are not
// (1024 x 2048 x 4096 45.5 / 41.9; 1024^3 13.3 / 9.2), nor where K is short (1536 x 2048 x 128 5.6 / 5.3 up to 192 tiles,
// 1920 x 2048 x 128 6.0 / 6.6).  In fp32 the line lies between 192 tiles (1536 x 2048 x 1024 80.4 / 73.0) and 208
// (1664 x 2048 x 1024 81.3 / 88.1; both sides before 128 x 128 tiles took to three bf16 parts).  Aligned operands of less than a tile in one dimension and many tiles in the other are
// streamed by the big-tile kernels as well while K is short (fp32 1000000 x 9 x 100 178.9 / 193.1, bf16 300000 x 9 x 32
// 14.2 / 15.8; but 24 x 200000 x 512 38.7 / 33.8).
template <typename T>
bool split_takes(const DenseArgs<T>& a) {
    using Tr = GemmTraits<T>;
    if (a.M < Tr::VEC || a.N < Tr::VEC || a.K < Tr::BK) return false;
    const int64_t lim = (int64_t(1) << 31) / (256 * (int64_t)sizeof(T));
    if (std::max(a.A.sr, a.A.sk) >= lim || std::max(a.B.sr, a.B.sk) >= lim) return false;
    const int64_t cus = num_cus() > 0 ? num_cus() : 256;
    if (ceil_div(a.M, 64) * ceil_div(a.N, 64) * split::THREADS >= kMostThreads) return false;        // the big-tile kernels are persistent
    if (a.A.vec_ok && a.B.vec_ok && a.K <= 128 && std::min(a.M, a.N) < 64 && ceil_div(std::max(a.M, a.N), 64) > 4 * cus) return false;
    const int64_t busy = sizeof(T) == 2 && a.K >= 512 ? cus / 2 : cus * 3 / 4;
    return !(whole_tiles<T, 128, 128>(a) && (int64_t)(a.M / 128) * (a.N / 128) > busy);
}

template <typename T>
bool launch_split(hipStream_t s, DenseArgs<T>& a, bool ak, bool bk, int* rc) {
    if (!split_takes(a)) return false;
    if constexpr (sizeof(T) == 4) {
        if (launch_small(s, a, ak, bk, rc)) return true;
    }
    const split::Choice c = split::choose<T>(a.M, a.N, a.K);
    *rc = c.w == 2 ? split::launch_layouts<T, 2>(s, a, ak, bk, c.slices) : split::launch_layouts<T, 1>(s, a, ak, bk, c.slices);
    return true;
}

// One launch for two products that do not depend on each other (dW: both operands contiguous along m / n; dx: both along
// k), where both are small, but too large for gemm_small.hip: a launch of its own costs 2 to 4 us.
template <typename T>
bool launch_split_pair(hipStream_t s, DenseArgs<T>& a, DenseArgs<T>& b, int* rc) {
    using namespace split;
    if (!split_takes(a) || !split_takes(b)) return false;
    const Choice ca = choose<T>(a.M, a.N, a.K), cb = choose<T>(b.M, b.N, b.K);
    const int64_t cus = num_cus() > 0 ? num_cus() : 256;
    if (ca.w != 1 || cb.w != 1) return false;
    size_t front = 0;
    Plan pa = make_plan<T, 1>(a, ca.slices, &front), pb = make_plan<T, 1>(b, cb.slices, &front);
    if (front > 0 && !workspace_holds(s, front)) {
        front = 0;
        pa = make_plan<T, 1>(a, 1, &front);
        pb = make_plan<T, 1>(b, 1, &front);
    }
    const int64_t na = (int64_t)a.tiles_m * a.tiles_n * pa.slices, nb = (int64_t)b.tiles_m * b.tiles_n * pb.slices;
    if (na > 2 * cus && nb > 2 * cus) return false;               // each fills the chip by itself
    // one counter for each tile of a product with slices, those of b behind those of a
    const int64_t counters_a = pa.slices > 1 ? (int64_t)a.tiles_m * a.tiles_n : 0;
    const int64_t counters_b = pb.slices > 1 ? (int64_t)b.tiles_m * b.tiles_n : 0;
    if (counters_a + counters_b > (int64_t)kWorkspaceCounters || (na + nb) * THREADS >= kMostThreads) return false;
    if (front > 0) {
        Workspace ws;
        *rc = get_workspace(s, front, &ws);
        if (*rc != LUXHIP_OK) return true;
        place(pa, ws, 0);
        place(pb, ws, (int)counters_a);
    }
    ProfScope ps(sizeof(T) == 2 ? "split_gemm_pair_kernel<bf16>" : "split_gemm_pair_kernel<f32>", s);
    constexpr size_t lds = std::max(Body<T, 1, false, false>::LDS_BYTES, Body<T, 1, true, true>::LDS_BYTES);
    split_gemm_pair_kernel<T><<<dim3((unsigned)(na + nb)), dim3(THREADS), lds, s>>>(a, pa, b, pb, (int)na);
    const hipError_t e = hipGetLastError();
    *rc = e == hipSuccess ? LUXHIP_OK : set_error(LUXHIP_HIP_ERROR, "kernel launch failed: %s", hipGetErrorString(e));
    return true;
}

}  // namespace luxhip
