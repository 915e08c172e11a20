// Tile, slices and launch of the kernels of conv_any.h.
#pragma once

#include "conv_any.h"

namespace luxhip {
namespace cany {

// Cost of one k of a tile in us: with the compute unit to itself (latency), and of a full compute unit's time.  Fitted to
// forced launches of 24 problems (M from 196 to 400000 rows, 16 to 208 columns, K from 16 to 5200); a tile's prologue and
// epilogue count as another 100 k.  (fp32 128 x 128: of the fp32 instruction, on which the other fp32 tiles still are.  In three bf16 parts
// those take about 0.65 of it, so that sizes near the line go to smaller tiles that no longer are the faster ones.)
struct Tile { int m, n; double alone, shared; };
template <typename T>
inline const Tile* tiles() {
    static const Tile bf16[5] = {{64, 64, 9e-3, 5.6e-3}, {128, 64, 14e-3, 9.6e-3}, {128, 128, 18e-3, 19e-3}, {256, 32, 18e-3, 12e-3}, {128, 32, 13e-3, 6.4e-3}};
    static const Tile f32[5] = {{64, 64, 29e-3, 20e-3}, {128, 64, 48e-3, 37e-3}, {128, 128, 80e-3, 70e-3}, {256, 32, 60e-3, 45e-3}, {128, 32, 36e-3, 21.5e-3}};
    return sizeof(T) == 2 ? bf16 : f32;
}

template <typename T, int WM, int WN, int NWM, int NWN>
int launch_shape(hipStream_t s, Args<T>& a, int blocks, int groups, bool dgrad) {
    using S = Shape<T, WM, WN, NWM, NWN>;
    static const char* const names[2][2] = {{"conv_fprop_kernel<f32>", "conv_dgrad_kernel<f32>"}, {"conv_fprop_kernel<bf16>", "conv_dgrad_kernel<bf16>"}};
    ProfScope ps(names[sizeof(T) == 2][dgrad], s);
    ps.in_parts(split_f32<T, WM, WN>());
    const dim3 grid((unsigned)blocks, (unsigned)groups);
    if constexpr (sizeof(T) == 2) {
        if (a.run > 0) {
            conv_any_kernel<T, WM, WN, NWM, NWN, false, true><<<grid, dim3(split::THREADS), S::Core::LDS_BYTES, s>>>(a);
            LUX_CHECK_LAUNCH();
            return LUXHIP_OK;
        }
    }
    if (a.merged) conv_any_kernel<T, WM, WN, NWM, NWN, true><<<grid, dim3(split::THREADS), S::Core::LDS_BYTES, s>>>(a);
    else conv_any_kernel<T, WM, WN, NWM, NWN, false><<<grid, dim3(split::THREADS), S::Core::LDS_BYTES, s>>>(a);
    LUX_CHECK_LAUNCH();
    return LUXHIP_OK;
}

template <typename T>
Choice choose_any(Sub* sub, int subs, int Ncols, int groups, bool may_slice) {
    constexpr int BK = GemmTraits<T>::BK;
    constexpr size_t most_bytes = size_t(32) << 20;
    const int64_t cus = num_cus() > 0 ? num_cus() : 256;
    const Tile* tl = tiles<T>();
    Choice best{3, 1, 0};                                            // 256 rows: no output has more tiles than a launch
    double t_best = 1e30;
    int kmax = 0;
    for (int i = 0; i < subs; ++i) kmax = std::max(kmax, sub[i].Kpad);
    for (int c = 0; c < 5; ++c) {
        int64_t nt = 0;
        double work = 0.0;                                           // tiles x k
        for (int i = 0; i < subs; ++i) {
            const int64_t t = ceil_div(sub[i].M, tl[c].m) * ceil_div(Ncols, tl[c].n);
            nt += t * groups;
            work += (double)t * groups * (sub[i].Kpad + 100);
        }
        for (int sl = 1; sl <= 8; ++sl) {
            if (nt * sl * split::THREADS >= kMostThreads) break;
            if (sl > 1 && (!may_slice || kmax / sl < 2 * BK || nt > 16384 || (size_t)(nt * sl) * tl[c].m * tl[c].n * sizeof(float) > most_bytes)) break;
            const double k = (double)kmax / sl + 100;
            const double per_cu = nt * sl <= 4 * cus ? (double)ceil_div(nt * sl, cus) * k : work / cus;
            double t = std::max(tl[c].alone * k, tl[c].shared * per_cu);
            if (sl > 1) t += 1.5 + 0.5 * (tl[c].m * tl[c].n / 4096.0) * sl + (double)nt * sl * tl[c].m * tl[c].n * 8.0 / 5e6;
            if (t < t_best) { t_best = t; best.tile = c; best.slices = sl; }
        }
    }
    for (int i = 0; i < subs; ++i) {
        Sub& q = sub[i];
        q.tiles_m = (int)ceil_div(q.M, tl[best.tile].m);
        q.tiles_n = (int)ceil_div(Ncols, tl[best.tile].n);
        q.kslice = (int)(ceil_div(ceil_div(q.Kpad, best.slices), BK) * BK);
        q.slices = q.kslice > 0 ? (int)ceil_div(q.Kpad, q.kslice) : 1;
        q.partial = (int64_t)best.bytes;
        if (q.slices > 1) best.bytes += (size_t)q.tiles_m * q.tiles_n * q.slices * tl[best.tile].m * tl[best.tile].n * sizeof(float);
    }
    return best;
}

// conv_any_bf16.hip
bool launch_few(hipStream_t s, const Args<bf16_t>& a, int* rc);

template <typename T>
int launch_any(hipStream_t s, Args<T>& a, int groups, size_t ws_front, bool dgrad, bool may_slice) {
    if constexpr (sizeof(T) == 2) {
        if (dgrad && groups == 1 && a.merged) {
            Workspace ws;
            int rc = get_workspace(s, ws_front, &ws);
            if (rc != LUXHIP_OK) return rc;
            a.zero = ws.zeros;
            if (launch_few(s, a, &rc)) return rc;
        }
    }
    const Choice c = choose_any<T>(a.sub, a.subs, a.Ncols, groups, may_slice);
    int blocks = 0, nt = 0;
    for (int i = 0; i < a.subs; ++i) {
        Sub& q = a.sub[i];
        q.first_block = blocks;
        q.first_tile = nt;
        const int64_t t = (int64_t)q.tiles_m * q.tiles_n;
        LUX_UNSUPPORTED_IF((blocks + t * q.slices) * groups * split::THREADS >= kMostThreads, "conv: too many tiles");
        blocks += (int)(t * q.slices);
        if (q.slices > 1) nt += (int)t;
    }
    if (blocks == 0) return LUXHIP_OK;
    Workspace ws;
    const int rc = get_workspace(s, ws_front + c.bytes * groups, &ws);
    if (rc != LUXHIP_OK) return rc;
    a.partial = ws.data + ws_front;
    a.partial_group = (int64_t)c.bytes;
    a.sliced_tiles = nt;
    a.counters = ws.counters;
    a.zero = ws.zeros;
    switch (c.tile) {
        case 0: return launch_shape<T, 1, 1, 2, 2>(s, a, blocks, groups, dgrad);
        case 1: return launch_shape<T, 2, 1, 2, 2>(s, a, blocks, groups, dgrad);
        case 2: return launch_shape<T, 2, 2, 2, 2>(s, a, blocks, groups, dgrad);
        case 3: return launch_shape<T, 2, 1, 4, 1>(s, a, blocks, groups, dgrad);
        default: return launch_shape<T, 1, 1, 4, 1>(s, a, blocks, groups, dgrad);
    }
}

template <typename T, int WM, int WN, int NWM, int NWN>
int launch_wgrad_shape(hipStream_t s, WgradArgs<T>& a, int slices) {
    using S = WgradShape<T, WM, WN, NWM, NWN>;
    a.tiles_m = (int)ceil_div(a.Mrows, S::TILE_M);
    a.tiles_n = (int)ceil_div(a.Ncols, S::TILE_N);
    ProfScope ps(sizeof(T) == 2 ? "conv_wgrad_kernel<bf16>" : "conv_wgrad_kernel<f32>", s);
    ps.in_parts(split_f32<T, WM, WN>());
    conv_any_wgrad_kernel<T, WM, WN, NWM, NWN><<<dim3((unsigned)(a.tiles_m * a.tiles_n * slices)), dim3(split::THREADS), S::Core::LDS_BYTES, s>>>(a);
    LUX_CHECK_LAUNCH();
    return LUXHIP_OK;
}
template <typename T>
int launch_any_wgrad(hipStream_t s, WgradArgs<T>& a, int slices, bool narrow) {
    return narrow ? launch_wgrad_shape<T, 1, 1, 2, 2>(s, a, slices) : launch_wgrad_shape<T, 2, 2, 2, 2>(s, a, slices);
}

}  // namespace cany
}  // namespace luxhip
