// Implicit-GEMM convolutions of any channel count, stride and size (the kernels of conv_kernels.h, conv_patch.h and
// conv_wgrad_patch.h want channels in multiples of 32 or 64 and, for the input gradient, a unit stride).
//
// Activations are channel-contiguous with the channels of a group padded with zeros to whole 16-byte chunks (8 bf16 or 4
// fp32), so every chunk of the im2col matrix is one aligned load: a run of channels at one position and filter tap.  The
// tap of a chunk is found once per thread and stage and shared by its rows; rows are decoded once per tile.
//
// The input gradient of a strided convolution is a set of unit-stride problems.  With i + pad = stride q + r, the input
// positions of residue r see the taps ka with ka dil = r (mod stride), at output positions q - (ka dil - r) / stride: a
// dense gather with an affine tap list, no test of divisibility, no multiplication by structural zeros.  Each residue is a
// sub-problem of one launch.  Where a residue has few channels (the first layer of an image network: 3) all residues
// become columns of one problem instead, over the union of their taps: 2 x 2 residues of 3 channels share the rows they
// read, and fill 12 columns of a 32-column tile instead of 3.
// A tap that a residue lacks is a zero weight there, and zero times a non-finite cotangent is NaN where the residue does not
// see that cotangent at all.  So a sum that comes out NaN is taken again over the residue's own taps (own_taps_sum below);
// the others pay one comparison.  (Residues apart would need no such thing, at three times the gathers: 49 taps against 16.)
//
// The main loop is the one of gemm_split.h: several stages per trip to memory, K cut into slices where tiles are few.
//
// Measured against the kernels that gathered element by element with four divisions each and skipped what a stride does not
// divide (bf16, 7 x 7, stride 2, 3 -> 64 channels on 224 x 224 x 32): forward 349 -> 67 us, input gradient 4572 -> 82, filter
// gradient 144 -> 75, layout transform of x 33 -> 11; the whole step 5154 -> 286.  What bounds the three products now is the
// gather: 128 bytes of LDS stores and loads per 16-byte chunk of a 64-column tile, at 10 to 15 % of the matrix rate.
#pragma once

#include "common.h"
#include "conv_kernels.h"
#include "gemm_split.h"

namespace luxhip {
namespace cany {

// One dense gather problem: rows (a, b, n), a < RA, b < RB; taps (tw, th); source position a ss + w0 + tw wstep.
struct Sub {
    int RA, RAB, M;            // row grid (RAB = RA RB), rows in all
    int w0, wstep, h0, hstep, TW, TH;
    int K, Kpad;               // TW TH Cp, and padded to whole stages (row length of the packed filter)
    int ow0, oh0;              // output position of row a: a os + ow0 (merged residues: + the residue)
    int tiles_m, tiles_n, slices, kslice;
    int first_block, first_tile;
    int64_t wm;                // element offset of the packed filter
    int64_t partial;           // byte offset of the partial sums
    FastDiv divRA, divRAB, divTW;
};
constexpr int MAX_SUBS = 4;       // a stride of 2; larger strides take more launches

template <typename T>
struct Args {
    const T* src;              // channel-contiguous, first channel of the first group of the launch (one blockIdx.y each)
    const T* wm;               // its packed filter
    int64_t wm_group;          // packed filter elements per group
    const void* zero;
    const T* bias;
    T *out, *pre;
    int Ctot, Cp, SP, SQ, ss_w, ss_h;
    int P, Q, PQ;              // output planes
    int os_w, os_h;
    int Ncols, Cch;            // columns; channels per residue (merged: Ncols = residues * Cch)
    int res_w;                 // merged: residues along w
    int col_off, Ctot_out, act;
    int subs, merged;          // merged: the residues are columns
    int sliced_tiles;          // counters per group
    char* partial;
    int64_t partial_group;     // bytes of partial sums per group
    uint32_t* counters;
    FastDiv divCp, divCch;
    Sub sub[MAX_SUBS];
    int kW, kH;                // merged (dilation 1): tap t of residue r is filter tap t * os + r, where there is one
    int run;                   // RUNS: elements of a stage that belong to the row's window, the rest count as zero
};

// A chunk of a row.  Runs of positions (see Runs in conv.hip) start at any position, and one of four bf16 channels is eight bytes; the
// load is the same instruction as an aligned one.
typedef uint32_t chunk8_t __attribute__((ext_vector_type(4), aligned(8)));

// A: K-major rows of the im2col matrix.  RUNS: a stage is the window's positions of one source row (see Runs in conv.hip); what
// lies behind them in memory is data of other windows, and is cut off here (a zero in the filter would turn an infinity into NaN).
template <typename T, int ROWS, bool RUNS>
struct RowLoader {
    using Tr = GemmTraits<T>;
    static constexpr bool KMAJOR = true;
    static constexpr int CPR = Tr::BK / Tr::VEC, PER = ROWS * CPR / split::THREADS, STEP = split::THREADS / CPR;
    static_assert(PER >= 1, "at least one chunk per thread");
    const Args<T>& g;
    const Sub& q;
    const T* src;
    int pos[PER], ps[PER], qs[PER];
    int chunk;
    __device__ __forceinline__ RowLoader(const Args<T>& gg, const Sub& s, const T* x, int m0) : g(gg), q(s), src(x) {
        chunk = (threadIdx.x % CPR) * Tr::VEC;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int m = m0 + (int)threadIdx.x / CPR + i * STEP;
            ps[i] = -(1 << 28);                                        // never valid
            qs[i] = 0;
            pos[i] = 0;
            if (m < s.M) {
                const int n = (int)s.divRAB.div((uint32_t)m), rem = m - n * s.RAB;
                const int b = (int)s.divRA.div((uint32_t)rem), a = rem - b * s.RA;
                ps[i] = a * g.ss_w + s.w0;
                qs[i] = b * g.ss_h + s.h0;
                pos[i] = n * g.SQ;                                     // + the source row, below
            }
        }
    }
    __device__ __forceinline__ void load(int k, u32x4_v (&reg)[PER]) const {
        const int kc = k + chunk;
        const int t = (int)g.divCp.div((uint32_t)kc), c = kc - t * g.Cp;
        const int th = (int)q.divTW.div((uint32_t)t), tw = t - th * q.TW;
        const int dp = tw * q.wstep, dq = th * q.hstep;
        const bool tap = kc < q.K;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int sp = ps[i] + dp, sq = qs[i] + dq;
            const bool valid = tap && (unsigned)sp < (unsigned)g.SP && (unsigned)sq < (unsigned)g.SQ;
            const T* p = src + ((int64_t)((pos[i] + sq) * g.SP + sp) * g.Ctot + c);
            reg[i] = *reinterpret_cast<const chunk8_t*>(valid ? static_cast<const void*>(p) : g.zero);
        }
    }
    template <bool SPLIT>
    __device__ __forceinline__ void store(u32x4_v (&reg)[PER], T* lds, int) const {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            u32x4_v v = reg[i];
            if constexpr (RUNS) {
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = chunk + e * (Tr::VEC / 4) < g.run ? v[e] : 0u;
            }
            put_chunk<T, true, ROWS, SPLIT>(lds, (int)threadIdx.x / CPR + i * STEP, chunk, v);
        }
    }
};

template <typename T, int WM, int WN, int NWM, int NWN, bool RUNS = false>
struct Shape {
    static constexpr int TILE_M = NWM * WM * 32, TILE_N = NWN * WN * 32;
    using LA = RowLoader<T, TILE_M, RUNS>;
    using LB = split::Loader<T, true, TILE_N>;
    using Core = split::Core<T, WM, WN, NWM, NWN, LA, LB>;
};

// Merged residues: the sum of row (a, b, n) and column col over the taps that the column's residue (rw, rh) has.  A NaN among
// the terms ends it, so a cotangent that is NaN throughout costs one term per element.
template <typename T>
__device__ __forceinline__ float own_taps_sum(const Args<T>& g, const Sub& q, const T* src, const T* wm, int a, int b, int n, int col, int rw, int rh) {
    const int nw = (g.kW - rw + g.os_w - 1) / g.os_w, nh = (g.kH - rh + g.os_h - 1) / g.os_h;
    const T* wcol = wm + q.wm + (int64_t)col * q.Kpad;
    float sum = 0.0f;
    for (int th = 0; th < nh; ++th) {
        const int sq = b * g.ss_h + q.h0 + th * q.hstep;
        if ((unsigned)sq >= (unsigned)g.SQ) continue;
        for (int tw = 0; tw < nw; ++tw) {
            const int sp = a * g.ss_w + q.w0 + tw * q.wstep;
            if ((unsigned)sp >= (unsigned)g.SP) continue;
            const T* x = src + (int64_t)((n * g.SQ + sq) * g.SP + sp) * g.Ctot;
            const T* w = wcol + (th * q.TW + tw) * g.Cp;
#pragma unroll 1
            for (int c = 0; c < g.Cp; ++c) sum = fmaf(ld(x + c), ld(w + c), sum);
            if (sum != sum) return sum;
        }
    }
    return sum;
}

// MERGED: the residues of an input gradient are columns and a NaN among the sums is looked into.  A kernel of its own: the test
// costs 2 to 4 %, and a register that takes a wave from every SIMD unless it is told to stay below (256 x 32 tiles of the first
// layer, 78 us with four waves, 85 with three).
template <typename T, int WM, int WN, int NWM, int NWN, bool MERGED, bool RUNS = false>
__global__ __launch_bounds__(split::THREADS, MERGED && WM * WN < 4 ? 4 : (split_waves<T, WM, WN>())) void conv_any_kernel(Args<T> g) {
    using S = Shape<T, WM, WN, NWM, NWN, RUNS>;
    using Core = typename S::Core;
    using ML = typename Core::ML;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    Sub q = g.sub[0];                  // selected by comparison: an index into the arguments would copy them to scratch memory
#pragma unroll
    for (int i = 1; i < MAX_SUBS; ++i)
        if (i < g.subs && (int)blockIdx.x >= g.sub[i].first_block) q = g.sub[i];
    const int id = (int)blockIdx.x - q.first_block, grp = blockIdx.y;
    const T *const src = g.src + (int64_t)grp * g.Cp, *const wm = g.wm + grp * g.wm_group;
    const int col_off = g.col_off + grp * g.Cch;
    const int tile = id / q.slices, slice = id - tile * q.slices;
    int tm, tn;
    tile_coords(tile, q.tiles_m, q.tiles_n, tm, tn);
    const int m0 = tm * S::TILE_M, n0 = tn * S::TILE_N;
    static_assert(WM <= 2 && WN <= 2, "32 accumulator bits per i below");
    f32x16_v acc[WM][WN];
    {
        const typename S::LA la(g, q, src, m0);
        Operand<T> B;
        B.p = wm + q.wm; B.sr = q.Kpad; B.sk = 1; B.vec_ok = 1;
        B.rows = g.Ncols - n0;                                         // the last tile clamps its rows
        B.p += (int64_t)n0 * q.Kpad;
        const typename S::LB lb(B, 0);
        const int kbeg = slice * q.kslice;
        Core::run(la, lb, kbeg, min(kbeg + q.kslice, q.Kpad), reinterpret_cast<T*>(lds_raw), acc);
    }
    if (q.slices > 1) {
        split::Plan p{q.slices, q.kslice, reinterpret_cast<float*>(g.partial + grp * g.partial_group + q.partial),
                      g.counters + grp * g.sliced_tiles + q.first_tile};
        if (!Core::combine(p, tile, slice, acc)) return;
    }
    bool nan = false;                  // among this lane's sums (here, where no lane is masked off: two instructions per sum)
    if constexpr (MERGED) {
        static_for<WM * WN * 16>([&](auto E) {
            constexpr int e = decltype(E)::value;
            const float v = acc[e / (WN * 16)][e / 16 % WN][e % 16];
            nan |= v != v;
        });
    }
    // rows -> output positions
    const int mb = ML::lane_m(m0), nb = ML::lane_n(n0);
    int64_t row[WM];
    int iw[WM], ih[WM];
    bool ok[WM];
#pragma unroll
    for (int i = 0; i < WM; ++i) {
        const int m = mb + 32 * i;
        ok[i] = m < q.M;
        const int n = (int)q.divRAB.div((uint32_t)(ok[i] ? m : 0)), rem = (ok[i] ? m : 0) - n * q.RAB;
        const int b = (int)q.divRA.div((uint32_t)rem), a = rem - b * q.RA;
        iw[i] = a * g.os_w + q.ow0;
        ih[i] = b * g.os_h + q.oh0;
        row[i] = (int64_t)n * g.Ctot_out * g.PQ + (int64_t)ih[i] * g.P + iw[i];
    }
    if (!MERGED && g.bias) {           // all loads before the first column's condition: behind it each is a trip to memory of its own
        static_for<WN * 16>([&](auto JR) {
            constexpr int j = decltype(JR)::value / 16, r = decltype(JR)::value % 16;
            const float bv = ld(g.bias + col_off + min(nb + j * 32 + ((r >> 2) << 3) + (r & 3), g.Ncols - 1));
#pragma unroll
            for (int i = 0; i < WM; ++i) acc[i][j][r] += bv;
        });
    }
    // One activation's code for all columns in one piece: with the choice inside, every column jumped over the other activations' code to a line
    // that no prefetch had brought, sixteen waits for instructions per workgroup (bf16 1 x 1, 14 x 14 x 48 -> 214 x 2: forward 9.3 -> 5.7 us; 3 x 3,
    // 70 x 70 x 51 -> 32 x 11: forward 19.0 -> 13.4, input gradient 17.6 -> 9.9; the first layer's step, 7 x 7 on 224 x 224 x 32: 184 -> 166).
    auto emit = [&](auto ACT) {
        static_for<WN * 16>([&](auto JR) {
            constexpr int j = decltype(JR)::value / 16, r = decltype(JR)::value % 16;
            const int col = nb + j * 32 + ((r >> 2) << 3) + (r & 3);
            if (col < g.Ncols) {
                int ch = col, rw = 0, rh = 0;
                if constexpr (MERGED) {
                    const int res = (int)g.divCch.div((uint32_t)col);
                    ch = col - res * g.Cch;
                    rh = res / g.res_w;
                    rw = res - rh * g.res_w;
                }
                const int64_t coff = (int64_t)(col_off + ch) * g.PQ + (int64_t)rh * g.P + rw;
                float v[WM];
                bool st_ok[WM];
#pragma unroll
                for (int i = 0; i < WM; ++i) {
                    v[i] = acc[i][j][r];
                    st_ok[i] = ok[i];
                    if constexpr (MERGED) st_ok[i] = ok[i] && (unsigned)(iw[i] + rw) < (unsigned)g.P && (unsigned)(ih[i] + rh) < (unsigned)g.Q;
                }
                if (!MERGED && g.pre != nullptr) {
#pragma unroll
                    for (int i = 0; i < WM; ++i)
                        if (st_ok[i]) st(g.pre + coff + row[i], v[i]);
                }
                act_vec_as<decltype(ACT)::value>(v);
#pragma unroll
                for (int i = 0; i < WM; ++i)
                    if (st_ok[i]) st(g.out + coff + row[i], v[i]);
            }
        });
    };
    if constexpr (MERGED) {                // an input gradient: no bias, no activation
        emit(std::integral_constant<int, LUXHIP_ACT_IDENTITY>{});
    } else {
#define CONV_ANY_EMIT(A) emit(std::integral_constant<int, A>{})
        LUX_DISPATCH_ACT(g.act, CONV_ANY_EMIT);
#undef CONV_ANY_EMIT
    }
    if constexpr (MERGED) {
        if (!nan) return;
        uint64_t nans = 0;                 // bit 32 i + 16 j + r
        static_for<WM * WN * 16>([&](auto E) {
            constexpr int i = decltype(E)::value / (WN * 16), jr = decltype(E)::value % (WN * 16);
            const float v = acc[i][jr / 16][jr % 16];
            if (v != v) nans |= uint64_t(1) << (32 * i + jr);
        });
        while (nans != 0) {
            const int e = __builtin_ctzll(nans), r = e & 15;
            nans &= nans - 1;
            const int m = mb + (e & 32), col = nb + 2 * (e & 16) + ((r >> 2) << 3) + (r & 3);
            if (m >= q.M || col >= g.Ncols) continue;
            const int n = (int)q.divRAB.div((uint32_t)m), rem = m - n * q.RAB;
            const int b = (int)q.divRA.div((uint32_t)rem), a = rem - b * q.RA;
            const int res = (int)g.divCch.div((uint32_t)col), ch = col - res * g.Cch, rh = res / g.res_w, rw = res - rh * g.res_w;
            const int ow = a * g.os_w + q.ow0 + rw, oh = b * g.os_h + q.oh0 + rh;
            if ((unsigned)ow < (unsigned)g.P && (unsigned)oh < (unsigned)g.Q)
                st(g.out + ((int64_t)n * g.Ctot_out + col_off + ch) * g.PQ + (int64_t)oh * g.P + ow, own_taps_sum<T>(g, q, src, wm, a, b, n, col, rw, rh));
        }
    }
}

// ----------------------------------------------------------------------------- filter gradient
// dw[(tap, ci), co] = sum over (ow, oh, n) of xT[position][ci] dzT[(ow, oh, n)][co]: both operands contiguous along their
// rows (channels), the contraction runs over output positions and is cut into slices of fp32 partial sums.
template <typename T>
struct WgradArgs {
    const T *src, *dyT;        // channel-contiguous, padded channels; first channel of the group
    const void* zero;
    int Ctot, Cp, Mrows;       // source channels in all, per group and tap; rows = taps * Cp
    int OW, OWOH, SP, SQ, kW, sw, sh, pw, ph, dw, dh;
    int Ytot, Ncols;           // channels of dyT in all; columns of the group (padded)
    int Ktotal, kslice, tiles_m, tiles_n;
    int positions;             // OW OH N; Ktotal is larger only where that is less than a stage
    float* partial;            // [slice][column][row]
    FastDiv divOW, divOWOH, divCp, divkW;
};

template <typename T, int ROWS>
struct WgradRowLoader {
    using Tr = GemmTraits<T>;
    static constexpr bool KMAJOR = false;
    static constexpr int CPR = ROWS / Tr::VEC, PER = ROWS * Tr::BK / Tr::VEC / split::THREADS, STEP = split::THREADS / CPR;
    static_assert(PER >= 1, "at least one chunk per thread");
    const WgradArgs<T>& g;
    int r, dp, dq, c;
    bool in;
    __device__ __forceinline__ WgradRowLoader(const WgradArgs<T>& gg, int m0) : g(gg) {
        r = ((int)threadIdx.x % CPR) * Tr::VEC;
        in = m0 + r < g.Mrows;
        const int m = in ? m0 + r : 0;
        const int t = (int)g.divCp.div((uint32_t)m);
        c = m - t * g.Cp;
        const int kb = (int)g.divkW.div((uint32_t)t), ka = t - kb * g.kW;
        dp = ka * g.dw - g.pw;
        dq = kb * g.dh - g.ph;
    }
    __device__ __forceinline__ void load(int k, u32x4_v (&reg)[PER]) const {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int kp = k + (int)threadIdx.x / CPR + i * STEP;
            const int n = (int)g.divOWOH.div((uint32_t)kp), rem = kp - n * g.OWOH;
            const int oh = (int)g.divOW.div((uint32_t)rem), ow = rem - oh * g.OW;
            const int sp = ow * g.sw + dp, sq = oh * g.sh + dq;
            const bool valid = in && kp < g.positions && (unsigned)sp < (unsigned)g.SP && (unsigned)sq < (unsigned)g.SQ;
            const T* p = g.src + ((int64_t)((n * g.SQ + sq) * g.SP + sp) * g.Ctot + c);
            reg[i] = *reinterpret_cast<const chunk8_t*>(valid ? static_cast<const void*>(p) : g.zero);
        }
    }
    template <bool SPLIT>
    __device__ __forceinline__ void store(u32x4_v (&reg)[PER], T* lds, int skip) const {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int k = (int)threadIdx.x / CPR + i * STEP;
            const u32x4_v v = k < skip ? u32x4_v{0u, 0u, 0u, 0u} : reg[i];
            put_chunk<T, false, ROWS, SPLIT>(lds, r, k, v);
        }
    }
};

template <typename T, int WM, int WN, int NWM, int NWN>
struct WgradShape {
    static constexpr int TILE_M = NWM * WM * 32, TILE_N = NWN * WN * 32;
    using LA = WgradRowLoader<T, TILE_M>;
    using LB = split::Loader<T, false, TILE_N>;
    using Core = split::Core<T, WM, WN, NWM, NWN, LA, LB>;
};

template <typename T, int WM, int WN, int NWM, int NWN>
__global__ __launch_bounds__(split::THREADS, (split_waves<T, WM, WN>())) void conv_any_wgrad_kernel(WgradArgs<T> g) {
    using S = WgradShape<T, WM, WN, NWM, NWN>;
    using Core = typename S::Core;
    using ML = typename Core::ML;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    const int tiles = g.tiles_m * g.tiles_n;
    const int slice = blockIdx.x / tiles, tile = blockIdx.x - slice * tiles;
    const int m0 = (tile % g.tiles_m) * S::TILE_M, n0 = (tile / g.tiles_m) * S::TILE_N;
    f32x16_v acc[WM][WN];
    const typename S::LA la(g, m0);
    Operand<T> B;
    B.p = g.dyT + n0; B.sr = 1; B.sk = g.Ytot; B.rows = g.Ncols - n0; B.vec_ok = 1;
    const typename S::LB lb(B, 0);
    const int kbeg = slice * g.kslice;
    Core::run(la, lb, kbeg, min(kbeg + g.kslice, g.Ktotal), reinterpret_cast<T*>(lds_raw), acc);
    float* out = g.partial + (size_t)slice * g.Mrows * g.Ncols;
    ML::for_each(acc, m0, n0, [&](int m, int col, float v) {
        if (m < g.Mrows && col < g.Ncols) out[(size_t)m + (size_t)col * g.Mrows] = v;
    });
}

// Tile and slices of a launch over `groups` groups, and the bytes that its slices take per group (32 MiB in all at most)
struct Choice { int tile, slices; size_t bytes; };
template <typename T>
Choice choose_any(Sub* sub, int subs, int Ncols, int groups, bool may_slice);    // conv_any_*.hip; fills in the tiling of sub[]
template <typename T>
int launch_any(hipStream_t s, Args<T>& a, int groups, size_t ws_front, bool dgrad, bool may_slice);
template <typename T>
int launch_any_wgrad(hipStream_t s, WgradArgs<T>& a, int slices, bool narrow);

}  // namespace cany
}  // namespace luxhip
