// Input gradients with few channels (bf16): all residues of a strided convolution as at most 32 columns of one problem
// (conv_any.h, merged), 2 .. 4 taps along each dimension of every residue.
//
// The dense gather of conv_any.h reads every cotangent position once per tap from the caches and writes it to LDS as often:
// 822 MB for 401408 rows of 16 taps x 64 channels.  Here the cotangents that a tile of 32 x 16 rows sees go to LDS once
// ((32 + TW - 1) x (16 + TH - 1) positions of 128 bytes) and the taps read them from there; the filter (at most 32 columns x
// 1024 k) stays in LDS for all tiles of a workgroup.  What bounds it then are the LDS reads (three fragments per two matrix
// instructions).  224 x 224 x 3 x 32 <- 64 channels, 7 x 7, stride 2: 80 -> 52 us.
// LDS: chunk c (16 bytes) of window position j is at slot c ^ (j / 2) % 8 of its 128 bytes, chunk c of a filter column at
// c ^ column % 16: sixteen consecutive positions (columns) lie in sixteen different chunks of the bank period.
#pragma once

#include "conv_any.h"

namespace luxhip {
namespace cany {

constexpr int FEW_THREADS = 512, FEW_A = 32, FEW_B = 16, FEW_TAPS = 4;
constexpr int FEW_WINDOW = (FEW_A + FEW_TAPS - 1) * (FEW_B + FEW_TAPS - 1) * 128;      // 85120 bytes
constexpr size_t FEW_LDS = FEW_WINDOW + 32 * 1024 * 2;                                 // and the filter: 150656

__host__ __device__ inline int few_pitch(int K) { return (K + 127) / 128 * 256; }      // bytes of a filter column in LDS

// CPP: 16-byte chunks per position
template <int CPP>
__global__ __launch_bounds__(FEW_THREADS, 2) void conv_few_kernel(Args<bf16_t> g, int tiles_a, int tiles_b, int tiles, FastDiv divWW) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    char* const win = reinterpret_cast<char*>(lds_raw);
    char* const fil = win + FEW_WINDOW;
    const Sub& q = g.sub[0];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, h = lane >> 5;
    const int RB = q.RAB / q.RA, WW = FEW_A + q.TW - 1, WH = FEW_B + q.TH - 1;
    const int chunks = WW * WH * CPP, pitch = few_pitch(q.K);
    const bf16_t* const wm = g.wm + q.wm;
    for (int i = threadIdx.x; i < 32 * (pitch / 16); i += FEW_THREADS) {
        const int col = i / (pitch / 16), c = i - col * (pitch / 16);
        raw16_t v = {0u, 0u, 0u, 0u};
        if (col < g.Ncols && c * 8 < q.K) v = *reinterpret_cast<const raw16_t*>(wm + (int64_t)col * q.Kpad + c * 8);
        *reinterpret_cast<raw16_t*>(fil + col * pitch + ((c ^ (col & 15)) << 4)) = v;
    }
    constexpr int PER = (FEW_WINDOW / 16 + FEW_THREADS - 1) / FEW_THREADS;
    raw16_t reg[PER];
    int a0, b0, n;
    auto locate = [&](int t) {
        n = t / (tiles_a * tiles_b);
        const int r = t - n * (tiles_a * tiles_b);
        b0 = r / tiles_a * FEW_B;
        a0 = r % tiles_a * FEW_A;
    };
    auto fetch = [&]() {                       // source position of window column j: a0 + w0 - (TW - 1) + j (taps go backwards)
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int id = threadIdx.x + i * FEW_THREADS, pos = id / CPP, c = id - pos * CPP;
            const int wj = (int)divWW.div((uint32_t)pos), j = pos - wj * WW;
            const int sp = a0 + q.w0 - (q.TW - 1) + j, sq = b0 + q.h0 - (q.TH - 1) + wj;
            const bool in = id < chunks && (unsigned)sp < (unsigned)g.SP && (unsigned)sq < (unsigned)g.SQ;
            const bf16_t* p = g.src + ((int64_t)(n * g.SQ + sq) * g.SP + sp) * g.Ctot + c * 8;
            reg[i] = *reinterpret_cast<const raw16_t*>(in ? static_cast<const void*>(p) : g.zero);
        }
    };
    // this lane's columns (8 (r / 4) + 4 h + r % 4): offset from the output of residue (0, 0), channel 0 (-1: no such column),
    // and the residue, rh in the upper half
    int at[16], rwh[16];
    static_for<16>([&](auto R) {
        constexpr int r = decltype(R)::value;
        const int col = 8 * (r >> 2) + 4 * h + (r & 3), res = (int)g.divCch.div((uint32_t)col), ch = col - res * g.Cch, rh = res / g.res_w;
        const int rw = res - rh * g.res_w;
        at[r] = col < g.Ncols ? ch * g.PQ + rh * g.P + rw : -1;
        rwh[r] = rh << 16 | rw;
    });
    int t = blockIdx.x;
    locate(t);
    fetch();
    for (;;) {
        __syncthreads();                       // the window is free (and, the first time, nothing)
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int id = threadIdx.x + i * FEW_THREADS, pos = id / CPP, c = id - pos * CPP;
            if (id < chunks) *reinterpret_cast<raw16_t*>(win + pos * 128 + ((c ^ ((pos >> 1) & 7)) << 4)) = reg[i];
        }
        __syncthreads();
        const int ca = a0, cb = b0, cn = n, next = t + (int)gridDim.x;
        if (next < tiles) {
            locate(next);
            fetch();
        }
        f32x16_v acc[2];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][r] = 0.0f;
        int k = 0;                             // 16-byte chunk of the filter column
        for (int th = 0; th < q.TH; ++th)
            for (int tw = 0; tw < q.TW; ++tw) {
                int pos[2];
#pragma unroll
                for (int i = 0; i < 2; ++i) pos[i] = (2 * w + i + q.TH - 1 - th) * WW + (lane & 31) + q.TW - 1 - tw;
                // the fragments of a tap are on their way before the first product waits for one
                bf16x8_v fb[CPP / 2], fa[2][CPP / 2];
#pragma unroll
                for (int c = 0; c < CPP / 2; ++c) {
                    fb[c] = __builtin_bit_cast(bf16x8_v, *reinterpret_cast<const raw16_t*>(fil + (lane & 31) * pitch + (((k + 2 * c + h) ^ (lane & 15)) << 4)));
#pragma unroll
                    for (int i = 0; i < 2; ++i)
                        fa[i][c] = __builtin_bit_cast(bf16x8_v, *reinterpret_cast<const raw16_t*>(win + pos[i] * 128 + (((2 * c + h) ^ ((pos[i] >> 1) & 7)) << 4)));
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int c = 0; c < CPP / 2; ++c)
#pragma unroll
                    for (int i = 0; i < 2; ++i) acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[c], fa[i][c], acc[i], 0, 0, 0);
                k += CPP;
            }
        // lane: row a = ca + lane % 32 of b = cb + 2 w + i; register r: column 8 (r / 4) + 4 h + r % 4
        const int a = ca + (lane & 31), iw = a * g.os_w + q.ow0;
        uint32_t nans = 0;                     // bit 16 i + r
        bf16_t* out[2];
        int yy[2];
        bool in[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int b = cb + 2 * w + i;
            in[i] = a < q.RA && b < RB;
            yy[i] = b * g.os_h + q.oh0;
            out[i] = g.out + ((int64_t)cn * g.Ctot_out + g.col_off) * g.PQ + ((int64_t)yy[i] * g.P + iw);
        }
        auto fits = [&](int i, int r) {
            return in[i] && at[r] >= 0 && (unsigned)(iw + (rwh[r] & 0xffff)) < (unsigned)g.P && (unsigned)(yy[i] + (rwh[r] >> 16)) < (unsigned)g.Q;
        };
        static_for<32>([&](auto E) {
            constexpr int i = decltype(E)::value / 16, r = decltype(E)::value % 16;
            if (fits(i, r)) {
                st(out[i] + at[r], acc[i][r]);
                if (acc[i][r] != acc[i][r]) nans |= 1u << decltype(E)::value;
            }
        });
        // a NaN may be an infinite cotangent times a tap that this residue does not have
        while (nans != 0) {
            const int e = __builtin_ctz(nans), r = e & 15, b = cb + 2 * w + (e >> 4), col = 8 * (r >> 2) + 4 * h + (r & 3);
            nans &= nans - 1;
            const int res = (int)g.divCch.div((uint32_t)col), ch = col - res * g.Cch, rh = res / g.res_w, rw = res - rh * g.res_w;
            st(g.out + ((int64_t)cn * g.Ctot_out + g.col_off + ch) * g.PQ + (int64_t)(b * g.os_h + q.oh0 + rh) * g.P + iw + rw,
               own_taps_sum<bf16_t>(g, q, g.src, g.wm, a, b, cn, col, rw, rh));
        }
        if (next >= tiles) break;
        t = next;
    }
}

}  // namespace cany
}  // namespace luxhip
