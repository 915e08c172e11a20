// Convolution entry points: layout transforms, filter repacking, launch logic of the
// implicit-GEMM kernels (conv_kernels.h) and the split-K reduction of the filter gradient.
#include <algorithm>
#include <cmath>
#include <utility>
#include <vector>

#include "common.h"
#include "act_vec.h"
#include "conv_kernels.h"
#include "conv_patch.h"
#include "conv_wgrad_patch.h"
#include "conv_any.h"

namespace luxhip {

int bias_act_bwd_dispatch(hipStream_t s, int dtype, int act, int64_t I, int64_t C, int64_t N, const void* delta,
                          const void* out, const void* pre, void* dx, void* dbias);   // elementwise.hip

// ----------------------------------------------------------------------------- layout transforms
// in (P, C, N) with p contiguous  ->  out (C, P, N) with c contiguous
template <typename T>
__global__ __launch_bounds__(256) void whcn_to_cwhn_kernel(const T* __restrict__ in, T* __restrict__ out, int P, int C) {
    __shared__ T tile[32][33];
    const int n = blockIdx.z;
    const int p0 = blockIdx.x * 32, c0 = blockIdx.y * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;       // 32 x 8
    const T* src = in + (size_t)n * C * P;
    T* dst = out + (size_t)n * C * P;
#pragma unroll
    for (int j = 0; j < 32; j += 8) {
        const int c = c0 + ty + j, p = p0 + tx;
        if (c < C && p < P) tile[ty + j][tx] = src[(size_t)c * P + p];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 32; j += 8) {
        const int p = p0 + ty + j, c = c0 + tx;
        if (c < C && p < P) dst[(size_t)p * C + c] = tile[tx][ty + j];
    }
}

// Same transform with 16-byte global accesses on both sides (P and C multiples of the vector
// length, aligned pointers): a 64(p) x 64(c) tile goes through LDS as tile[c][p]; the row pitch
// (66 two-byte or 65 four-byte elements) spreads the strided reads of the second phase over
// the banks.
template <typename T>
__device__ __forceinline__ void whcn_to_cwhn_vec_tile(const T* __restrict__ in, T* __restrict__ out, int P, int C) {
    constexpr int V = 16 / sizeof(T), TP = 64, TC = 64;
    constexpr int PITCH = TP + 4 / sizeof(T);   // 66 (bf16) / 65 (fp32) elements: rows stay 4-byte aligned
    __shared__ __align__(16) T tile[TC * PITCH];
    const int n = blockIdx.z;
    const int p0 = blockIdx.x * TP, c0 = blockIdx.y * TC;
    const T* src = in + (size_t)n * C * P;
    T* dst = out + (size_t)n * C * P;
    // phase 1: vectors along p
    constexpr int VP = TP / V;                       // vectors per tile row
#pragma unroll
    for (int it = 0; it < TC * VP / 256; ++it) {
        const int idx = threadIdx.x + it * 256;
        const int c = idx / VP, pv = idx % VP;
        if (c0 + c < C && p0 + pv * V < P) {
            const raw16_t v = *reinterpret_cast<const raw16_t*>(src + (size_t)(c0 + c) * P + p0 + pv * V);
            uint32_t* row = reinterpret_cast<uint32_t*>(tile + c * PITCH + pv * V);
#pragma unroll
            for (int k = 0; k < 4; ++k) row[k] = v[k];
        }
    }
    __syncthreads();
    // phase 2: vectors along c
    constexpr int VC = TC / V;
#pragma unroll
    for (int it = 0; it < TP * VC / 256; ++it) {
        const int idx = threadIdx.x + it * 256;
        const int pp = idx / VC, cv = idx % VC;
        if (p0 + pp < P && c0 + cv * V < C) {
            raw16_t r;
            T* e = reinterpret_cast<T*>(&r);
#pragma unroll
            for (int k = 0; k < V; ++k) e[k] = tile[(cv * V + k) * PITCH + pp];
            *reinterpret_cast<raw16_t*>(dst + (size_t)(p0 + pp) * C + c0 + cv * V) = r;
        }
    }
}

template <typename T>
__global__ __launch_bounds__(256) void whcn_to_cwhn_vec_kernel(const T* __restrict__ in, T* __restrict__ out, int P, int C) {
    whcn_to_cwhn_vec_tile<T>(in, out, P, C);
}

// wF[(co*T + t)*Cin_g + ci] (fprop, K = T*Cin_g) or wD[((g*Cin_g + ci)*T + t)*Cout_g + col]
// (dgrad, K = T*Cout_g) from w[a + kW*(b + kH*(ci + Cin_g*co))]; tap t = ka + kW*kb with
// a = flip ? ka : kW-1-ka (same for b).
template <typename T>
__device__ __forceinline__ void pack_filter_element(const T* __restrict__ w, T* __restrict__ out, const ConvGeom& g, int for_dgrad, int idx) {
    const int total = g.kW * g.kH * g.Cin_g * g.Cout;
    if (idx >= total) return;
    const int Tt = g.kW * g.kH;
    int co, t, ci;
    if (!for_dgrad) {
        ci = idx % g.Cin_g;
        t = (idx / g.Cin_g) % Tt;
        co = idx / (g.Cin_g * Tt);
    } else {
        const int col = idx % g.Cout_g;
        t = (idx / g.Cout_g) % Tt;
        const int cig = idx / (g.Cout_g * Tt);       // g*Cin_g + ci
        const int grp = cig / g.Cin_g;
        ci = cig - grp * g.Cin_g;
        co = grp * g.Cout_g + col;
    }
    const int ka = t % g.kW, kb = t / g.kW;
    const int a = g.flip ? ka : g.kW - 1 - ka, b = g.flip ? kb : g.kH - 1 - kb;
    out[idx] = w[a + g.kW * (b + g.kH * (ci + g.Cin_g * co))];
}
template <typename T>
__global__ void pack_filter_kernel(const T* __restrict__ w, T* __restrict__ out, ConvGeom g, int for_dgrad) {
    pack_filter_element<T>(w, out, g, for_dgrad, (int)(blockIdx.x * blockDim.x + threadIdx.x));
}
// The layout transform of a tensor and the repacking of the filter in one launch (the filter is a few hundred
// KiB: a launch of its own costs more than the work): the z slices 0 .. N - 1 of the grid transform image n, the
// slices behind them repack 256 filter elements per workgroup.
template <typename T>
__global__ __launch_bounds__(256) void whcn_to_cwhn_pack_kernel(const T* __restrict__ in, T* __restrict__ out, int P, int C, int N,
                                                                const T* __restrict__ w, T* __restrict__ wout, ConvGeom g, int for_dgrad) {
    if ((int)blockIdx.z < N) {
        whcn_to_cwhn_vec_tile<T>(in, out, P, C);
    } else {
        const int block = ((int)(blockIdx.z - N) * (int)gridDim.y + (int)blockIdx.y) * (int)gridDim.x + (int)blockIdx.x;
        pack_filter_element<T>(w, wout, g, for_dgrad, block * 256 + (int)threadIdx.x);
    }
}

// Channel-contiguous copy with the channels of every group padded with zeros to Cp, for any number of positions and
// channels: out (groups * Cp, P, N) from the first groups * Cg channels of in (P, Cin, N), 16-byte stores.  Tiles of 64 positions x 64 padded channels
// go through LDS; the reads are one element per lane (64 consecutive positions of a channel per wave), since the rows of a
// ragged plane start at any address.  `zeros` positions of zeros follow the last image.  Blocks behind the transform's
// repack the filter.
struct PackSub {
    int rw, rh, s0w, stw, s0h, sth;      // residue and tap shifts (shift s of residue r is tap (s stride + r) / dilation)
    int TW, K, Kpad, merged_w;           // merged_w > 0: the residue comes from the column, merged_w residues along w
    int64_t wm, first;                   // element offset in the packed filter; first element of this part
};
struct PackSubs {
    PackSub sub[cany::MAX_SUBS];
    int n, dgrad, Cp, Ncols, Cch;
    int64_t per_group, wm_group, total;  // elements of a group in this launch and in all launches; in this launch over all groups
};
template <typename T>
__device__ __forceinline__ void pack_sub_element(const T* __restrict__ w, T* __restrict__ out, const ConvGeom& g, const PackSubs& ps, int64_t idx) {
    if (idx >= ps.total) return;
    const bool small = ps.total < (int64_t(1) << 31);      // uniform; 64-bit divisions take longer than the rest
    const int grp = small ? (int)((uint32_t)idx / (uint32_t)ps.per_group) : (int)(idx / ps.per_group);
    idx -= grp * ps.per_group;
    PackSub q = ps.sub[0];
#pragma unroll
    for (int i = 1; i < cany::MAX_SUBS; ++i)
        if (i < ps.n && idx >= ps.sub[i].first) q = ps.sub[i];
    const int64_t e = idx - q.first;
    const int col = small ? (int)((uint32_t)e / (uint32_t)q.Kpad) : (int)(e / q.Kpad), k = (int)(e - (int64_t)col * q.Kpad);
    T v = T(0);
    const int t = k / ps.Cp, c = k - t * ps.Cp;
    const int th = t / q.TW, tw = t - th * q.TW;
    if (k < q.K && c < (ps.dgrad ? g.Cout_g : g.Cin_g)) {
        int ci = c, co = grp * g.Cout_g + col, ka = tw, kb = th;
        bool tap = true;
        if (ps.dgrad) {
            const int res = q.merged_w > 0 ? col / ps.Cch : 0;
            ci = col - res * ps.Cch;
            co = grp * g.Cout_g + c;
            const int rh = q.merged_w > 0 ? res / q.merged_w : q.rh, rw = q.merged_w > 0 ? res % q.merged_w : q.rw;
            const int nw = (q.s0w + tw * q.stw) * g.sw + rw, nh = (q.s0h + th * q.sth) * g.sh + rh;
            ka = nw / g.dw;
            kb = nh / g.dh;
            tap = nw >= 0 && nh >= 0 && ka * g.dw == nw && kb * g.dh == nh && ka < g.kW && kb < g.kH;
        }
        if (tap) {
            const int a = g.flip ? ka : g.kW - 1 - ka, b = g.flip ? kb : g.kH - 1 - kb;
            v = w[a + g.kW * (b + g.kH * (ci + g.Cin_g * co))];
        }
    }
    out[grp * ps.wm_group + q.wm + e] = v;
}
template <typename T>
__global__ __launch_bounds__(256) void pad_to_cwhn_pack_kernel(const T* __restrict__ in, T* __restrict__ out, int P, int Cin, int Cg, int Cp, int groups,
                                                               int N, int zeros, int tiles_p, int tiles_c, int blocks, const T* __restrict__ w,
                                                               T* __restrict__ wout, ConvGeom g, PackSubs ps) {
    constexpr int V = 16 / (int)sizeof(T), PITCH = 64 + 4 / (int)sizeof(T);
    __shared__ __align__(16) T tile[64 * PITCH];
    if ((int)blockIdx.x >= blocks) {
        pack_sub_element<T>(w, wout, g, ps, (int64_t)((int)blockIdx.x - blocks) * 256 + threadIdx.x);
        return;
    }
    const int Ct = groups * Cp;
    if (Ct == V) {                                   // a chunk per position: no transpose
        const int64_t pos = (int64_t)blockIdx.x * 256 + threadIdx.x;
        if (pos >= (int64_t)P * N + zeros) return;
        T e[V];
#pragma unroll
        for (int c = 0; c < V; ++c) e[c] = T(0);
        if (pos < (int64_t)P * N) {
            const int n = (int)(pos / P);
            const T* src = in + (int64_t)n * P * Cin + (pos - (int64_t)n * P);
#pragma unroll
            for (int c = 0; c < V; ++c)
                if (c < Cg) e[c] = src[(int64_t)c * P];     // one group: Cp == V
        }
        *reinterpret_cast<raw16_t*>(out + pos * V) = *reinterpret_cast<const raw16_t*>(e);
        return;
    }
    const int n = blockIdx.x / (tiles_p * tiles_c), rest = blockIdx.x - n * (tiles_p * tiles_c);
    const int c0 = (rest / tiles_p) * 64, p0 = (rest % tiles_p) * 64;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (n < N) {
        const T* src = in + (int64_t)n * P * Cin;
        T v[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int cp = c0 + wave + 4 * j, grp = cp / Cp, c = cp - grp * Cp;
            const bool ok = cp < Ct && c < Cg && p0 + lane < P;
            v[j] = src[ok ? (int64_t)(grp * Cg + c) * P + p0 + lane : 0];
            if (!ok) v[j] = T(0);
        }
#pragma unroll
        for (int j = 0; j < 16; ++j) tile[(wave + 4 * j) * PITCH + lane] = v[j];
    } else {
#pragma unroll
        for (int j = 0; j < 16; ++j) tile[(wave + 4 * j) * PITCH + lane] = T(0);
    }
    __syncthreads();
    constexpr int VC = 64 / V;
    const int Pn = n < N ? P : zeros;
    T* dst = out + (int64_t)n * P * Ct;
#pragma unroll
    for (int it = 0; it < 64 * VC / 256; ++it) {
        const int idx = threadIdx.x + it * 256, pp = idx / VC, cv = idx % VC;
        if (p0 + pp < Pn && c0 + cv * V < Ct) {
            raw16_t r;
            T* e = reinterpret_cast<T*>(&r);
#pragma unroll
            for (int k = 0; k < V; ++k) e[k] = tile[(cv * V + k) * PITCH + pp];
            *reinterpret_cast<raw16_t*>(dst + (int64_t)(p0 + pp) * Ct + c0 + cv * V) = r;
        }
    }
}

// The first layer of an image network (bf16, at most four channels, a window of 5 to 8 positions along w): x is copied with four
// channels per position and the rows' padding in place, so that the positions of a window in one source row are one run of at
// most 32 elements.  A stage of the contraction is such a run: kH stages instead of kW kH / 4 over channels padded to eight (7 x 7:
// 224 against 392; 224 x 224 x 3 x 32 -> 64 channels at stride 2: output 66 -> 53 us, filter gradient 75 -> 42, each copy of x 12 -> 7).
struct Runs {
    int W2 = 0;                // positions of a copied row, even; 0: not this kind of layer
    static constexpr int EL = 32;
};
template <typename T>
static Runs runs_of(const ConvGeom& g) {
    Runs r;
    const int64_t w2 = ((int64_t)(g.OW - 1) * g.sw + Runs::EL / 4 + 1) / 2 * 2;
    if (sizeof(T) == 2 && g.groups == 1 && g.Cin <= 4 && g.kW >= 5 && g.kW <= Runs::EL / 4 && g.dw == 1 &&
        w2 * g.H * g.N < (int64_t(1) << 28))
        r.W2 = (int)w2;
    return r;
}
// Blocks behind the copy's pack the filter: wout[co][kb][ka][4 channels], 32 elements per kb
__global__ __launch_bounds__(256) void runs_copy_pack_kernel(const bf16_t* __restrict__ x, bf16_t* __restrict__ out, FastDiv div_half, FastDiv divH,
                                                             uint32_t pairs, int W2, int blocks, const bf16_t* __restrict__ w, bf16_t* __restrict__ wout,
                                                             ConvGeom g) {
    if ((int)blockIdx.x >= blocks) {
        const int e = ((int)blockIdx.x - blocks) * 256 + (int)threadIdx.x, K = g.kH * Runs::EL;
        if (e >= g.Cout * K) return;
        const int co = e / K, k = e - co * K, kb = k / Runs::EL, ka = (k - kb * Runs::EL) / 4, ci = k & 3;
        bf16_t v = 0;
        if (ka < g.kW && ci < g.Cin) {
            const int a = g.flip ? ka : g.kW - 1 - ka, b = g.flip ? kb : g.kH - 1 - kb;
            v = w[a + (int64_t)g.kW * (b + g.kH * (ci + g.Cin * co))];
        }
        wout[e] = v;
        return;
    }
    const uint32_t idx = blockIdx.x * 256u + threadIdx.x;
    if (idx >= pairs) return;
    const uint32_t row = div_half.div(idx), n = divH.div(row), h = row - n * (uint32_t)g.H;
    const int p = (int)(idx - row * div_half.d) * 2 - g.pw;
    bf16_t e[8];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const bool in = c < g.Cin && (unsigned)(p + j) < (unsigned)g.W;
            e[4 * j + c] = x[in ? (((int64_t)n * g.Cin + c) * g.H + h) * g.W + p + j : 0];
            if (!in) e[4 * j + c] = 0;
        }
    *reinterpret_cast<raw16_t*>(out + (size_t)idx * 8) = *reinterpret_cast<const raw16_t*>(e);
}
static int runs_copy_pack(hipStream_t s, const ConvGeom& g, Runs r, const bf16_t* x, bf16_t* out, const bf16_t* w, bf16_t* wout) {
    const int64_t pairs = (int64_t)g.N * g.H * (r.W2 / 2), blocks = ceil_div(pairs, 256);
    const int64_t pack = wout != nullptr ? ceil_div((int64_t)g.Cout * g.kH * Runs::EL, 256) : 0;
    LUX_UNSUPPORTED_IF((int64_t)g.Cout * g.kH * Runs::EL >= (int64_t(1) << 30), "conv: filter too large");
    ProfScope ps("whcn_to_cwhn_kernel", s);
    runs_copy_pack_kernel<<<(unsigned)(blocks + pack), 256, 0, s>>>(x, out, FastDiv((uint32_t)(r.W2 / 2)), FastDiv((uint32_t)g.H), (uint32_t)pairs, r.W2,
                                                                    (int)blocks, w, wout, g);
    LUX_CHECK_LAUNCH();
    return LUXHIP_OK;
}

// First pass of the fused pullback: one pass over delta writes dz = delta .* act'(y, pre) channel-contiguous with its channels padded to Cp (dzT: what
// the input-gradient and the general filter-gradient kernels read), as it lies (dz, may be null: what the window and the direct filter-gradient
// kernels read) and the bias gradient's partial sums, where a pass for dz and the bias gradient followed by a transposing copy
// reads dz once more and always writes it.  A workgroup walks `chunk` tiles of 64 positions x 64 channels of one image; a tile goes through LDS as fp32 (rows
// of 65 words: the 64 lanes of a wave hit 64 banks in both phases).  Phase 1: 16-byte vectors along p, dz stored, per-channel sums
// kept in registers; phase 2: a vector of channels of one position per thread, 16 bytes of dzT.  The threads of a
// channel add their sums in a fixed order; partial[(n * gridDim.x + blockIdx.x) * C + c].  The z slices behind
// the N images repack the filter for the input-gradient kernel (for its first launch where that is a general one, ps.total > 0).
// RAGGED: any P, C and alignment of delta, y, pre and dz; otherwise P and C are whole vectors, Cp is C and every pointer is 16-byte aligned.
// Bound by HBM (5.6 TB/s at large sizes).  56 x 56 x 128 x 64 in fp32, swish: 57 + 37 us in two passes, 63 in one; 112 x 112 x 64 x 32 in bf16 (nothing reads dz as it
// lies): 36.8 + 4.8 for the filter, 29.7 together; 14 x 14 x 16 -> 32 x 4 in fp32, whole step: 44 -> 38.3.
template <typename T, int ACT, bool RAGGED>
__global__ __launch_bounds__(256) void conv_dz_cwhn_pack_kernel(const T* __restrict__ delta, const T* __restrict__ y, const T* __restrict__ pre, T* dz,
                                                                T* __restrict__ dzT, float* __restrict__ partial, int P, int C, int Cp, int N, int chunk,
                                                                const T* __restrict__ w, T* __restrict__ wout, ConvGeom g, PackSubs ps) {
    constexpr int V = Vec<T>::N, VR = 64 / V, PER = 64 * VR / 256, PITCH = 65;
    if ((int)blockIdx.z >= N) {
        const int64_t block = ((int64_t)(blockIdx.z - N) * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x;
        if (ps.total > 0) pack_sub_element<T>(w, wout, g, ps, block * 256 + threadIdx.x);
        else pack_filter_element<T>(w, wout, g, 1, (int)(block * 256 + threadIdx.x));
        return;
    }
    __shared__ float tile[64 * PITCH];
    const int n = blockIdx.z, c0 = blockIdx.y * 64;
    const size_t image = (size_t)n * C * P, imageT = (size_t)n * Cp * P;
    float bsum[PER] = {};
    const int tiles_p = (P + 63) / 64;
    const int t_end = min(tiles_p, ((int)blockIdx.x + 1) * chunk);
    for (int tp = blockIdx.x * chunk; tp < t_end; ++tp) {
        const int p0 = tp * 64;
        float r[PER][V];
#pragma unroll
        for (int it = 0; it < PER; ++it) {               // loads first, then the stores
            const int idx = threadIdx.x + it * 256, c = c0 + idx / VR, p = p0 + idx % VR * V;
            const size_t off = image + (size_t)c * P + p;
            if (c < C && p + V <= P) {
                dx_vec<T, ACT, V, RAGGED>(delta, y, pre, off, r[it]);
            } else {
#pragma unroll
                for (int k = 0; k < V; ++k) {
                    float v[1] = {0.0f};
                    if constexpr (RAGGED) {
                        if (c < C && p + k < P) dx_vec<T, ACT, 1>(delta, y, pre, off + k, v);
                    }
                    r[it][k] = v[0];
                }
            }
        }
#pragma unroll
        for (int it = 0; it < PER; ++it) {
            const int idx = threadIdx.x + it * 256, cl = idx / VR, pv = idx % VR, c = c0 + cl, p = p0 + pv * V;
            if (dz != nullptr && c < C) {
                const size_t off = image + (size_t)c * P + p;
                if (p + V <= P) {
                    row_store<T, V, RAGGED>(dz, off, r[it], 0);
                } else if constexpr (RAGGED) {
#pragma unroll
                    for (int k = 0; k < V; ++k)
                        if (p + k < P) st(dz + off + k, r[it][k]);
                }
            }
            float t = 0.0f;
#pragma unroll
            for (int k = 0; k < V; ++k) {
                tile[cl * PITCH + pv * V + k] = r[it][k];
                t += r[it][k];
            }
            bsum[it] += t;
        }
        __syncthreads();
#pragma unroll
        for (int it = 0; it < PER; ++it) {
            const int idx = threadIdx.x + it * 256, pl = idx / VR, cv = idx % VR;
            if (p0 + pl < P && c0 + cv * V < Cp) {
                float v[V];
#pragma unroll
                for (int k = 0; k < V; ++k) v[k] = tile[(cv * V + k) * PITCH + pl];
                store_vec<T, V>(dzT, imageT + (size_t)(p0 + pl) * Cp + c0 + cv * V, v);
            }
        }
        __syncthreads();
    }
    if (partial != nullptr) {
#pragma unroll
        for (int it = 0; it < PER; ++it) {
            const int idx = threadIdx.x + it * 256, cl = idx / VR, pv = idx % VR;
            // the threads of a channel are neighbouring lanes: (((s0 + s1) + (s2 + s3)) + ((s4 + s5) + (s6 + s7))) ...
            float t = bsum[it];
#pragma unroll
            for (int o = 1; o < VR; o *= 2) t += __shfl_xor(t, o);
            if (pv == 0 && c0 + cl < C) partial[((size_t)n * gridDim.x + blockIdx.x) * C + c0 + cl] = t;
        }
    }
}

// dbias[c] = sum over slices of partial[slice][c]: one workgroup per channel, thread t adds slices t, t + 256, ...;
// the threads' sums are added in a fixed order (within a wave, then the four waves in turn).
// What is left of the bias gradient after conv_dz_cwhn_pack_kernel: `slices` partial sums per channel.  Either a launch of
// its own or extra workgroups of the launch that adds up the filter gradient's partial sums (both are a few microseconds).
struct BiasPartials {
    const float* partial = nullptr;
    void* dbias = nullptr;
    int C = 0, slices = 0;
};
template <typename T>
__device__ __forceinline__ void conv_dbias_finalize_channel(const float* __restrict__ partial, T* dbias, int C, int S, int c) {
    __shared__ float sw[4];
    float t = 0.0f;
    for (int sl = threadIdx.x; sl < S; sl += 256) t += partial[(size_t)sl * C + c];
    t = wave_sum(t);
    if ((threadIdx.x & 63) == 0) sw[threadIdx.x >> 6] = t;
    __syncthreads();
    if (threadIdx.x == 0) st(dbias + c, ((sw[0] + sw[1]) + sw[2]) + sw[3]);
}
template <typename T>
__global__ __launch_bounds__(256) void conv_dbias_finalize_kernel(const float* __restrict__ partial, T* dbias, int C, int S) {
    conv_dbias_finalize_channel<T>(partial, dbias, C, S, (int)blockIdx.x);
}

// dw[a, b, ci, g*Cout_g + col] = sum over slices of partial[slice][m' = t*Cin_g + ci][col].
// A thread owns 4 consecutive m' (one 16-byte load per slice, eight slices in flight) of every `parts`-th slice; the parts of a
// workgroup's values are added in order through LDS.  Bound by the latency of its trips to memory: with a thread per value (parts = 1) a filter of
// few values on many slices is a handful of workgroups with 64 trips each (64 x 51 values, 419 slices: 23.0 us, in 32 parts 6.9).
template <typename T>
__global__ __launch_bounds__(256) void wgrad_reduce_kernel(const float* __restrict__ partial, T* __restrict__ dw, ConvGeom g,
                                                           int grp, int slices, int parts, int reduce_blocks, int Mrows, int Cp, int run, int64_t slice_stride,
                                                           BiasPartials bp) {
    if ((int)blockIdx.x >= reduce_blocks) {       // workgroups behind the reduction: one channel of the bias gradient each
        conv_dbias_finalize_channel<T>(bp.partial, static_cast<T*>(bp.dbias), bp.C, bp.slices, (int)blockIdx.x - reduce_blocks);
        return;
    }
    // Cp: channels per tap in the partial sums (padded); run > 0: rows are [kb][run / 4 positions][4 channels] instead
    __shared__ float sums[256 * 4];
    const int total = Mrows * g.Cout_g;
    const int quads = 256 / parts, part = (int)threadIdx.x / quads;
    const int idx = ((int)blockIdx.x * quads + (int)threadIdx.x % quads) * 4;
    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    const bool vec = (total & 3) == 0 && (slice_stride & 3) == 0;   // then idx + 3 < total and every slice row is 16-byte aligned
    if (vec && idx < total) {
        int sl = part;
        for (; sl + 7 * parts < slices; sl += 8 * parts) {
            float4 v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = *reinterpret_cast<const float4*>(partial + (size_t)(sl + u * parts) * slice_stride + idx);
#pragma unroll
            for (int u = 0; u < 8; ++u) { acc[0] += v[u].x; acc[1] += v[u].y; acc[2] += v[u].z; acc[3] += v[u].w; }
        }
#pragma unroll 4
        for (; sl < slices; sl += parts) {
            const float4 v = *reinterpret_cast<const float4*>(partial + (size_t)sl * slice_stride + idx);
            acc[0] += v.x; acc[1] += v.y; acc[2] += v.z; acc[3] += v.w;
        }
    } else {
        for (int sl = part; sl < slices; sl += parts)
            for (int e = 0; e < 4; ++e)
                if (idx + e < total) acc[e] += partial[(size_t)sl * slice_stride + idx + e];
    }
    if (parts > 1) {
#pragma unroll
        for (int e = 0; e < 4; ++e) sums[threadIdx.x * 4 + e] = acc[e];
        __syncthreads();
        if (part != 0) return;
        for (int p = 1; p < parts; ++p)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[e] += sums[(threadIdx.x + p * quads) * 4 + e];
    }
    for (int e = 0; e < 4; ++e) {
        const int id = idx + e;
        if (id >= total) break;
        const int m = id % Mrows, col = id / Mrows;
        const int t = m / Cp, ci = m - t * Cp;
        const int taps = run > 0 ? run / 4 : g.kW, ka = t % taps, kb = t / taps;
        if (ci >= g.Cin_g || ka >= g.kW) continue;
        const int a = g.flip ? ka : g.kW - 1 - ka, b = g.flip ? kb : g.kH - 1 - kb;
        st(dw + a + g.kW * (b + g.kH * (ci + g.Cin_g * (grp * g.Cout_g + col))), acc[e]);
    }
}

// ----------------------------------------------------------------------------- host helpers
static int make_geom(const luxhip_conv_dims_t* d, ConvGeom* g) {
    LUX_INVALID_IF(d == nullptr, "conv: dims must not be NULL");
    LUX_INVALID_IF(d->W <= 0 || d->H <= 0 || d->Cin <= 0 || d->N < 0 || d->kW <= 0 || d->kH <= 0 || d->Cout <= 0,
                   "conv: non-positive dimension");
    LUX_INVALID_IF(d->stride_w <= 0 || d->stride_h <= 0 || d->dil_w <= 0 || d->dil_h <= 0 || d->groups <= 0,
                   "conv: stride, dilation and groups must be positive");
    LUX_INVALID_IF(d->pad_w_lo < 0 || d->pad_w_hi < 0 || d->pad_h_lo < 0 || d->pad_h_hi < 0, "conv: negative padding");
    LUX_INVALID_IF(d->Cin % d->groups != 0 || d->Cout % d->groups != 0, "conv: channels must be divisible by groups");
    const int64_t ow = (d->W + d->pad_w_lo + d->pad_w_hi - d->dil_w * (d->kW - 1) - 1) / d->stride_w + 1;
    const int64_t oh = (d->H + d->pad_h_lo + d->pad_h_hi - d->dil_h * (d->kH - 1) - 1) / d->stride_h + 1;
    LUX_INVALID_IF(ow <= 0 || oh <= 0, "conv: empty output");
    const long double big = 2147483648.0L;
    LUX_UNSUPPORTED_IF((long double)d->W * d->H * d->Cin * std::max<int64_t>(d->N, 1) >= big ||
                           (long double)ow * oh * d->Cout * std::max<int64_t>(d->N, 1) >= big,
                       "conv: tensors of 2^31 or more elements are not supported");
    g->W = (int)d->W; g->H = (int)d->H; g->Cin = (int)d->Cin; g->N = (int)d->N; g->kW = (int)d->kW; g->kH = (int)d->kH;
    g->Cout = (int)d->Cout; g->OW = (int)ow; g->OH = (int)oh; g->sw = (int)d->stride_w; g->sh = (int)d->stride_h;
    g->pw = (int)d->pad_w_lo; g->ph = (int)d->pad_h_lo; g->dw = (int)d->dil_w; g->dh = (int)d->dil_h;
    g->groups = (int)d->groups; g->Cin_g = (int)(d->Cin / d->groups); g->Cout_g = (int)(d->Cout / d->groups);
    g->flip = d->flipkernel != 0;
    return LUXHIP_OK;
}

static inline size_t align256(size_t b) { return (b + 255) & ~size_t(255); }

template <typename T>
static int transpose_to_cwhn(hipStream_t s, const T* in, T* out, int P, int C, int N) {
    ProfScope ps("whcn_to_cwhn_kernel", s);
    constexpr int V = 16 / (int)sizeof(T);
    const bool vec = P % V == 0 && C % V == 0 && aligned16(in) && aligned16(out);
    const int tile = vec ? 64 : 32;
    dim3 grid((unsigned)ceil_div(P, tile), (unsigned)ceil_div(C, tile), (unsigned)N);
    LUX_UNSUPPORTED_IF(grid.y > 65535 || grid.z > 65535, "conv: too many channels or images for the layout transform");
    if (vec) whcn_to_cwhn_vec_kernel<T><<<grid, 256, 0, s>>>(in, out, P, C);
    else whcn_to_cwhn_kernel<T><<<grid, 256, 0, s>>>(in, out, P, C);
    LUX_CHECK_LAUNCH();
    return LUXHIP_OK;
}

// out (C x P, C contiguous) = transpose of in (P x C, P contiguous); for the GEMM dispatch, which
// turns large operands into the K-major layout its fastest kernel reads
int transpose_matrix_bf16(hipStream_t s, const bf16_t* in, bf16_t* out, int64_t P, int64_t C) {
    LUX_UNSUPPORTED_IF(P >= (1ll << 31) || C >= (1ll << 31), "matrix too large for the layout transform");
    return transpose_to_cwhn<bf16_t>(s, in, out, (int)P, (int)C, 1);
}

template <typename T>
static int pack_filter(hipStream_t s, const T* w, T* out, const ConvGeom& g, int for_dgrad) {
    ProfScope ps("pack_filter_kernel", s);
    const int total = g.kW * g.kH * g.Cin_g * g.Cout;
    pack_filter_kernel<T><<<(unsigned)ceil_div(total, 256), 256, 0, s>>>(w, out, g, for_dgrad);
    LUX_CHECK_LAUNCH();
    return LUXHIP_OK;
}

template <typename T>
static int to_cwhn_padded(hipStream_t s, const T* in, T* out, int P, int Cin, int Cg, int groups, int N, int zeros, const ConvGeom& g);

// transpose_to_cwhn(in -> out) and pack_filter(w -> wout) in one launch where the 16-byte transform applies
template <typename T>
static int transpose_and_pack(hipStream_t s, const T* in, T* out, int P, int C, int N, const T* w, T* wout, const ConvGeom& g, int for_dgrad) {
    constexpr int V = 16 / (int)sizeof(T);
    const bool vec = P % V == 0 && C % V == 0 && aligned16(in) && aligned16(out);
    const int64_t gx = ceil_div(P, 64), gy = ceil_div(C, 64);
    const int64_t pack_blocks = ceil_div((int64_t)g.kW * g.kH * g.Cin_g * g.Cout, 256);
    const int64_t gz = N + ceil_div(pack_blocks, gx * gy);
    if (!vec || N < 1 || gy > 65535 || gz > 65535) {
        int rc = to_cwhn_padded<T>(s, in, out, P, C, C / g.groups, g.groups, N, 0, g);
        if (rc != LUXHIP_OK) return rc;
        return pack_filter<T>(s, w, wout, g, for_dgrad);
    }
    ProfScope ps("whcn_to_cwhn_kernel", s);
    whcn_to_cwhn_pack_kernel<T><<<dim3((unsigned)gx, (unsigned)gy, (unsigned)gz), 256, 0, s>>>(in, out, P, C, N, w, wout, g, for_dgrad);
    LUX_CHECK_LAUNCH();
    return LUXHIP_OK;
}

// Tiles of 64 positions that one workgroup of conv_dz_cwhn_pack_kernel walks: as many as leave about four workgroups
// per compute unit, eight at most (each workgroup contributes one slice of partial sums per channel)
static int dz_cwhn_chunk(int P, int C, int N) {
    const int64_t tiles = ceil_div(P, 64) * ceil_div(C, 64) * N;
    return (int)std::min<int64_t>(8, std::max<int64_t>(1, tiles / (4 * (int64_t)std::max(1, num_cus()))));
}
static size_t dz_cwhn_partial_bytes(int P, int C, int N) {
    const int64_t groups = ceil_div(ceil_div(P, 64), dz_cwhn_chunk(P, C, N));
    return align256((size_t)groups * N * C * sizeof(float));
}

// ----------------------------------------------------------------------------- any channel count, any stride (conv_any.h)
// Channels of a group padded to whole 16-byte chunks
template <typename T>
static int padded(int c) {
    constexpr int V = GemmTraits<T>::VEC;
    return (c + V - 1) / V * V;
}
// The 3 x 3 window kernel of conv_patch.h takes the problem (pointer alignment is checked again at the launch)
template <typename T>
static bool window_shape(const ConvGeom& g, bool dgrad) {
    if (sizeof(T) != 2 || g.sw != 1 || g.sh != 1 || g.dw != 1 || g.dh != 1 || g.OW != g.W || g.OH != g.H) return false;
    cpatch::Problem p{};
    p.Ctot = dgrad ? g.Cout : g.Cin; p.Cg = dgrad ? g.Cout_g : g.Cin_g; p.P = g.W; p.Q = g.H; p.N = g.N; p.kW = g.kW; p.kH = g.kH;
    p.Ncols = dgrad ? g.Cin_g : g.Cout_g;
    return cpatch::applicable(p);
}
// The whole-tap kernels: channels per group in whole stages, for the input gradient a unit stride, and enough work to fill
// the chip with their large tiles.  Below that the kernels of conv_any.h are ahead: bf16 5 x 5, 192 -> 16 channels on 25 x 25
// x 18 107 us against 33, fp32 5 x 5, 208 -> 40 on 66 x 66 x 4 417 against 162; with the chip full they are not: bf16 3 x 3,
// 128 channels on 56 x 56 x 64 63 us (window kernel) against 132, fp32 541 against 550 (both on the fp32 instruction then).
template <typename T>
static bool tap_shape(const ConvGeom& g, bool dgrad) {
    const int Cg = dgrad ? g.Cout_g : g.Cin_g, Ncols = dgrad ? g.Cin_g : g.Cout_g;
    const int64_t src = dgrad ? (int64_t)g.OW * g.OH * g.Cout * g.N : (int64_t)g.W * g.H * g.Cin * g.N;
    if (Cg % GemmTraits<T>::BK != 0 || (dgrad && (g.sw != 1 || g.sh != 1)) || src >= (int64_t(1) << 30)) return false;
    if (option_conv_tile() != 0) return true;
    const int64_t rows = dgrad ? (int64_t)g.W * g.H * g.N : (int64_t)g.OW * g.OH * g.N, cus = num_cus() > 0 ? num_cus() : 256;
    const int64_t tiles_n = ceil_div(Ncols, 128);
    if (window_shape<T>(g, dgrad)) return ceil_div(rows, 256) * ceil_div(Ncols, 64) >= cus;
    return ceil_div(rows, sizeof(T) == 2 ? 512 : 128) * tiles_n >= cus && Ncols * 4 >= tiles_n * 128 * 3;
}

struct Residue { int r, count, q0, s0, sstep, taps; };      // residue, rows, first q, first shift and step, taps
// Residue r of one dimension of the input gradient: input positions i = stride q + r - pad in [0, L); k0 is its first tap (taps
// if it has none)
static Residue residue(int r, int k0, int L, int pad, int stride, int dil, int taps) {
    auto floor_div = [](int64_t a, int64_t b) { return a >= 0 ? a / b : -((-a + b - 1) / b); };
    Residue z{r, 0, 0, 0, 1, 0};
    z.q0 = (int)-floor_div((int64_t)r - pad, stride);        // ceil((pad - r) / stride)
    z.count = (int)std::max<int64_t>(0, floor_div((int64_t)L - 1 + pad - r, stride) - z.q0 + 1);
    int gq = stride, t = dil;
    while (t) { const int u = gq % t; gq = t; t = u; }
    z.sstep = dil / gq;
    if (k0 < taps) { z.taps = (taps - 1 - k0) / (stride / gq) + 1; z.s0 = (int)(((int64_t)k0 * dil - r) / stride); }
    return z;
}
// The residues that have taps (no more than there are taps), by number, and with `all` also those without; a position of a
// residue without taps has a gradient of zero
static std::vector<Residue> residues(bool all, int L, int pad, int stride, int dil, int taps) {
    std::vector<Residue> z;
    std::vector<std::pair<int, int>> first;                  // (residue, its first tap)
    int gq = stride, t = dil;
    while (t) { const int u = gq % t; gq = t; t = u; }
    for (int k = 0; k < std::min(taps, stride / gq); ++k) first.emplace_back((int)((int64_t)k * dil % stride), k);
    if (all)
        for (int r = 0; r < stride; ++r)
            if (std::none_of(first.begin(), first.end(), [&](const std::pair<int, int>& f) { return f.first == r; })) first.emplace_back(r, taps);
    std::sort(first.begin(), first.end());
    for (const auto& f : first) z.push_back(residue(f.first, f.second, L, pad, stride, dil, taps));
    return z;
}

// The sub-problems of one convolution, in groups of one launch each.
template <typename T>
struct AnyPlan {
    struct Launch { cany::Sub sub[cany::MAX_SUBS]; PackSub pack[cany::MAX_SUBS]; int n; };
    std::vector<Launch> launches;
    int Ncols = 0, Cch = 0, res_w = 0, merged = 0, Cp = 0;
    Runs runs;                                               // fprop: stages are runs of positions
    bool zero_first = false;                                 // some positions of dx belong to no sub-problem: clear it before
    int64_t wm_elems = 0;                                    // packed filter of one group
    bool slices = true;                                      // contractions may be cut (workspace for the partial sums)
    // Memory for the slices of any launch: what a call reserves behind its `front` bytes, unless the stream is recording and
    // its workspace has no room for them (then the contractions stay whole)
    size_t reserve(hipStream_t s, size_t front, int at_a_time, int groups) {
        size_t most = 0;
        for (Launch& l : launches)
            for (int n : {at_a_time, groups % at_a_time})    // the last of them may be fewer
                if (n > 0) most = std::max(most, cany::choose_any<T>(l.sub, l.n, Ncols, n, true).bytes * n);
        slices = workspace_holds(s, front + most);
        return front + (slices ? most : 0);
    }
    void add(const Residue& rw, int RA, const Residue& rh, int RB, int N, int w0, int wstep, int TW, int h0, int hstep, int TH, int ow0, int oh0) {
        if (RA <= 0 || RB <= 0) return;
        if (launches.empty() || launches.back().n == cany::MAX_SUBS) { launches.emplace_back(); launches.back().n = 0; }
        Launch& l = launches.back();
        cany::Sub& q = l.sub[l.n];
        q.RA = RA; q.RAB = RA * RB; q.M = RA * RB * N;
        q.w0 = w0; q.wstep = wstep; q.h0 = h0; q.hstep = hstep; q.TW = std::max(TW, 1); q.TH = TH;
        q.K = TW * TH * Cp;
        q.Kpad = (q.K + GemmTraits<T>::BK - 1) / GemmTraits<T>::BK * GemmTraits<T>::BK;
        q.ow0 = ow0; q.oh0 = oh0; q.wm = wm_elems;
        q.divRA = FastDiv((uint32_t)RA); q.divRAB = FastDiv((uint32_t)(RA * RB)); q.divTW = FastDiv((uint32_t)q.TW);
        PackSub& k = l.pack[l.n];
        k = PackSub{rw.r, rh.r, rw.s0, rw.sstep, rh.s0, rh.sstep, q.TW, q.K, q.Kpad, res_w, wm_elems, 0};
        wm_elems += (int64_t)Ncols * q.Kpad;
        ++l.n;
    }
    AnyPlan(const ConvGeom& g, bool dgrad) {
        Cp = padded<T>(dgrad ? g.Cout_g : g.Cin_g);
        Ncols = Cch = dgrad ? g.Cin_g : g.Cout_g;
        const Residue none{0, 0, 0, 0, 1, 0};
        if (!dgrad) {
            runs = runs_of<T>(g);
            if (runs.W2 > 0) {
                Cp = Runs::EL;
                add(none, g.OW, none, g.OH, g.N, 0, 0, 1, -g.ph, g.dh, g.kH, 0, 0);
            } else {
                add(none, g.OW, none, g.OH, g.N, -g.pw, g.dw, g.kW, -g.ph, g.dh, g.kH, 0, 0);
            }
            return;
        }
        // Where all residues fit one launch, those without taps write their zeros in it; of more (a stride of 32 has 1024)
        // only those with taps are problems, and dx is cleared first if there are others (64 x 64 x 32 x 16, 1 x 1, stride 32:
        // 43 us, against 2022 with 256 launches)
        const int64_t R = (int64_t)g.sw * g.sh;
        const bool all = R <= cany::MAX_SUBS;
        const std::vector<Residue> rw = residues(all, g.W, g.pw, g.sw, g.dw, g.kW), rh = residues(all, g.H, g.ph, g.sh, g.dh, g.kH);
        // One problem per residue, or all residues as columns of one: whichever is less work in 32-column tiles.  A launch
        // and the repacking of its filters (10 us, at the rates that such problems reach) count as work.  (64 -> 256 channels,
        // 16 x 16, stride 16 on 64 x 64 x 16, forward and pullback in bf16: 849 us with 64 launches, 148 with one.)
        auto cols = [](double n) { return std::ceil(n / 32.0) * 32.0; };
        const double per_launch = (sizeof(T) == 2 ? 1.5e9 : 3e8) / ((double)g.N * Cp);
        double apart = std::ceil((double)rw.size() * rh.size() / cany::MAX_SUBS - 1.0) * per_launch, together = 1e30, rows = 0.0;
        for (const Residue& a : rw)
            for (const Residue& b : rh) { apart += (double)a.count * b.count * a.taps * b.taps * cols(g.Cin_g); rows += (double)a.count * b.count; }
        auto unite = [](int L, int pad, int stride, const std::vector<Residue>& v) {      // dilation 1: every residue starts at shift 0
            Residue u{0, (L - 1 + pad) / stride - pad / stride + 1, pad / stride, 0, 1, 0};
            for (const Residue& z : v) u.taps = std::max(u.taps, z.taps);
            return u;
        };
        Residue uw{}, uh{};
        if (R > 1 && R * g.Cin_g <= 65536 && g.dw == 1 && g.dh == 1) {
            uw = unite(g.W, g.pw, g.sw, rw);
            uh = unite(g.H, g.ph, g.sh, rh);
            if ((double)uw.taps * uh.taps * Cp * R * g.Cin_g * sizeof(T) < 2147483648.0)
                together = (double)uw.count * uh.count * uw.taps * uh.taps * cols((double)R * g.Cin_g);
        }
        if (together < apart) {
            merged = 1;
            res_w = g.sw;
            Ncols = (int)R * g.Cin_g;
            add(uw, uw.count, uh, uh.count, g.N, uw.q0, -1, uw.taps, uh.q0, -1, uh.taps, g.sw * uw.q0 - g.pw, g.sh * uh.q0 - g.ph);
            return;
        }
        zero_first = rows < (double)g.W * g.H;
        for (const Residue& b : rh)
            for (const Residue& a : rw)
                add(a, a.count, b, b.count, g.N, a.q0 - a.s0, -a.sstep, a.taps, b.q0 - b.s0, -b.sstep, b.taps, g.sw * a.q0 + a.r - g.pw,
                    g.sh * b.q0 + b.r - g.ph);
    }
    PackSubs pack(const ConvGeom& g, bool dgrad, size_t launch) const {
        PackSubs p;
        p.n = launches[launch].n; p.dgrad = dgrad; p.Cp = Cp; p.Ncols = Ncols; p.Cch = Cch; p.wm_group = wm_elems; p.per_group = 0;
        for (int i = 0; i < p.n; ++i) {
            p.sub[i] = launches[launch].pack[i];
            p.sub[i].first = p.per_group;
            p.per_group += (int64_t)Ncols * p.sub[i].Kpad;
        }
        p.total = p.per_group * g.groups;
        return p;
    }
};

// Padded channel-contiguous copy of the first `groups` groups of `in`, which has Cin channels (if out != NULL), and the packed
// filter of all groups of a launch (if wout != NULL), in one launch
template <typename T>
static int pad_and_pack(hipStream_t s, const T* in, T* out, int P, int Cin, int Cg, int groups, int N, int zeros, const T* w, T* wout, const ConvGeom& g,
                        const PackSubs* ps) {
    constexpr int V = GemmTraits<T>::VEC;
    const int Cp = padded<T>(Cg), Ct = groups * Cp;
    PackSubs none;
    none.n = 0; none.total = 0;
    int64_t blocks = 0;
    const int tiles_p = (int)ceil_div(std::max(P, zeros), 64), tiles_c = (int)ceil_div(Ct, 64);
    if (out != nullptr) blocks = Ct == V ? ceil_div((int64_t)P * N + zeros, 256) : (int64_t)tiles_p * tiles_c * (N + (zeros > 0));
    const int64_t pack = wout != nullptr ? ceil_div(ps->total, 256) : 0;
    LUX_UNSUPPORTED_IF((blocks + pack) * 256 >= kMostThreads, "conv: tensor too large for the layout transform");
    if (blocks + pack == 0) return LUXHIP_OK;
    ProfScope prof("whcn_to_cwhn_kernel", s);
    pad_to_cwhn_pack_kernel<T><<<(unsigned)(blocks + pack), 256, 0, s>>>(in, out, P, Cin, Cg, Cp, groups, N, zeros, tiles_p, tiles_c, (int)blocks, w, wout,
                                                                         g, wout != nullptr ? *ps : none);
    LUX_CHECK_LAUNCH();
    return LUXHIP_OK;
}

// Channel-contiguous copy of a tensor in the padded layout (the plain layout where no padding is needed)
template <typename T>
static int to_cwhn_padded(hipStream_t s, const T* in, T* out, int P, int Cin, int Cg, int groups, int N, int zeros, const ConvGeom& g) {
    if (padded<T>(Cg) == Cg && Cin == Cg * groups && zeros == 0 && P % GemmTraits<T>::VEC == 0 && aligned16(in))
        return transpose_to_cwhn<T>(s, in, out, P, Cin, N);
    return pad_and_pack<T>(s, in, out, P, Cin, Cg, groups, N, zeros, nullptr, nullptr, g, nullptr);
}

// The single pass pays where a tile is not mostly empty; smaller ragged planes and channel counts take the two passes
template <typename T>
static bool dz_cwhn_ok(int P, int C, int N) {
    return ((P >= 32 && C >= 16) || (sizeof(T) == 2 && P % 8 == 0 && C % 8 == 0)) && ceil_div(C, 64) <= 65535 && N >= 1 && N + 4096 <= 65535;
}

// dz may be null; wout: the filter for the input gradient, packed by `ps` (general kernels) or as pack_filter does (ps null)
template <typename T>
static int conv_dz_cwhn_pack(hipStream_t s, int act, const ConvGeom& g, int Cp, const T* delta, const T* y, const T* pre, T* dz, T* dzT, float* partial, T* dbias,
                             const T* w, T* wout, const PackSubs* ps, BiasPartials* later) {
    constexpr int V = Vec<T>::N;
    const int P = g.OW * g.OH, C = g.Cout, N = g.N;
    const int chunk = dz_cwhn_chunk(P, C, N);
    const int64_t gx = ceil_div(ceil_div(P, 64), chunk), gy = ceil_div(C, 64);
    // a filter that is large beside the cotangent does not fit the z slices: it has a launch of its own then, as in the two passes
    const int64_t pack_blocks = wout == nullptr ? 0 : ceil_div(ps != nullptr ? ps->total : (int64_t)g.kW * g.kH * g.Cin_g * g.Cout, 256);
    const int64_t pack_z = ceil_div(pack_blocks, gx * gy);
    const bool fits = N + pack_z <= 65535 && (ps != nullptr || pack_z * gx * gy * 256 < (int64_t(1) << 31));
    if (!fits) {
        const int rc = ps != nullptr ? pad_and_pack<T>(s, nullptr, nullptr, 0, 1, 1, 1, 0, 0, w, wout, g, ps) : pack_filter<T>(s, w, wout, g, 1);
        if (rc != LUXHIP_OK) return rc;
    }
    const int64_t gz = N + (fits ? pack_z : 0);
    float* const part = dbias != nullptr ? partial : nullptr;
    PackSubs subs;
    subs.n = 0; subs.total = 0;
    if (wout != nullptr && ps != nullptr) subs = *ps;
    const bool whole = P % V == 0 && C % V == 0 && Cp == C && aligned16(delta) && aligned16(y) && aligned16(pre) && aligned16(dz);
    const dim3 grid((unsigned)gx, (unsigned)gy, (unsigned)gz);
#define LAUNCH_DZC(A)                                                                                                                         \
    do {                                                                                                                                      \
        if (whole) conv_dz_cwhn_pack_kernel<T, A, false><<<grid, 256, 0, s>>>(delta, y, pre, dz, dzT, part, P, C, Cp, N, chunk, w, wout, g, subs); \
        else conv_dz_cwhn_pack_kernel<T, A, true><<<grid, 256, 0, s>>>(delta, y, pre, dz, dzT, part, P, C, Cp, N, chunk, w, wout, g, subs);        \
    } while (0)
    {
        ProfScope prof("conv_dz_cwhn_pack_kernel", s);
        LUX_DISPATCH_ACT(act, LAUNCH_DZC);
    }
#undef LAUNCH_DZC
    LUX_CHECK_LAUNCH();
    if (dbias != nullptr) {
        if (later != nullptr) {           // the caller adds the channels' sums to a later launch
            later->partial = partial; later->dbias = dbias; later->C = C; later->slices = (int)(gx * N);
            return LUXHIP_OK;
        }
        ProfScope ps2("conv_dbias_finalize_kernel", s);
        conv_dbias_finalize_kernel<T><<<(unsigned)C, 256, 0, s>>>(partial, dbias, C, (int)(gx * N));
        LUX_CHECK_LAUNCH();
    }
    return LUXHIP_OK;
}

// Groups [first, first + n) of a convolution.  Where channels are padded, the copies hold as many groups at a time as take no
// more memory than the tensor itself or 64 MiB: a depthwise bf16 layer would need eight times the tensor for all of them.
struct Groups { int first, n; };
template <typename T>
static int groups_at_a_time(const ConvGeom& g, bool x, bool y) {
    int64_t n = g.groups;
    auto fit = [&](int64_t positions, int Cg) {
        if (padded<T>(Cg) == Cg) return;
        const int64_t room = std::max<int64_t>(int64_t(64) << 20, positions * Cg * g.groups * (int64_t)sizeof(T));
        n = std::min(n, std::max<int64_t>(1, room / (positions * padded<T>(Cg) * (int64_t)sizeof(T))));
    };
    if (x) fit((int64_t)g.W * g.H * g.N, g.Cin_g);
    if (y) fit((int64_t)g.OW * g.OH * g.N, g.Cout_g);
    return (int)std::min<int64_t>(n, 32768);                 // (a dimension of the grid)
}

template <typename T>
__global__ __launch_bounds__(256) void clear_kernel(T* out, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) out[i] = T(0);
}
template <typename T>
static int clear_elements(hipStream_t s, T* out, int64_t n) {
    if ((reinterpret_cast<uintptr_t>(out) & 3u) == 0) return luxhip_fill_zero(out, (size_t)n * sizeof(T), s);
    clear_kernel<T><<<(unsigned)std::min<int64_t>(ceil_div(n, 256), 4096), 256, 0, s>>>(out, n);
    LUX_CHECK_LAUNCH();
    return LUXHIP_OK;
}

// fprop / dgrad of the groups `gr` through conv_any.h.  src: padded channel-contiguous activations, of these groups alone
// where channels are padded, else of all; wm: workspace for the packed filter of all groups; packed: launch 0 of the filter is
// already there.  ws_front: bytes of the workspace in use.
template <typename T>
static int run_conv_any(hipStream_t s, const ConvGeom& g, bool dgrad, const AnyPlan<T>& plan, Groups gr, const T* src, const T* w, T* wm, bool packed,
                        const T* bias, T* out, T* pre, int act, size_t ws_front) {
    const bool alone = plan.Cp != (dgrad ? g.Cout_g : g.Cin_g);
    if (plan.zero_first && gr.first == 0) {
        const int rc = clear_elements<T>(s, out, (int64_t)g.W * g.H * g.Cin * g.N);
        if (rc != LUXHIP_OK) return rc;
    }
    for (size_t li = 0; li < plan.launches.size(); ++li) {
        const typename AnyPlan<T>::Launch& l = plan.launches[li];
        if (gr.first == 0 && !(packed && li == 0)) {
            const PackSubs ps = plan.pack(g, dgrad, li);
            const int rc = pad_and_pack<T>(s, nullptr, nullptr, 0, 1, 1, 1, 0, 0, w, wm, g, &ps);
            if (rc != LUXHIP_OK) return rc;
        }
        cany::Args<T> a;
        a.src = src + (alone ? 0 : (size_t)gr.first * plan.Cp);
        a.wm = wm + gr.first * plan.wm_elems; a.wm_group = plan.wm_elems; a.bias = bias; a.out = out; a.pre = pre;
        a.Ctot = (alone ? gr.n : g.groups) * plan.Cp; a.Cp = plan.Cp;
        if (!dgrad) { a.SP = g.W; a.SQ = g.H; a.ss_w = g.sw; a.ss_h = g.sh; a.P = g.OW; a.Q = g.OH; a.os_w = a.os_h = 1; a.Ctot_out = g.Cout; }
        else { a.SP = g.OW; a.SQ = g.OH; a.ss_w = a.ss_h = 1; a.P = g.W; a.Q = g.H; a.os_w = g.sw; a.os_h = g.sh; a.Ctot_out = g.Cin; }
        a.run = 0;
        if (plan.runs.W2 > 0) { a.Ctot = 4; a.SP = plan.runs.W2; a.run = 4 * g.kW; }
        a.PQ = a.P * a.Q;
        a.Cch = plan.Cch; a.res_w = std::max(plan.res_w, 1); a.merged = plan.merged; a.kW = g.kW; a.kH = g.kH;
        a.act = act; a.subs = l.n;
        a.divCp = FastDiv((uint32_t)plan.Cp); a.divCch = FastDiv((uint32_t)plan.Cch);
        int kmax = 0;
        for (int i = 0; i < l.n; ++i) kmax = std::max(kmax, l.sub[i].Kpad);
        // the kernel's offsets into a tile's filter columns have 32 bits: of filters of 4 GiB fewer columns at a time
        const int most = plan.merged ? plan.Ncols : (int)std::min<int64_t>(plan.Ncols, std::max<int64_t>(1, ((int64_t(1) << 31) / (int64_t)sizeof(T)) / std::max(kmax, 1)));
        const int at_a_time = most >= std::min(plan.Ncols, 128) ? plan.Ncols : most;
        for (int col = 0; col < plan.Ncols; col += at_a_time) {
            a.Ncols = std::min(at_a_time, plan.Ncols - col);
            a.col_off = gr.first * plan.Cch + col;
            for (int i = 0; i < l.n; ++i) {
                a.sub[i] = l.sub[i];
                a.sub[i].wm += (int64_t)col * l.sub[i].Kpad;
            }
            const int rc = cany::launch_any<T>(s, a, gr.n, ws_front, dgrad, plan.slices && at_a_time == plan.Ncols);
            if (rc != LUXHIP_OK) return rc;
        }
    }
    return LUXHIP_OK;
}

// fprop (dgrad == false): out = y; dgrad: out = dx, for problems of tap_shape().  src is the channel-contiguous activation,
// wm the packed filter (all groups), zeros a few zero bytes in device memory.
template <typename T>
static int run_conv_gemm(hipStream_t s, const ConvGeom& g, bool dgrad, const T* src, const T* wm, const T* bias, T* out,
                         T* pre, int act, const void* zeros) {
    const int Tt = g.kW * g.kH;
    const int Cg = dgrad ? g.Cout_g : g.Cin_g;
    for (int grp = 0; grp < g.groups; ++grp) {
        const int Ncols = dgrad ? g.Cin_g : g.Cout_g;
        const int K = Tt * Cg;
        Operand<T> Wm;
        Wm.p = wm + (size_t)grp * Ncols * K;
        Wm.sr = K; Wm.sk = 1; Wm.rows = Ncols;
        Wm.vec_ok = aligned16(Wm.p) && ((size_t)K * sizeof(T)) % 16 == 0;
        int rc;
        if constexpr (sizeof(T) == 2) {
            // unit stride and dilation, output as large as the input: the kernel that keeps a tile's input window in LDS
            if (option_conv_tile() <= 2 && g.sw == 1 && g.sh == 1 && g.dw == 1 && g.dh == 1 && g.OW == g.W && g.OH == g.H) {
                cpatch::Problem p;
                p.src = reinterpret_cast<const bf16_t*>(src) + (size_t)grp * Cg;
                p.wm = reinterpret_cast<const bf16_t*>(Wm.p);
                p.bias = reinterpret_cast<const bf16_t*>(bias);
                p.out = reinterpret_cast<bf16_t*>(out); p.pre = reinterpret_cast<bf16_t*>(pre); p.zero = zeros;
                p.Ctot = dgrad ? g.Cout : g.Cin; p.Cg = Cg; p.P = g.W; p.Q = g.H; p.N = g.N;
                p.kW = g.kW; p.kH = g.kH; p.pad_w = g.pw; p.pad_h = g.ph; p.dgrad = dgrad;
                p.Ncols = Ncols; p.col_off = grp * Ncols; p.Ctot_out = dgrad ? g.Cin : g.Cout; p.act = act;
                if (cpatch::applicable(p)) {
                    if ((rc = cpatch::launch(s, p)) != LUXHIP_OK) return rc;
                    continue;
                }
            }
        }
        ConvTapArgs<T> a;
        TapGeom<T>& q = a.tap;
        q.kW = g.kW; q.sw = g.sw; q.sh = g.sh; q.pw = g.pw; q.ph = g.ph; q.dw = g.dw; q.dh = g.dh;
        q.dgrad = dgrad;
        q.Cg = Cg;
        if (!dgrad) { q.Ctot = g.Cin; q.P = g.OW; q.PQ = g.OW * g.OH; q.SP = g.W; q.SQ = g.H; }
        else { q.Ctot = g.Cout; q.P = g.W; q.PQ = g.W * g.H; q.SP = g.OW; q.SQ = g.OH; }
        q.M = q.PQ * g.N;
        q.divP = FastDiv((uint32_t)q.P); q.divPQ = FastDiv((uint32_t)q.PQ); q.divCg = FastDiv((uint32_t)q.Cg);
        q.divkW = FastDiv((uint32_t)g.kW);
        q.src = src + (size_t)grp * Cg;
        q.zero = zeros;
        a.Wm = Wm; a.K = K; a.Ncols = Ncols;
        a.out = out; a.pre = pre; a.bias = bias;
        a.Ctot_out = dgrad ? g.Cin : g.Cout;
        a.col_off = grp * Ncols;
        a.act = act;
        a.m_begin = 0;
        rc = launch_conv_tap_any<T>(s, a);
        if (rc != LUXHIP_OK) return rc;
    }
    return LUXHIP_OK;
}

// Rows (taps x padded channels), columns and slices of the filter gradient's partial sums
struct WgradPlan { int Mrows, Ncols, slices, kslice; bool narrow; };
template <typename T>
static int wgrad_plan(const ConvGeom& g, bool any, Runs runs, WgradPlan* p) {
    constexpr int BK = GemmTraits<T>::BK;
    p->Mrows = any && runs.W2 > 0 ? g.kH * Runs::EL : g.kW * g.kH * (any ? padded<T>(g.Cin_g) : g.Cin_g);
    p->Ncols = any ? padded<T>(g.Cout_g) : g.Cout_g;
    p->narrow = p->Mrows <= 64 || p->Ncols <= 64;
    const int tile = p->narrow ? 64 : 128;
    const int64_t tiles = ceil_div(p->Mrows, tile) * ceil_div(p->Ncols, tile);
    const int64_t Ktotal = (int64_t)g.OW * g.OH * g.N;
    // as many slices as keep every workgroup resident at once (two per compute unit): one more
    // would add a whole round for a single straggler.  The groups of the padded kernel run one after the other and fill the
    // chip each (28 x 28 x 96 x 8 fp32, depthwise 5 x 5: 115 us per group with the slices of a 96th of the chip)
    int64_t want = std::max<int64_t>(1, 2 * (int64_t)std::max(1, num_cus()) / (tiles * (any ? 1 : g.groups)));
    int64_t ks = ceil_div(ceil_div(Ktotal, want), BK) * BK;
    ks = std::max<int64_t>(ks, 4 * BK);
    p->kslice = (int)ks;
    p->slices = (int)ceil_div(Ktotal, ks);
    LUX_UNSUPPORTED_IF(p->slices > 65535, "conv wgrad: too many k slices");
    LUX_UNSUPPORTED_IF((int64_t)p->Mrows * p->Ncols >= (int64_t(1) << 31), "conv wgrad: filter of 2^31 or more elements");
    return LUXHIP_OK;
}

// The filter gradient with the tile's input window in LDS (bf16, 3 x 3, unit stride and dilation, output as large
// as the input): one partial sum per image.  Pointer alignment is checked again at the launch.
template <typename T>
static bool wgrad_window_shape(const ConvGeom& g) {
    if (sizeof(T) != 2 || option_conv_tile() > 2) return false;
    if (g.kW != 3 || g.kH != 3 || g.sw != 1 || g.sh != 1 || g.dw != 1 || g.dh != 1 || g.OW != g.W || g.OH != g.H) return false;
    wpatch::Problem p;
    p.src = nullptr; p.dz = nullptr; p.partial = nullptr; p.zero = nullptr;
    p.Ctot = g.Cin; p.Cg = g.Cin_g; p.Cout = g.Cout; p.Ncols = g.Cout_g; p.P = g.W; p.Q = g.H; p.N = g.N; p.pad_w = g.pw; p.pad_h = g.ph;
    return wpatch::applicable(p, num_cus() > 0 ? num_cus() : 256);
}

// bf16 fast path of the filter gradient: conditions under which conv_wgrad_direct_kernel applies
template <typename T>
static bool wgrad_direct_ok(const ConvGeom& g, const void* xT, const void* dy) {
    if (sizeof(T) != 2) return false;
    const int64_t PQ = (int64_t)g.OW * g.OH;
    return PQ % GemmTraits<T>::BK == 0 && g.Cin_g % 8 == 0 && g.Cin % 8 == 0 && aligned16(xT) && aligned16(dy) &&
           (int64_t)g.W * g.H * g.Cin * g.N < (int64_t(1) << 30) && PQ * g.Cout * g.N < (int64_t(1) << 30);
}

template <typename T>
static size_t wgrad_partial_bytes(const ConvGeom& g) {
    size_t bytes = 0;
    for (int any = 0; any < 3; ++any) {
        WgradPlan p;
        if (wgrad_plan<T>(g, any != 0, any == 2 ? runs_of<T>(g) : Runs(), &p) != LUXHIP_OK) continue;      // run_wgrad refuses it if it is the one
        if (wgrad_window_shape<T>(g))
            p.slices = std::max(p.slices, wpatch::image_lanes(g.N, (g.Cin_g / 64) * ((g.Cout_g + 63) / 64), num_cus() > 0 ? num_cus() : 256));
        bytes = std::max(bytes, (size_t)p.slices * p.Mrows * p.Ncols * sizeof(float));
    }
    return align256(bytes);
}

// runs: xT is the copy of runs_copy_pack.  dy: WHCN cotangent (used by the window and the direct bf16 kernels; null: not there); dyT: its channel-contiguous copy with padded channels,
// followed by BK positions of zeros where there are fewer than BK positions in all (used by the general kernel).  Where
// channels are padded, xT / dyT hold the groups `gr` alone, else all of them.
template <typename T>
static int run_wgrad(hipStream_t s, const ConvGeom& g, Groups gr, Runs runs, const T* xT, const T* dy, const T* dyT, float* partial, T* dw,
                     const void* zeros, const BiasPartials* bias = nullptr) {
    const bool direct = dy != nullptr && wgrad_direct_ok<T>(g, xT, dy);
    const bool window = dy != nullptr && wgrad_window_shape<T>(g) && aligned16(xT) && aligned16(dy) && aligned16(partial);
    WgradPlan plan;
    int rc = wgrad_plan<T>(g, !direct && !window, runs, &plan);
    if (rc != LUXHIP_OK) return rc;
    int slices = plan.slices;
    const int kslice = plan.kslice;
    for (int grp = gr.first; grp < gr.first + gr.n; ++grp) {
        const int Mrows = plan.Mrows;
        if (window) {
            if constexpr (sizeof(T) == 2) {
                wpatch::Problem p;
                p.src = reinterpret_cast<const bf16_t*>(xT) + (size_t)grp * g.Cin_g;
                p.dz = reinterpret_cast<const bf16_t*>(dy) + (size_t)grp * g.Cout_g * g.OW * g.OH;
                p.partial = partial; p.zero = zeros;
                p.Ctot = g.Cin; p.Cg = g.Cin_g; p.Cout = g.Cout; p.Ncols = g.Cout_g;
                p.P = g.W; p.Q = g.H; p.N = g.N; p.pad_w = g.pw; p.pad_h = g.ph;
                rc = wpatch::launch(s, p);
                slices = wpatch::image_lanes(g.N, (g.Cin_g / 64) * ((g.Cout_g + 63) / 64), num_cus() > 0 ? num_cus() : 256);
            }
        } else if (direct) {
            if constexpr (sizeof(T) == 2) {
                ConvWgradDirectArgs a;
                WgradGeomA& q = a.A;
                q.src = reinterpret_cast<const bf16_t*>(xT) + (size_t)grp * g.Cin_g;
                q.zero = zeros;
                q.Ctot = g.Cin; q.Cg = g.Cin_g; q.Mrows = Mrows;
                q.OW = g.OW; q.OWOH = g.OW * g.OH; q.SP = g.W; q.SQ = g.H;
                q.kW = g.kW; q.sw = g.sw; q.sh = g.sh; q.pw = g.pw; q.ph = g.ph; q.dw = g.dw; q.dh = g.dh;
                q.divOW = FastDiv((uint32_t)q.OW); q.divOWOH = FastDiv((uint32_t)q.OWOH);
                q.divCg = FastDiv((uint32_t)q.Cg); q.divkW = FastDiv((uint32_t)g.kW);
                WgradGeomB& b = a.B;
                b.dy = reinterpret_cast<const bf16_t*>(dy);
                b.zero = zeros;
                b.PQ = g.OW * g.OH; b.Cout = g.Cout; b.co_off = grp * g.Cout_g; b.Ncols = g.Cout_g;
                b.divPQ = FastDiv((uint32_t)b.PQ);
                a.Ktotal = g.OW * g.OH * g.N; a.kslice = kslice; a.partial = partial;
                rc = launch_conv_wgrad_direct(s, a, slices);
            }
        } else {
            cany::WgradArgs<T> a;
            const int Cp = padded<T>(g.Cin_g);
            const bool x_alone = Cp != g.Cin_g, y_alone = plan.Ncols != g.Cout_g;
            a.src = xT + (size_t)(x_alone ? grp - gr.first : grp) * Cp; a.Ctot = (x_alone ? gr.n : g.groups) * Cp; a.Cp = Cp; a.Mrows = Mrows;
            a.dyT = dyT + (size_t)(y_alone ? grp - gr.first : grp) * plan.Ncols; a.Ytot = (y_alone ? gr.n : g.groups) * plan.Ncols; a.Ncols = plan.Ncols;
            a.zero = zeros;
            a.OW = g.OW; a.OWOH = g.OW * g.OH; a.SP = g.W; a.SQ = g.H;
            a.kW = g.kW; a.sw = g.sw; a.sh = g.sh; a.pw = g.pw; a.ph = g.ph; a.dw = g.dw; a.dh = g.dh;
            a.divOW = FastDiv((uint32_t)a.OW); a.divOWOH = FastDiv((uint32_t)a.OWOH); a.divCp = FastDiv((uint32_t)Cp); a.divkW = FastDiv((uint32_t)g.kW);
            if (runs.W2 > 0) {                                 // xT holds runs of positions
                a.Ctot = 4; a.Cp = Runs::EL; a.divCp = FastDiv((uint32_t)Runs::EL); a.kW = 1; a.divkW = FastDiv(1); a.pw = 0; a.SP = runs.W2;
            }
            a.positions = g.OW * g.OH * g.N;
            a.Ktotal = std::max(a.positions, GemmTraits<T>::BK);
            a.kslice = kslice; a.partial = partial;
            rc = cany::launch_any_wgrad<T>(s, a, slices, plan.narrow);
        }
        if (rc != LUXHIP_OK) return rc;
        ProfScope ps("wgrad_reduce_kernel", s);
        const int total = Mrows * g.Cout_g;
        // parts of at least four slices, as many as give every compute unit a workgroup: beyond that they cost (36864 threads in one part 8.4 us, in two 9.8)
        int parts = 1;
        while (parts < 64 && (int64_t)total / 4 * parts * 2 <= 256 * (int64_t)std::max(1, num_cus()) && parts * 8 <= slices) parts *= 2;
        const int reduce_blocks = (int)ceil_div(ceil_div(total, 4), 256 / parts);
        BiasPartials bp;
        if (bias != nullptr && grp == g.groups - 1) bp = *bias;       // the bias gradient's channels ride on the last group's launch
        wgrad_reduce_kernel<T><<<(unsigned)(reduce_blocks + bp.C), 256, 0, s>>>(partial, dw, g, grp, slices, parts, reduce_blocks, Mrows,
                                                                           runs.W2 > 0 ? 4 : Mrows / (g.kW * g.kH), runs.W2 > 0 ? Runs::EL : 0,
                                                                           (int64_t)Mrows * plan.Ncols, bp);
        LUX_CHECK_LAUNCH();
    }
    return LUXHIP_OK;
}

// ----------------------------------------------------------------------------- typed entry points
// Positions of zeros that follow the channel-contiguous cotangent: the filter gradient contracts at least one stage
template <typename T>
static int dy_zeros(const ConvGeom& g) {
    const int64_t pos = (int64_t)g.OW * g.OH * g.N;
    return pos < GemmTraits<T>::BK ? GemmTraits<T>::BK : 0;
}
// Bytes of the padded channel-contiguous copies and of the packed filter (either form)
template <typename T>
static size_t xt_bytes(const ConvGeom& g, int n) {       // n: groups at a time, where padded
    const int Cp = padded<T>(g.Cin_g);
    const size_t runs = (size_t)runs_of<T>(g).W2 * g.H * g.N * 4 * sizeof(T);      // either form
    return align256(std::max(runs, (size_t)g.W * g.H * g.N * (Cp != g.Cin_g ? n : g.groups) * Cp * sizeof(T)));
}
template <typename T>
static size_t dyt_bytes(const ConvGeom& g, int n) {
    const int Cp = padded<T>(g.Cout_g);
    return align256(((size_t)g.OW * g.OH * g.N + dy_zeros<T>(g)) * (Cp != g.Cout_g ? n : g.groups) * Cp * sizeof(T));
}
template <typename T>
static size_t filter_bytes(const ConvGeom& g, bool any, const AnyPlan<T>& plan) {
    return align256(any ? (size_t)plan.wm_elems * g.groups * sizeof(T) : (size_t)g.kW * g.kH * g.Cin_g * g.Cout * sizeof(T));
}
// A caller's channel-contiguous copy of x serves the kernels as it is
template <typename T>
static bool kept_usable(const ConvGeom& g, const T* kept) { return kept != nullptr && padded<T>(g.Cin_g) == g.Cin_g && aligned16(kept); }

// (C, P) -> (Cp, P) per group with zeros in the new channels, for the groups whose first channel is at `in` (Cin channels in a
// row): a caller's unpadded copy of x, when x itself is not given
template <typename T>
__global__ __launch_bounds__(256) void repad_cwhn_kernel(const T* __restrict__ in, T* __restrict__ out, int64_t total, int Cin, int Cg, int groups, int Cp) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
        const int64_t row = i / Cp, pos = row / groups;
        const int c = (int)(i - row * Cp), grp = (int)(row - pos * groups);
        out[i] = c < Cg ? in[pos * Cin + grp * Cg + c] : T(0);
    }
}

template <typename T>
static int conv_fwd_t(hipStream_t s, int act, const ConvGeom& g, const T* x, const T* w, const T* bias, T* y, T* pre,
                      T* xt_keep) {
    const bool any = !tap_shape<T>(g, false);
    AnyPlan<T> plan(g, false);
    // xt_keep: caller's buffer of x's size that keeps the channel-contiguous copy of x for the pullback
    const bool keep = kept_usable<T>(g, xt_keep);
    const int n = keep ? std::min(g.groups, 32768) : groups_at_a_time<T>(g, true, false);
    const size_t xb = keep ? 0 : xt_bytes<T>(g, n), wb = filter_bytes<T>(g, any, plan);
    Workspace ws;
    // the slices of conv_any.h take memory behind these; reserve it here, where no pointer into the workspace is live yet
    int rc = get_workspace(s, any ? plan.reserve(s, xb + wb, n, g.groups) : xb + wb, &ws);
    if (rc != LUXHIP_OK) return rc;
    T* xT = keep ? xt_keep : reinterpret_cast<T*>(ws.data);
    T* wF = reinterpret_cast<T*>(ws.data + xb);
    if (xt_keep != nullptr && !keep) {
        if ((rc = transpose_to_cwhn<T>(s, x, xt_keep, g.W * g.H, g.Cin, g.N)) != LUXHIP_OK) return rc;
    }
    if (!any) {
        if ((rc = transpose_and_pack<T>(s, x, xT, g.W * g.H, g.Cin, g.N, w, wF, g, 0)) != LUXHIP_OK) return rc;
        return run_conv_gemm<T>(s, g, false, xT, wF, bias, y, pre, act, ws.zeros);
    }
    const PackSubs ps = plan.pack(g, false, 0);
    for (Groups gr{0, 0}; gr.first < g.groups; gr.first += gr.n) {
        gr.n = std::min(n, g.groups - gr.first);
        const bool first = gr.first == 0;
        if (plan.Cp != g.Cin_g || first) {
            const int copied = plan.Cp != g.Cin_g ? gr.n : g.groups;
            if constexpr (sizeof(T) == 2) {
                if (plan.runs.W2 > 0) {
                    if ((rc = runs_copy_pack(s, g, plan.runs, x, xT, w, wF)) != LUXHIP_OK) return rc;
                }
            }
            if (plan.runs.W2 == 0)
                rc = pad_and_pack<T>(s, x + (size_t)gr.first * g.Cin_g * g.W * g.H, xT, g.W * g.H, g.Cin, g.Cin_g, copied, g.N, 0, w, first ? wF : nullptr, g, &ps);
            if (rc != LUXHIP_OK) return rc;
        }
        if ((rc = run_conv_any<T>(s, g, false, plan, gr, xT, w, wF, true, bias, y, pre, act, xb + wb)) != LUXHIP_OK) return rc;
    }
    return LUXHIP_OK;
}

// dx of the groups `gr` from the channel-contiguous cotangent; packed: the filter of the first launch is in wD.  The whole-tap
// kernels (no padding: one call for all groups) know no part of the groups.
template <typename T>
static int run_dgrad(hipStream_t s, const ConvGeom& g, bool any, const AnyPlan<T>& plan, Groups gr, const T* dyT, const T* w, T* wD, bool packed, T* dx,
                     size_t ws_front, const void* zeros) {
    if (any) return run_conv_any<T>(s, g, true, plan, gr, dyT, w, wD, packed, nullptr, dx, nullptr, LUXHIP_ACT_IDENTITY, ws_front);
    return gr.first == 0 ? run_conv_gemm<T>(s, g, true, dyT, wD, nullptr, dx, nullptr, LUXHIP_ACT_IDENTITY, zeros) : LUXHIP_OK;
}
// dyT of the groups `gr` (of all groups with the first ones, where nothing is padded)
template <typename T>
static int dy_copy(hipStream_t s, const ConvGeom& g, Groups gr, const T* dy, T* dyT) {
    const bool alone = padded<T>(g.Cout_g) != g.Cout_g;
    if (!alone && gr.first > 0) return LUXHIP_OK;
    return to_cwhn_padded<T>(s, dy + (size_t)gr.first * g.Cout_g * g.OW * g.OH, dyT, g.OW * g.OH, g.Cout, g.Cout_g, alone ? gr.n : g.groups, g.N,
                             dy_zeros<T>(g), g);
}
// The same, and with the first groups the filter packed for the input gradient, in one launch
template <typename T>
static int dy_copy_and_pack(hipStream_t s, const ConvGeom& g, bool any, const AnyPlan<T>& plan, Groups gr, const T* dy, T* dyT, const T* w, T* wD) {
    if (gr.first > 0 || plan.launches.empty()) return dy_copy<T>(s, g, gr, dy, dyT);
    if (!any && dy_zeros<T>(g) > 0) {
        const int rc = dy_copy<T>(s, g, gr, dy, dyT);
        return rc != LUXHIP_OK ? rc : pack_filter<T>(s, w, wD, g, 1);
    }
    if (!any) return transpose_and_pack<T>(s, dy, dyT, g.OW * g.OH, g.Cout, g.N, w, wD, g, 1);
    const PackSubs ps = plan.pack(g, true, 0);
    return pad_and_pack<T>(s, dy, dyT, g.OW * g.OH, g.Cout, g.Cout_g, plan.Cp != g.Cout_g ? gr.n : g.groups, g.N, dy_zeros<T>(g), w, wD, g, &ps);
}
// xT of the groups `gr`, likewise; from the caller's unpadded copy where x is not given
template <typename T>
static int x_copy(hipStream_t s, const ConvGeom& g, Groups gr, Runs runs, const T* x, const T* unpadded, T* xT) {
    if constexpr (sizeof(T) == 2) {
        if (runs.W2 > 0) return runs_copy_pack(s, g, runs, x, xT, nullptr, nullptr);
    }
    const int Cp = padded<T>(g.Cin_g);
    const bool alone = Cp != g.Cin_g;
    if (!alone && gr.first > 0) return LUXHIP_OK;
    const int n = alone ? gr.n : g.groups;
    if (x != nullptr)
        return to_cwhn_padded<T>(s, x + (size_t)gr.first * g.Cin_g * g.W * g.H, xT, g.W * g.H, g.Cin, g.Cin_g, n, g.N, 0, g);
    const int64_t total = (int64_t)g.W * g.H * g.N * n * Cp;
    repad_cwhn_kernel<T><<<(unsigned)std::min<int64_t>(ceil_div(total, 256), 65536), 256, 0, s>>>(unpadded + (size_t)gr.first * g.Cin_g, xT, total, g.Cin,
                                                                                               g.Cin_g, n, Cp);
    LUX_CHECK_LAUNCH();
    return LUXHIP_OK;
}

template <typename T>
static int conv_bwd_data_t(hipStream_t s, const ConvGeom& g, const T* dy, const T* w, T* dx) {
    const bool any = !tap_shape<T>(g, true);
    AnyPlan<T> plan(g, true);
    const int n = groups_at_a_time<T>(g, false, true);
    const size_t yb = dyt_bytes<T>(g, n), wb = filter_bytes<T>(g, any, plan);
    Workspace ws;
    int rc = get_workspace(s, any ? plan.reserve(s, yb + wb, n, g.groups) : yb + wb, &ws);
    if (rc != LUXHIP_OK) return rc;
    T* dyT = reinterpret_cast<T*>(ws.data);
    T* wD = reinterpret_cast<T*>(ws.data + yb);
    for (Groups gr{0, 0}; gr.first < g.groups; gr.first += gr.n) {
        gr.n = std::min(n, g.groups - gr.first);
        if ((rc = dy_copy_and_pack<T>(s, g, any, plan, gr, dy, dyT, w, wD)) != LUXHIP_OK) return rc;
        if ((rc = run_dgrad<T>(s, g, any, plan, gr, dyT, w, wD, true, dx, yb + wb, ws.zeros)) != LUXHIP_OK) return rc;
    }
    return LUXHIP_OK;
}

template <typename T>
static int conv_bwd_filter_t(hipStream_t s, const ConvGeom& g, const T* x, const T* dy, T* dw) {
    const int n = groups_at_a_time<T>(g, true, true);
    const size_t xb = xt_bytes<T>(g, n), yb = dyt_bytes<T>(g, n), pb = wgrad_partial_bytes<T>(g);
    Workspace ws;
    int rc = get_workspace(s, xb + yb + pb, &ws);
    if (rc != LUXHIP_OK) return rc;
    T* xT = reinterpret_cast<T*>(ws.data);
    T* dyT = reinterpret_cast<T*>(ws.data + xb);
    float* partial = reinterpret_cast<float*>(ws.data + xb + yb);
    const Runs runs = runs_of<T>(g);
    for (Groups gr{0, 0}; gr.first < g.groups; gr.first += gr.n) {
        gr.n = std::min(n, g.groups - gr.first);
        if ((rc = x_copy<T>(s, g, gr, runs, x, nullptr, xT)) != LUXHIP_OK) return rc;
        // the direct kernel reads dy as it is
        if (!wgrad_direct_ok<T>(g, xT, dy) && (rc = dy_copy<T>(s, g, gr, dy, dyT)) != LUXHIP_OK) return rc;
        if ((rc = run_wgrad<T>(s, g, gr, runs, xT, dy, dyT, partial, dw, ws.zeros)) != LUXHIP_OK) return rc;
    }
    return LUXHIP_OK;
}

template <typename T>
static int fused_conv_bwd_t(hipStream_t s, int dtype, int act, const ConvGeom& g, const T* delta, const T* y,
                            const T* pre, const T* x, const T* w, T* dz, T* dw, T* dx, T* dbias, const T* xt_kept) {
    const bool any = !tap_shape<T>(g, true), kept = kept_usable<T>(g, xt_kept);
    AnyPlan<T> plan(g, true);
    const int n = groups_at_a_time<T>(g, dw != nullptr && !kept, true);
    const size_t xb = kept ? 0 : xt_bytes<T>(g, n), yb = dyt_bytes<T>(g, n), wb = filter_bytes<T>(g, any, plan), pb = wgrad_partial_bytes<T>(g);
    // dz channel-contiguous, the bias gradient and, where the filter gradient reads it, dz as it lies in one pass, when both a pass over
    // delta and a transposing copy would run
    const int Cp = padded<T>(g.Cout_g);
    const bool one_pass = (act != LUXHIP_ACT_IDENTITY || dbias != nullptr) && (dw != nullptr || dx != nullptr) &&
                          (Cp == g.Cout_g || g.groups == 1) && dy_zeros<T>(g) == 0 && dz_cwhn_ok<T>(g.OW * g.OH, g.Cout, g.N);
    const size_t bb = one_pass && dbias != nullptr ? dz_cwhn_partial_bytes(g.OW * g.OH, g.Cout, g.N) : 0;
    // reserve everything up front: the bias-gradient pass below uses the start of the same
    // workspace, and the buffer must not be reallocated while pointers into it are live
    Workspace ws;
    int rc = get_workspace(s, any && dx != nullptr ? plan.reserve(s, xb + yb + wb + pb + bb, n, g.groups) : xb + yb + wb + pb + bb, &ws);
    if (rc != LUXHIP_OK) return rc;
    const T* xT = kept ? xt_kept : reinterpret_cast<const T*>(ws.data);
    T* dzT = reinterpret_cast<T*>(ws.data + xb);
    T* wD = reinterpret_cast<T*>(ws.data + xb + yb);
    float* partial = reinterpret_cast<float*>(ws.data + xb + yb + wb);
    const T* dzp = delta;
    bool packed = dx != nullptr;          // the filter is in wD when the input gradient starts
    BiasPartials bias_later;              // set by the single pass when the filter gradient's reduction will finish the bias gradient
    if (one_pass) {
        const bool lies = dw != nullptr && (wgrad_direct_ok<T>(g, xT, dz) || (wgrad_window_shape<T>(g) && aligned16(xT) && aligned16(dz)));
        T* const dz_out = act != LUXHIP_ACT_IDENTITY && lies ? dz : nullptr;
        packed = packed && !(any && plan.launches.empty());
        PackSubs ps;
        if (packed && any) ps = plan.pack(g, true, 0);
        rc = conv_dz_cwhn_pack<T>(s, act, g, g.groups == 1 ? Cp : g.Cout, delta, y, pre, dz_out, dzT, reinterpret_cast<float*>(ws.data + xb + yb + wb + pb), dbias, w,
                                  packed ? wD : nullptr, packed && any ? &ps : nullptr, dw != nullptr ? &bias_later : nullptr);
        if (rc != LUXHIP_OK) return rc;
        if (act != LUXHIP_ACT_IDENTITY) dzp = dz_out;             // null: only the channel-contiguous one is there
    } else {
        if (act != LUXHIP_ACT_IDENTITY || dbias != nullptr) {
            T* dz_out = act == LUXHIP_ACT_IDENTITY ? nullptr : dz;
            rc = bias_act_bwd_dispatch(s, dtype, act, (int64_t)g.OW * g.OH, g.Cout, g.N, delta, y, pre, dz_out, dbias);
            if (rc != LUXHIP_OK) return rc;
            if (dz_out) dzp = dz_out;
        }
        if (dw == nullptr && dx == nullptr) return LUXHIP_OK;
    }
    for (Groups gr{0, 0}; gr.first < g.groups; gr.first += gr.n) {
        gr.n = std::min(n, g.groups - gr.first);
        if (!one_pass) {
            rc = dx != nullptr ? dy_copy_and_pack<T>(s, g, any, plan, gr, dzp, dzT, w, wD) : dy_copy<T>(s, g, gr, dzp, dzT);
            if (rc != LUXHIP_OK) return rc;
        }
        if (dx != nullptr) {
            if ((rc = run_dgrad<T>(s, g, any, plan, gr, dzT, w, wD, packed, dx, xb + yb + wb + pb + bb, ws.zeros)) != LUXHIP_OK) return rc;
        }
        if (dw != nullptr) {
            const Runs runs = !kept && x != nullptr ? runs_of<T>(g) : Runs();
            if (!kept && (rc = x_copy<T>(s, g, gr, runs, x, xt_kept, reinterpret_cast<T*>(ws.data))) != LUXHIP_OK) return rc;
            rc = run_wgrad<T>(s, g, gr, runs, xT, dzp, dzT, partial, dw, ws.zeros, bias_later.dbias != nullptr ? &bias_later : nullptr);
            if (rc != LUXHIP_OK) return rc;
        }
    }
    return LUXHIP_OK;
}

static int conv_check(int dtype, int act) {
    LUX_UNSUPPORTED_IF(dtype != LUXHIP_F32 && dtype != LUXHIP_BF16, "unsupported dtype %d", dtype);
    LUX_UNSUPPORTED_IF(act < 0 || act >= LUXHIP_ACT_COUNT, "unsupported activation id %d", act);
    return LUXHIP_OK;
}

}  // namespace luxhip

using namespace luxhip;

extern "C" {

int luxhip_conv_fwd(luxhip_stream_t s, int dtype, int act, const luxhip_conv_dims_t* d, const void* x, const void* w,
                    const void* bias, void* y, void* pre, void* xt_keep) {
    LUX_REQUIRE_INIT();
    int rc = conv_check(dtype, act);
    if (rc != LUXHIP_OK) return rc;
    ConvGeom g;
    if ((rc = make_geom(d, &g)) != LUXHIP_OK) return rc;
    if (g.N == 0) return LUXHIP_OK;
    LUX_INVALID_IF(x == nullptr || w == nullptr || y == nullptr, "conv_fwd: x, w and y must not be NULL");
    if (dtype == LUXHIP_F32)
        return conv_fwd_t<float>((hipStream_t)s, act, g, (const float*)x, (const float*)w, (const float*)bias, (float*)y, (float*)pre,
                                 (float*)xt_keep);
    return conv_fwd_t<bf16_t>((hipStream_t)s, act, g, (const bf16_t*)x, (const bf16_t*)w, (const bf16_t*)bias, (bf16_t*)y, (bf16_t*)pre,
                              (bf16_t*)xt_keep);
}

int luxhip_conv_bwd_data(luxhip_stream_t s, int dtype, const luxhip_conv_dims_t* d, const void* dy, const void* w, void* dx) {
    LUX_REQUIRE_INIT();
    int rc = conv_check(dtype, 0);
    if (rc != LUXHIP_OK) return rc;
    ConvGeom g;
    if ((rc = make_geom(d, &g)) != LUXHIP_OK) return rc;
    if (g.N == 0) return LUXHIP_OK;
    LUX_INVALID_IF(dy == nullptr || w == nullptr || dx == nullptr, "conv_bwd_data: dy, w and dx must not be NULL");
    if (dtype == LUXHIP_F32) return conv_bwd_data_t<float>((hipStream_t)s, g, (const float*)dy, (const float*)w, (float*)dx);
    return conv_bwd_data_t<bf16_t>((hipStream_t)s, g, (const bf16_t*)dy, (const bf16_t*)w, (bf16_t*)dx);
}

int luxhip_conv_bwd_filter(luxhip_stream_t s, int dtype, const luxhip_conv_dims_t* d, const void* x, const void* dy, void* dw) {
    LUX_REQUIRE_INIT();
    int rc = conv_check(dtype, 0);
    if (rc != LUXHIP_OK) return rc;
    ConvGeom g;
    if ((rc = make_geom(d, &g)) != LUXHIP_OK) return rc;
    LUX_INVALID_IF(dw == nullptr, "conv_bwd_filter: dw must not be NULL");
    if (g.N == 0) return luxhip_fill_zero(dw, (size_t)g.kW * g.kH * g.Cin_g * g.Cout * (dtype == LUXHIP_F32 ? 4 : 2), s);
    LUX_INVALID_IF(x == nullptr || dy == nullptr, "conv_bwd_filter: x and dy must not be NULL");
    if (dtype == LUXHIP_F32) return conv_bwd_filter_t<float>((hipStream_t)s, g, (const float*)x, (const float*)dy, (float*)dw);
    return conv_bwd_filter_t<bf16_t>((hipStream_t)s, g, (const bf16_t*)x, (const bf16_t*)dy, (bf16_t*)dw);
}

int luxhip_fused_conv_bwd(luxhip_stream_t s, int dtype, int act, const luxhip_conv_dims_t* d, const void* delta,
                          const void* y, const void* pre, const void* x, const void* w, void* dz, void* dw, void* dx,
                          void* dbias, const void* xt_kept) {
    LUX_REQUIRE_INIT();
    int rc = conv_check(dtype, act);
    if (rc != LUXHIP_OK) return rc;
    ConvGeom g;
    if ((rc = make_geom(d, &g)) != LUXHIP_OK) return rc;
    const size_t esz = dtype == LUXHIP_F32 ? 4 : 2;
    if (g.N == 0) {
        if (dw) { rc = luxhip_fill_zero(dw, (size_t)g.kW * g.kH * g.Cin_g * g.Cout * esz, s); if (rc) return rc; }
        if (dbias) { rc = luxhip_fill_zero(dbias, (size_t)g.Cout * esz, s); if (rc) return rc; }
        return LUXHIP_OK;
    }
    LUX_INVALID_IF(delta == nullptr, "fused_conv_bwd: delta must not be NULL");
    LUX_INVALID_IF(act != LUXHIP_ACT_IDENTITY && dz == nullptr, "fused_conv_bwd: dz scratch is required");
    LUX_INVALID_IF(act != LUXHIP_ACT_IDENTITY && !act_needs_pre(act) && y == nullptr, "fused_conv_bwd: activation %d needs y", act);
    LUX_INVALID_IF(act_needs_pre(act) && pre == nullptr, "fused_conv_bwd: activation %d needs the pre-activation", act);
    LUX_INVALID_IF((dw != nullptr && x == nullptr && xt_kept == nullptr) || (dx != nullptr && w == nullptr), "fused_conv_bwd: x / w must not be NULL");
    if (dtype == LUXHIP_F32)
        return fused_conv_bwd_t<float>((hipStream_t)s, dtype, act, g, (const float*)delta, (const float*)y, (const float*)pre,
                                       (const float*)x, (const float*)w, (float*)dz, (float*)dw, (float*)dx, (float*)dbias,
                                       (const float*)xt_kept);
    return fused_conv_bwd_t<bf16_t>((hipStream_t)s, dtype, act, g, (const bf16_t*)delta, (const bf16_t*)y, (const bf16_t*)pre,
                                    (const bf16_t*)x, (const bf16_t*)w, (bf16_t*)dz, (bf16_t*)dw, (bf16_t*)dx, (bf16_t*)dbias,
                                    (const bf16_t*)xt_kept);
}

}  // extern "C"
