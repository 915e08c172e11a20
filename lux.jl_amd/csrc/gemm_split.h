// MFMA products for the sizes and alignments that leave the big-tile kernels idle: few tiles (the contraction is split
// over workgroups), leading dimensions or pointers that are no multiple of 16 bytes, dimensions below a tile.
//
// What bounds these problems is latency, not rate: a 64 x 64 tile over K = 1000 alone takes 16 dependent stages, and
// the chip has 256 compute units for a handful of tiles.  Three things follow.
//   * Loads are 16 bytes wide whatever the alignment (the hardware takes global addresses aligned to the element), so a
//     ragged operand costs the same instructions as an aligned one.  Nothing outside the operand is touched: a tile that
//     would stick out of the matrix is moved back until it ends with it (its overlap is computed twice, with the same
//     result), the last stage of the contraction is moved back likewise and what it repeats is set to zero in both
//     operands.  A dimension smaller than the tile clamps its rows instead and checks the stores.
//   * A workgroup loads U stages (64 or 128 k) at once, which is one trip to memory, one barrier and U stages of MFMAs,
//     instead of a trip and a barrier per stage; the next U stages are requested before the MFMAs start.
//   * The contraction of a tile is cut into S slices.  Every slice hands its fp32 accumulators over through device
//     memory; the workgroup that arrives last adds them in slice order (the same sum on every run) and runs the epilogue.
// Measured (one launch; the bounds-checked kernels of gemm_dense.h before): fp32 517 x 301 x 1023 116 -> 13 us, 1023 x 301 x
// 517 69 -> 11, 704 x 1329 x 2176 191 -> 48 (85 TFLOP/s); bf16 517 x 301 x 1023 93 -> 8.5 us, 3651 x 2048 x 1350 160 -> 36
// (560 TFLOP/s), 1350 x 2048 x 3651 362 -> 64.
#pragma once

#include "common.h"
#include "gemm_core.h"
#include "gemm_dense.h"

namespace luxhip {
namespace split {

constexpr int THREADS = 256;

// One stage (BK of k) of an operand tile of ROWS rows in registers, rows r0 .. r0 + ROWS - 1 (r0 + ROWS <= rows, or
// r0 = 0 and rows < ROWS: `bounded`).
template <typename T, bool KMAJOR_, int ROWS>
struct Loader {
    static constexpr bool KMAJOR = KMAJOR_;
    using Tr = GemmTraits<T>;
    static constexpr int CHUNKS = ROWS * Tr::BK / Tr::VEC;
    static constexpr int PER = CHUNKS > THREADS ? CHUNKS / THREADS : 1;
    static_assert(CHUNKS % THREADS == 0 || THREADS % CHUNKS == 0, "a stage splits evenly over the workgroup");
    static constexpr int CPR = KMAJOR ? Tr::BK / Tr::VEC : ROWS / Tr::VEC;      // chunks per LDS row
    const char* base;          // uniform: element (r0, k = 0)
    int64_t k_bytes;           // uniform
    uint32_t voff[PER];        // per thread
    int sh[PER];               // MN-major, bounded: elements that the chunk at the end of the rows is moved by
    bool bounded;              // uniform
    __device__ __forceinline__ static void coords(int i, int& r, int& k) {
        const int id = CHUNKS < THREADS ? (int)threadIdx.x % CHUNKS : (int)threadIdx.x + i * THREADS;   // fewer chunks than threads: doubly
        if constexpr (KMAJOR) { r = id / CPR; k = (id % CPR) * Tr::VEC; }
        else { k = id / CPR; r = (id % CPR) * Tr::VEC; }
    }
    // back: an MN-major operand of fewer rows than a chunk (the end of a larger one) is read from `back` elements before its first row on, VEC - rows
    __device__ __forceinline__ Loader(const Operand<T>& op, int r0, int back = 0) {
        base = reinterpret_cast<const char*>(op.p + (KMAJOR ? (int64_t)r0 * op.sr : (int64_t)r0 - back));
        k_bytes = KMAJOR ? (int64_t)sizeof(T) : op.sk * (int64_t)sizeof(T);
        bounded = op.rows < ROWS;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            int r, k;
            coords(i, r, k);
            sh[i] = 0;
            if (bounded) {
                if constexpr (KMAJOR) {
                    r = min(r, op.rows - 1);
                } else if (r + Tr::VEC > op.rows) {
                    sh[i] = r + Tr::VEC - op.rows;
                    r = op.rows - Tr::VEC + back;
                }
            }
            voff[i] = (uint32_t)(((int64_t)r * op.sr + (int64_t)k * op.sk) * (int64_t)sizeof(T));
        }
    }
    __device__ __forceinline__ void load(int k, u32x4_v (&reg)[PER]) const {
        const char* p = base + k * k_bytes;
#pragma unroll
        for (int i = 0; i < PER; ++i)
            reg[i] = *reinterpret_cast<const typename UnalignedVec<T>::type*>(p + voff[i]);
    }
    // skip: leading k of the stage that are to count as zero
    template <bool SPLIT>
    __device__ __forceinline__ void store(u32x4_v (&reg)[PER], T* lds, int skip) const {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            int r, k;
            coords(i, r, k);
            u32x4_v v = reg[i];
            if constexpr (!KMAJOR) {
                if (bounded && sh[i] > 0) {                     // element e of the chunk is element e + sh of what was loaded
                    const uint64_t lo = ((uint64_t)v[1] << 32) | v[0], hi = ((uint64_t)v[3] << 32) | v[2];
                    const int bits = min(sh[i] * (int)sizeof(T) * 8, 127);
                    const uint64_t a = bits < 64 ? (lo >> bits) | (bits ? hi << (64 - bits) : 0ull) : hi >> (bits - 64);
                    const uint64_t b = bits < 64 ? hi >> bits : 0ull;
                    v = u32x4_v{(uint32_t)a, (uint32_t)(a >> 32), (uint32_t)b, (uint32_t)(b >> 32)};
                }
            }
            if (skip > 0) {
                if constexpr (KMAJOR) {
#pragma unroll
                    for (int w = 0; w < 4; ++w) {
                        if constexpr (sizeof(T) == 4) v[w] = k + w < skip ? 0u : v[w];
                        else v[w] &= (k + 2 * w < skip ? 0u : 0xffffu) | (k + 2 * w + 1 < skip ? 0u : 0xffff0000u);
                    }
                } else {
                    if (k < skip) v = u32x4_v{0u, 0u, 0u, 0u};
                }
            }
            put_chunk<T, KMAJOR, ROWS, SPLIT>(lds, r, k, v);
        }
    }
};

struct Plan {
    int slices, kslice;        // kslice: k per slice, a multiple of BK
    float* partial;            // [tile][slice][accumulator pair][thread] float2
    uint32_t* counters;        // one per tile
};

// The main loop over loaders of the two operands: a workgroup of NWM x NWN waves, each with WM x WN accumulators.
template <typename T, int WM, int WN, int NWM, int NWN, class LA, class LB>
struct Core {
    static constexpr bool AK = LA::KMAJOR, BKM = LB::KMAJOR;
    using ML = GemmMainloop<T, WM, WN, AK, BKM, false, NWN, 0, NWM>;
    using Tr = GemmTraits<T>;
    static constexpr int U = LA::PER + LB::PER <= 2 ? 4 : 2;
    static constexpr size_t LDS_BYTES = (size_t)U * ML::STAGE_ELEMS * sizeof(T);
    static_assert(NWM * NWN * 64 == THREADS, "four waves");

    template <bool SPLIT>
    __device__ __forceinline__ static void compute(const T* As, const T* Bs, int wave_m, int wave_n, f32x16_v (&acc)[WM][WN],
                                                   f32x16_v (&small)[WM][WN]) {
        if constexpr (sizeof(T) == 2) {
#pragma unroll
            for (int kk = 0; kk < Tr::BK / 16; ++kk) {
                bf16x8_v fa[WM], fb[WN];
#pragma unroll
                for (int i = 0; i < WM; ++i) fa[i] = load_frag_bf16<AK, ML::TILE_M>(As, wave_m + i * 32, kk);
#pragma unroll
                for (int j = 0; j < WN; ++j) fb[j] = load_frag_bf16<BKM, ML::TILE_N>(Bs, wave_n + j * 32, kk);
#pragma unroll
                for (int i = 0; i < WM; ++i)
#pragma unroll
                    for (int j = 0; j < WN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[j], fa[i], acc[i][j], 0, 0, 0);
            }
        } else {
            mfma_stage_f32<SPLIT, AK, BKM, ML::TILE_M, ML::TILE_N>(As, Bs, wave_m, wave_n, acc, small);
        }
    }

    // k range [kbeg, kend)
    __device__ __forceinline__ static void run(const LA& la, const LB& lb, int kbeg, int kend, T* lds, f32x16_v (&acc)[WM][WN]) {
        if constexpr (ML::SPLIT_F32) {
            if (__syncthreads_and(run_as<true>(la, lb, kbeg, kend, lds, acc))) return;
        }
        run_as<false>(la, lb, kbeg, kend, lds, acc);
    }
    template <bool SPLIT>          // false: see GemmMainloop::run_as
    __device__ __forceinline__ static bool run_as(const LA& la, const LB& lb, int kbeg, int kend, T* lds, f32x16_v (&acc)[WM][WN]) {
        const int w = threadIdx.x >> 6;
        const int wave_m = (w % NWM) * (WM * 32), wave_n = (w / NWM) * (WN * 32);
        ML::zero(acc);
        f32x16_v small[WM][WN];                                 // SPLIT: the smaller partial products
        if constexpr (SPLIT) ML::zero(small);
        u32x4_v ra[U][LA::PER], rb[U][LB::PER];
        int skip[U];
        auto fetch_stages = [&](int k0) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int k = k0 + u * Tr::BK;
                if (k < kend) {
                    const int kk = min(k, kend - Tr::BK);
                    skip[u] = k - kk;
                    la.load(kk, ra[u]);
                    lb.load(kk, rb[u]);
                }
            }
        };
        fetch_stages(kbeg);
        for (int k0 = kbeg; k0 < kend; k0 += U * Tr::BK) {
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (k0 + u * Tr::BK < kend) {
                    la.template store<SPLIT>(ra[u], lds + u * ML::STAGE_ELEMS, skip[u]);
                    lb.template store<SPLIT>(rb[u], lds + u * ML::STAGE_ELEMS + ML::A_ELEMS, skip[u]);
                }
            __syncthreads();
            if (k0 + U * Tr::BK < kend) fetch_stages(k0 + U * Tr::BK);
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (k0 + u * Tr::BK < kend) compute<SPLIT>(lds + u * ML::STAGE_ELEMS, lds + u * ML::STAGE_ELEMS + ML::A_ELEMS, wave_m, wave_n, acc, small);
            __syncthreads();
        }
        if constexpr (SPLIT) return finish_parts(acc, small);
        return true;
    }

    // hand-off of a slice's accumulators; true in the workgroup that holds the sum and runs the epilogue
    __device__ __forceinline__ static bool combine(const Plan& p, int tile, int slice, f32x16_v (&acc)[WM][WN]) {
        __shared__ uint32_t flag;
        constexpr int PAIRS = WM * WN * 8;
        uint64_t* mine = reinterpret_cast<uint64_t*>(p.partial) + ((size_t)tile * p.slices + slice) * (PAIRS * THREADS) + threadIdx.x;
        static_for<PAIRS>([&](auto Q) {
            constexpr int q = decltype(Q)::value, ij = q / 8, r = (q % 8) * 2;
            const uint64_t v = ((uint64_t)__float_as_uint(acc[ij / WN][ij % WN][r + 1]) << 32) | __float_as_uint(acc[ij / WN][ij % WN][r]);
            __hip_atomic_store(mine + q * THREADS, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        });
        publish_done();
        if (!arrive_last(p.counters + tile, (uint32_t)p.slices, &flag)) return false;
        ML::zero(acc);
        const uint64_t* all = reinterpret_cast<const uint64_t*>(p.partial) + (size_t)tile * p.slices * (PAIRS * THREADS) + threadIdx.x;
#pragma unroll WM * WN == 1 ? 4 : 1
        for (int s = 0; s < p.slices; ++s) {
            uint64_t v[PAIRS];
            static_for<PAIRS>([&](auto Q) {
                constexpr int q = decltype(Q)::value;
                v[q] = fetch_tagged(all + (size_t)s * (PAIRS * THREADS) + q * THREADS);
            });
            static_for<PAIRS>([&](auto Q) {
                constexpr int q = decltype(Q)::value, ij = q / 8, r = (q % 8) * 2;
                acc[ij / WN][ij % WN][r] += __uint_as_float((uint32_t)v[q]);
                acc[ij / WN][ij % WN][r + 1] += __uint_as_float((uint32_t)(v[q] >> 32));
            });
        }
        return true;
    }
};

template <typename T, int W, bool AK, bool BKM>
using Body = Core<T, W, W, 2, 2, Loader<T, AK, 64 * W>, Loader<T, BKM, 64 * W>>;

// One (tile, slice) of a product; `id` counts the slices of a tile together.
template <typename T, int W, bool AK, bool BKM, bool PLAIN = false>
__device__ __forceinline__ void tile_slice(const DenseArgs<T>& a, const Plan& p, int id, T* lds) {
    using B = Body<T, W, AK, BKM>;
    using ML = typename B::ML;
    const int tile = id / p.slices, slice = id - tile * p.slices;
    int tm, tn;
    tile_coords(tile, a.tiles_m, a.tiles_n, tm, tn);
    const int m0 = max(min(tm * ML::TILE_M, a.M - ML::TILE_M), 0), n0 = max(min(tn * ML::TILE_N, a.N - ML::TILE_N), 0);
    const int kbeg = slice * p.kslice, kend = min(kbeg + p.kslice, a.K);
    f32x16_v acc[W][W];
    const Loader<T, AK, 64 * W> la(a.A, m0);
    const Loader<T, BKM, 64 * W> lb(a.B, n0);
    B::run(la, lb, kbeg, kend, lds, acc);
    if (p.slices > 1 && !B::combine(p, tile, slice, acc)) return;
    if constexpr (PLAIN) dense_epilogue_as<ML, T, W, W, true, 0, false>(acc, a, m0, n0);      // no bias, no activation
    else if (a.M >= ML::TILE_M && a.N >= ML::TILE_N) dense_epilogue<ML, T, W, W, true>(acc, a, m0, n0);
    else dense_epilogue<ML, T, W, W, false>(acc, a, m0, n0);
}

template <typename T, int W, bool AK, bool BKM>
__global__ __launch_bounds__(THREADS, (split_waves<T, W, W>())) void split_gemm_kernel(DenseArgs<T> a, Plan p) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    tile_slice<T, W, AK, BKM>(a, p, blockIdx.x, reinterpret_cast<T*>(lds_raw));
}

// The two gradient products of a dense layer in one launch: workgroups [0, first) compute dW, the rest dx.
template <typename T>
__global__ __launch_bounds__(THREADS) void split_gemm_pair_kernel(DenseArgs<T> a, Plan pa, DenseArgs<T> b, Plan pb, int first) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    if ((int)blockIdx.x < first) tile_slice<T, 1, false, false, true>(a, pa, blockIdx.x, reinterpret_cast<T*>(lds_raw));
    else tile_slice<T, 1, true, true, true>(b, pb, (int)blockIdx.x - first, reinterpret_cast<T*>(lds_raw));
}

}  // namespace split
}  // namespace luxhip
