// fp32 products of batches (the step-by-step attention, batched_matmul) in tiles of 64 x 64 with the main loop of gemm_split.h: loads 16
// bytes wide at any alignment, two or four stages per trip to memory, the contraction cut into slices where the tiles are few.
//
// What bounds them is latency: a product of 96 features x 1685 tokens has 54 tiles of up to 1685 k, and 128 x 128 tiles of a few heads
// leave most compute units idle.  Measured beside the choice (gemm_split_batched_f32.hip).  A tile at the end of a dimension is not moved back here but clamps its rows (a triangular structure goes
// by the tiles' places: what a product leaves out, no other may read).
#pragma once

#include "gemm_split.h"

namespace luxhip {
namespace split {

// Rows r0 .. of an operand, clamped to those that there are
template <typename T>
__device__ __forceinline__ Operand<T> rows_from(Operand<T> op, int r0) {
    op.p += (int64_t)r0 * op.sr;
    op.rows -= r0;
    return op;
}

template <typename T, bool AK, bool BKM, bool EP>
__global__ __launch_bounds__(THREADS) void split_batched_kernel(DenseArgs<T> a, Plan p) {
    using B = Body<T, 1, AK, BKM>;
    using ML = typename B::ML;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    const int tiles = a.tiles_m * a.tiles_n;
    // the tiles of a product are neighbours on an XCD, the slices of a tile next to each other
    const int unit = xcd_regroup(blockIdx.x, tiles * a.batch * p.slices), id = unit / p.slices, slice = unit - id * p.slices;
    const int b = id / tiles, tile = id - b * tiles;
    const int tn = tile / a.tiles_m, tm = tile - tn * a.tiles_m;
    const int m0 = tm * ML::TILE_M, n0 = tn * ML::TILE_N;
    // a.structure as in batch_tile
    if (a.structure == 1 && m0 >= ((n0 + ML::TILE_N - 1) / 128 + 1) * 128) return;
    const int klo = a.structure == 3 ? min(n0, a.K) : 0, khi = a.structure == 2 ? min(a.K, n0 + ML::TILE_N) : a.K;
    const int slices = max((khi - klo + p.kslice - 1) / p.kslice, 1);      // of this tile
    if (slice >= slices) return;
    const int kbeg = klo + slice * p.kslice, kend = min(kbeg + p.kslice, khi);
    const int i0 = b % a.bdim[0], r0 = b / a.bdim[0], i1 = r0 % a.bdim[1], i2 = r0 / a.bdim[1];
    Operand<T> oa = a.A, ob = a.B;
    oa.p += i0 * a.bsA[0] + i1 * a.bsA[1] + i2 * a.bsA[2];
    ob.p += i0 * a.bsB[0] + i1 * a.bsB[1] + i2 * a.bsB[2];
    const int64_t coff = i0 * a.bsC[0] + i1 * a.bsC[1] + i2 * a.bsC[2];
    std::conditional_t<EP, SoftmaxRuleOperands<ML, T, 1, 1, false>, NoOperands> ep;
    if constexpr (EP) ep.load(a, coff, b, m0, n0);
    f32x16_v acc[1][1];
    constexpr int VEC = GemmTraits<T>::VEC;
    const Loader<T, AK, 64> la(rows_from(oa, m0), 0, AK ? 0 : max(VEC - (a.M - m0), 0));
    const Loader<T, BKM, 64> lb(rows_from(ob, n0), 0, BKM ? 0 : max(VEC - (a.N - n0), 0));
    B::run(la, lb, kbeg, kend, reinterpret_cast<T*>(lds_raw), acc);
    if constexpr (EP) {
        ep.store(acc, a, coff, m0, n0);
    } else {
        if (slices > 1) {
            Plan own = p;                                       // the slices that arrive; partial sums lie p.slices apart
            own.partial = p.partial + (size_t)id * p.slices * (64 * 64);
            own.counters = p.counters + id;
            own.slices = slices;
            if (!B::combine(own, 0, slice, acc)) return;
        }
        DenseArgs<T> out = a;
        out.C = a.C + coff;
        dense_epilogue_as<ML, T, 1, 1, true, 0, false>(acc, out, m0, n0);
    }
}

}  // namespace split
}  // namespace luxhip
