// scaled_dot_product_attention of bf16 tensors without the logits (and, in the pullback, without their cotangent) in memory.
//
//   forward    weights = softmax(scale k'q, causal mask), out = v weights
//   pullback   dP = v' d_out,  dS = scale weights .* (dP - d),  d = sum over a column of d_out .* out,
//              dv = d_out weights',  dk = q dS',  dq = k dS
//
// What the products read is what the step-by-step path stores: the weights and dS rounded to bf16, sums and the softmax
// in fp32, `out` also unrounded (fp32) for d.  The rounded weights are an output of the operator, so they do go to memory
// (2 bytes each, once) and the pullback reads them instead of forming them again.
//
// What bounds these kernels: the forward pass writes S x L weights per head, which for 2048 x 2048 x 32 x 4 is 1.07 GB, and
// everything else is arranged to hide behind that stream.  Two sweeps over the keys (column maxima and sums, then weights
// and output) cost a second product k'q but no traffic.  The pullback forms v' d_out twice, once per sweep (over queries
// for dk, dv; over keys for dq), because handing dS from one to the other would write and read it.
// Measured at 128 x 2048 x 32 x 4, causal (step-by-step path before): forward 1.15 ms -> 0.53 ms, pullback 0.85 ms -> 0.69 ms.
//
// Layout of the work: a workgroup is four waves; a wave owns 32 columns (queries in the forward and dq kernels, keys in the
// dk / dv kernel) and walks the other dimension.  Every product is v_mfma_f32_32x32x16_bf16 with the walked dimension (or
// the features) as rows and the wave's columns as columns, so that
//   * a column of the softmax lies in two lanes (l and l + 32), its reductions are in-lane plus one exchange;
//   * the accumulator of one product is the B operand of the next without a shuffle: accumulator register r of half-wave h
//     holds row 8 (r / 4) + 4 h + r % 4, and the A operand's k slots are read in the same order (frag_t).
// Tiles of 64 (32 in the dk / dv kernel) rows go global -> registers -> LDS, double buffered with one barrier per tile.
// An LDS row is 256 bytes = sixteen 16-byte chunks; chunk c of row r is stored at c ^ f(r), f(r) = (r % 4) * 4 + (r / 4) % 4:
// sixteen consecutive rows then lie in sixteen different chunks for the row-wise reads, and the four rows of a transposing
// read (ds_read_b64_tr_b16) in four different 64-byte granules.
#include <algorithm>

#include "common.h"
#include "gemm_core.h"
#include "gemm_dense_decl.h"

namespace luxhip {
namespace attn {

constexpr int WAVES = 4, THREADS = WAVES * 64, COLS = 32 * WAVES;      // columns of a workgroup
constexpr int PITCH = 256;                                             // bytes of an LDS row
constexpr int MAX_E = 128;

struct Args {
    const bf16_t *q, *k, *v, *d_out;
    bf16_t *probs, *out;      // out: forward only
    float* out_wide;
    const float* d;           // [b][h][l]
    bf16_t *dq, *dk, *dv;
    int E, Ev, S, L, H, r;    // r: query heads per key / value head
    int heads;                // H * batches
    int blocks;               // column blocks per head
    int causal;
    float c, scale;           // scale * log2(e), scale
    int64_t qt, qh, qb, kt, kh, kb, vt, vh, vb, dkr, dvr;   // strides in elements: token, head, batch; repeat (dk, dv)
};

// ------------------------------------------------------------------------------------------------ who works on what
// Heads are dealt to the XCDs (consecutive workgroups go to different ones), all blocks of a head to one: its k and v then
// stay in one L2.  Fewer heads than that: block by block over all heads.  Causal work grows with the query block, so the
// long blocks come first (`reverse`: the last block is the longest).
struct Where {
    int head, block, h, b, g, i0;
    __device__ __forceinline__ Where(const Args& a, bool reverse) {
        const int id = blockIdx.x;
        if ((a.heads & 7) == 0) {
            const int idx = id >> 3;
            block = idx % a.blocks;
            head = (idx / a.blocks) * 8 + (id & 7);
        } else {
            block = id / a.heads;
            head = id - block * a.heads;
        }
        if (reverse) block = a.blocks - 1 - block;
        h = head % a.H;
        b = head / a.H;
        g = h / a.r;
        i0 = h - g * a.r;
    }
};

// ------------------------------------------------------------------------------------------------ tiles
__device__ __forceinline__ int swz(int row) { return ((row & 3) << 2) | ((row >> 2) & 3); }

// ROWS rows of a (tokens x features) operand, feature chunks past E and rows past `rows` as zeros
template <int ROWS, int ET>
struct Tile {
    static constexpr int NCH = ET == 1 ? 4 : ET == 2 ? 8 : 16;          // chunks of a row that are loaded
    static constexpr int STEP = THREADS / NCH;                           // rows per pass
    static constexpr int N = (ROWS + STEP - 1) / STEP;
    raw16_t reg[N];
    uint32_t row, chunk_bytes, lds;
    bool live;
    __device__ __forceinline__ explicit Tile(int E) {
        const int ch = threadIdx.x % NCH;
        row = threadIdx.x / NCH;
        live = ch * 8 < E;
        chunk_bytes = live ? ch * 16 : 0;
        lds = row * PITCH + ((ch ^ swz(row)) << 4);                      // STEP is a multiple of 16: the same f for every pass
        static_assert(STEP % 16 == 0, "rows of the passes must share their swizzle");
    }
    __device__ __forceinline__ bool mine(int i) const { return ROWS % STEP == 0 || row + i * STEP < (uint32_t)ROWS; }
    // rows r0 .. r0 + ROWS - 1 of the operand at p; `rows` > 0
    __device__ __forceinline__ void load(const bf16_t* p, uint32_t pitch_bytes, int r0, int rows) {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int r = min(r0 + (int)row + i * STEP, rows - 1);
            reg[i] = *reinterpret_cast<const raw16_t*>(reinterpret_cast<const char*>(p) + ((uint32_t)r * pitch_bytes + chunk_bytes));
        }
    }
    __device__ __forceinline__ void store(char* tile, int r0, int rows) const {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const bool in = live && r0 + (int)row + i * STEP < rows;
            const raw16_t zero = {0u, 0u, 0u, 0u};
            if (mine(i)) *reinterpret_cast<raw16_t*>(tile + lds + i * STEP * PITCH) = in ? reg[i] : zero;
        }
    }
};

// Row-wise fragment (A operand): rows r0 .. r0 + 31 of the tile, features 16 kk .. 16 kk + 15
struct FragRow {
    uint32_t off, h;
    __device__ __forceinline__ FragRow() {
        const int l = threadIdx.x & 63;
        h = l >> 5;
        off = (l & 31) * PITCH + ((h ^ swz(l & 31)) << 4);
    }
    __device__ __forceinline__ bf16x8_v get(const char* tile, int r0, int kk) const {     // r0: a multiple of 32
        return __builtin_bit_cast(bf16x8_v, *reinterpret_cast<const raw16_t*>(tile + r0 * PITCH + (off ^ (kk << 5))));
    }
};
// Transposed fragment (A operand): features 32 t .. 32 t + 31 as rows, tile rows r0 + {4h .. 4h + 3, 8 + 4h ..} as k slots
// (the order in which an accumulator holds its rows).  r0: a multiple of 16.
struct FragT {
    uint32_t lo;
    __device__ __forceinline__ FragT() {
        const int l = threadIdx.x & 63, b = l >> 4, s = l & 15, h = b >> 1;
        const int row = 4 * h + (s >> 2), chunk = 2 * (b & 1) + ((s & 3) >> 1);
        lo = row * PITCH + ((chunk ^ swz(row)) << 4) + (s & 1) * 8;
    }
    __device__ __forceinline__ static s16x4_v tr(const char* p) {
        typedef __attribute__((address_space(3))) s16x4_v* lds_ptr;
        return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(p));
    }
    __device__ __forceinline__ bf16x8_v get(const char* tile, int r0, int t) const {
        // row + 8: (row / 4) % 4 changes by 2, one XOR
        const s16x4_v a = tr(tile + r0 * PITCH + (lo ^ (t << 6))), b = tr(tile + (r0 + 8) * PITCH + (lo ^ (t << 6) ^ (2 << 4)));
        const s16x8_v v = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
        return __builtin_bit_cast(bf16x8_v, v);
    }
};

// The operand of the wave's own 32 columns (B operand), straight from memory: column `row`, all features
template <int ET>
__device__ __forceinline__ void load_columns(bf16x8_v (&f)[2 * ET], const bf16_t* p, uint32_t pitch_bytes, int row, int rows, int E) {
    const int h = (threadIdx.x & 63) >> 5;
    const char* base = reinterpret_cast<const char*>(p) + (uint32_t)min(row, rows - 1) * pitch_bytes;
#pragma unroll
    for (int kk = 0; kk < 2 * ET; ++kk) {
        const int ch = 2 * kk + h;
        const bool in = ch * 8 < E && row < rows;
        const raw16_t v = *reinterpret_cast<const raw16_t*>(base + (ch * 8 < E ? ch * 16 : 0)), zero = {0u, 0u, 0u, 0u};
        f[kk] = __builtin_bit_cast(bf16x8_v, in ? v : zero);
    }
}

// Accumulator registers 8 n .. 8 n + 7 as bf16 pairs, in register order: the B operand of a product whose A operand comes from FragT
__device__ __forceinline__ raw16_t pack8(const f32x16_v& v, int n) {
    raw16_t w;
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = f32x2_to_bf16x2(v[8 * n + 2 * i], v[8 * n + 2 * i + 1]);
    return w;
}
// Between that order (half-wave h: rows 4h .. 4h + 3, 8 + 4h ..) and the order of memory (half-wave h: rows 8h .. 8h + 7);
// its own inverse
__device__ __forceinline__ raw16_t reorder(raw16_t w) {
    const auto a = __builtin_amdgcn_permlane32_swap(w[0], w[2], false, false);
    const auto b = __builtin_amdgcn_permlane32_swap(w[1], w[3], false, false);
    return raw16_t{a[0], b[0], a[1], b[1]};
}

typedef uint32_t raw16_u __attribute__((ext_vector_type(4), aligned(2)));
// Eight consecutive bf16 at p + at, of which only those below `end` exist (ragged rows: any alignment)
__device__ __forceinline__ void store8(bf16_t* p, int at, int end, raw16_t w) {
    if (at + 8 <= end) {
        *reinterpret_cast<raw16_u*>(p + at) = w;
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (at + i < end) p[at + i] = (bf16_t)(w[i >> 1] >> ((i & 1) * 16));
    }
}
__device__ __forceinline__ raw16_t load8(const bf16_t* p, int at, int end) {
    raw16_t w = {0u, 0u, 0u, 0u};
    if (at + 8 <= end) {
        w = *reinterpret_cast<const raw16_u*>(p + at);
    } else if (at < end) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (at + i < end) w[i >> 1] |= (uint32_t)p[at + i] << ((i & 1) * 16);
    }
    return w;
}

// rows (features) x columns (the wave's tokens) accumulators to a (tokens x features) tensor
template <int ET>
__device__ __forceinline__ void store_features(const f32x16_v (&acc)[ET], bf16_t* row, bool in, int E) {
    const int h = (threadIdx.x & 63) >> 5;
#pragma unroll
    for (int t = 0; t < ET; ++t)
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            const raw16_t w = reorder(pack8(acc[t], n));
            const int e = 32 * t + 16 * n + 8 * h;
            if (in && e < E) *reinterpret_cast<raw16_t*>(row + e) = w;
        }
}

__device__ __forceinline__ f32x16_v zero16() {
    f32x16_v z;
#pragma unroll
    for (int i = 0; i < 16; ++i) z[i] = 0.0f;
    return z;
}
// accumulator register i of half-wave h: its row
__device__ __forceinline__ int acc_row(int i, int h) { return 8 * (i >> 2) + 4 * h + (i & 3); }

// ------------------------------------------------------------------------------------------------ forward
constexpr int KB = 64;                                  // keys per tile
constexpr int TILE_BYTES = KB * PITCH;                  // 16 KiB
constexpr size_t FWD_LDS = 4 * TILE_BYTES;              // k and v, two of each

template <int ET>
__global__ __launch_bounds__(THREADS, 2) void fwd_kernel(Args a) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    char* const kt = reinterpret_cast<char*>(lds_raw);
    char* const vt = kt + 2 * TILE_BYTES;
    const Where wh(a, a.causal != 0);
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5;
    const int l0 = wh.block * COLS, wl0 = l0 + 32 * w, l = wl0 + (lane & 31);
    const bf16_t* const kp = a.k + wh.g * a.kh + wh.b * a.kb;
    const bf16_t* const vp = a.v + wh.g * a.vh + wh.b * a.vb;
    const uint32_t kpitch = (uint32_t)(a.kt * 2), vpitch = (uint32_t)(a.vt * 2);
    const int s_end = a.causal ? min(a.S, l0 + COLS) : a.S;                    // keys that any query of the workgroup sees
    const int tiles = (s_end + KB - 1) / KB;
    const int w_end = wl0 >= a.L ? 0 : a.causal ? min(a.S, wl0 + 32) : a.S;    // ... of the wave
    const int limit = a.causal ? min(l, a.S - 1) : a.S - 1;
    const FragRow fr;
    const FragT ft;
    bf16x8_v qf[2 * ET];
    load_columns<ET>(qf, a.q + wh.h * a.qh + wh.b * a.qb, (uint32_t)(a.qt * 2), l, a.L, a.E);

    // scaled logits (times log2 e) of keys s0 .. s0 + 31 of tile buffer `tile`, -inf where masked
    auto logits = [&](const char* tile, int j, int s0) {
        f32x16_v z = zero16();
#pragma unroll
        for (int kk = 0; kk < 2 * ET; ++kk) z = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fr.get(tile, 32 * j, kk), qf[kk], z, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 16; ++i) z[i] *= a.c;
        if (s0 + 31 > (a.causal ? min(wl0, a.S - 1) : a.S - 1)) {
#pragma unroll
            for (int i = 0; i < 16; ++i)
                if (s0 + acc_row(i, h) > limit) z[i] = -INFINITY;
        }
        return z;
    };

    Tile<KB, ET> tk(a.E);
    // sweep 1: maximum and sum of exponentials, per lane (half of the keys of its column).  A column of which nothing but
    // -inf has been seen keeps the sum 0 (the subtrahend is 0 then).
    float m = -INFINITY, sum = 0.0f;
    tk.load(kp, kpitch, 0, a.S);
    tk.store(kt, 0, a.S);
    __syncthreads();
    for (int t = 0; t < tiles; ++t) {
        const char* cur = kt + (t & 1) * TILE_BYTES;
        if (t + 1 < tiles) tk.load(kp, kpitch, (t + 1) * KB, a.S);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int s0 = t * KB + 32 * j;
            if (s0 < w_end) {
                const f32x16_v z = logits(cur, j, s0);
                float mt = z[0];
#pragma unroll
                for (int i = 1; i < 16; ++i) mt = fmaxf(mt, z[i]);
                const float mn = fmaxf(m, mt), ms = mn == -INFINITY ? 0.0f : mn;
                float add = 0.0f;
#pragma unroll
                for (int i = 0; i < 16; ++i) add += __builtin_amdgcn_exp2f(z[i] - ms);
                sum = sum * __builtin_amdgcn_exp2f(m - ms) + add;
                m = mn;
            }
        }
        if (t + 1 < tiles) tk.store(kt + ((t + 1) & 1) * TILE_BYTES, (t + 1) * KB, a.S);
        __syncthreads();
    }
    float mx;
    float inv;
    {
        const float mo = __shfl_xor(m, 32), so = __shfl_xor(sum, 32);
        mx = fmaxf(m, mo);
        const float ms = mx == -INFINITY ? 0.0f : mx;
        inv = 1.0f / (sum * __builtin_amdgcn_exp2f(m - ms) + so * __builtin_amdgcn_exp2f(mo - ms));
    }

    // the tiles of sweep 2 on their way while the masked part of the columns is filled
    Tile<KB, ET> tv(a.Ev);
    tk.load(kp, kpitch, 0, a.S);
    tv.load(vp, vpitch, 0, a.S);
    bf16_t* const wrow0 = a.probs + ((int64_t)wh.head * a.L + wl0) * a.S;        // row wl0 of this head
    if (wl0 < a.L) {
        const int rows = min(32, a.L - wl0);
        for (int i = 0; i < rows; ++i) {                                         // a masked weight: 0 times 1 / sum
            const float z0 = 0.0f * __shfl(inv, i);
            const uint32_t zz = f32x2_to_bf16x2(z0, z0);
            const raw16_t zw = {zz, zz, zz, zz};
            for (int s = w_end + 8 * lane; s < a.S; s += 512) store8(wrow0 + (int64_t)i * a.S, s, a.S, zw);
        }
    }
    tk.store(kt, 0, a.S);
    tv.store(vt, 0, a.S);
    __syncthreads();

    // sweep 2: the weights, rounded, to memory and into the product with v
    f32x16_v o[ET];
#pragma unroll
    for (int t = 0; t < ET; ++t) o[t] = zero16();
    bf16_t* const wrow = wrow0 + (int64_t)(lane & 31) * a.S;
    for (int t = 0; t < tiles; ++t) {
        const char *kc = kt + (t & 1) * TILE_BYTES, *vc = vt + (t & 1) * TILE_BYTES;
        if (t + 1 < tiles) {
            tk.load(kp, kpitch, (t + 1) * KB, a.S);
            tv.load(vp, vpitch, (t + 1) * KB, a.S);
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int s0 = t * KB + 32 * j;
            if (s0 < w_end) {
                f32x16_v z = logits(kc, j, s0);
#pragma unroll
                for (int i = 0; i < 16; ++i) z[i] = __builtin_amdgcn_exp2f(z[i] - mx) * inv;
#pragma unroll
                for (int n = 0; n < 2; ++n) {
                    const raw16_t pw = pack8(z, n);
                    const raw16_t mem = reorder(pw);
                    if (l < a.L) store8(wrow, s0 + 16 * n + 8 * h, w_end, mem);
                    const bf16x8_v pb = __builtin_bit_cast(bf16x8_v, pw);
#pragma unroll
                    for (int e = 0; e < ET; ++e)
                        o[e] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ft.get(vc, 32 * j + 16 * n, e), pb, o[e], 0, 0, 0);
                }
            }
        }
        if (t + 1 < tiles) {
            tk.store(kt + ((t + 1) & 1) * TILE_BYTES, (t + 1) * KB, a.S);
            tv.store(vt + ((t + 1) & 1) * TILE_BYTES, (t + 1) * KB, a.S);
        }
        __syncthreads();
    }
    // out (Ev, H, L, B), rounded and unrounded
    const int64_t orow = (((int64_t)wh.b * a.L + l) * a.H + wh.h) * a.Ev;
    store_features<ET>(o, a.out + orow, l < a.L, a.Ev);
    if (l < a.L) {
#pragma unroll
        for (int t = 0; t < ET; ++t)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int e = 32 * t + 8 * g + 4 * h;
                if (e < a.Ev)
                    *reinterpret_cast<float4*>(a.out_wide + orow + e) = make_float4(o[t][4 * g], o[t][4 * g + 1], o[t][4 * g + 2], o[t][4 * g + 3]);
            }
    }
}

// ------------------------------------------------------------------------------------------------ pullback
// scale weights .* (dP - d) of 16 rows, as the B operand of the next product: pw as loaded (bf16 pairs in accumulator order)
__device__ __forceinline__ raw16_t softmax_rule(raw16_t pw, const f32x16_v& dp, int n, const float (&d)[8], float scale) {
    raw16_t out;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float p0 = __uint_as_float(pw[i] << 16), p1 = __uint_as_float(pw[i] & 0xffff0000u);
        out[i] = f32x2_to_bf16x2(scale * p0 * (dp[8 * n + 2 * i] - d[2 * i]), scale * p1 * (dp[8 * n + 2 * i + 1] - d[2 * i + 1]));
    }
    return out;
}

// dq: a wave owns 32 queries and walks the keys
template <int ET>
__global__ __launch_bounds__(THREADS, 2) void dq_kernel(Args a) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    char* const kt = reinterpret_cast<char*>(lds_raw);
    char* const vt = kt + 2 * TILE_BYTES;
    const Where wh(a, a.causal != 0);
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5;
    const int l0 = wh.block * COLS, wl0 = l0 + 32 * w, l = wl0 + (lane & 31);
    const bf16_t* const kp = a.k + wh.g * a.kh + wh.b * a.kb;
    const bf16_t* const vp = a.v + wh.g * a.vh + wh.b * a.vb;
    const uint32_t kpitch = (uint32_t)(a.kt * 2), vpitch = (uint32_t)(a.vt * 2);
    const int s_end = a.causal ? min(a.S, l0 + COLS) : a.S;
    const int tiles = (s_end + KB - 1) / KB;
    const int w_end = wl0 >= a.L ? 0 : a.causal ? min(a.S, wl0 + 32) : a.S;
    const int lc = min(l, a.L - 1);
    const FragRow fr;
    const FragT ft;
    bf16x8_v df[2 * ET];
    load_columns<ET>(df, a.d_out + ((int64_t)wh.b * a.L * a.H + wh.h) * a.Ev, (uint32_t)(a.H * a.Ev * 2), l, a.L, a.Ev);
    const float dl = a.d[(int64_t)wh.head * a.L + lc];
    const bf16_t* const wrow = a.probs + ((int64_t)wh.head * a.L + lc) * a.S;
    raw16_t pw[4];                        // the weights of the tile about to be used: 64 keys of the lane's query
    auto load_weights = [&](int s0) {
#pragma unroll
        for (int n = 0; n < 4; ++n) pw[n] = load8(wrow, s0 + 16 * n + 8 * h, w_end);
    };
    Tile<KB, ET> tk(a.E), tv(a.Ev);
    tk.load(kp, kpitch, 0, a.S);
    tv.load(vp, vpitch, 0, a.S);
    load_weights(0);
    f32x16_v acc[ET];
#pragma unroll
    for (int t = 0; t < ET; ++t) acc[t] = zero16();
    const float dd[8] = {dl, dl, dl, dl, dl, dl, dl, dl};
    tk.store(kt, 0, a.S);
    tv.store(vt, 0, a.S);
    __syncthreads();
    for (int t = 0; t < tiles; ++t) {
        const char *kc = kt + (t & 1) * TILE_BYTES, *vc = vt + (t & 1) * TILE_BYTES;
        raw16_t pc[4];
#pragma unroll
        for (int n = 0; n < 4; ++n) pc[n] = pw[n];
        if (t + 1 < tiles) {
            tk.load(kp, kpitch, (t + 1) * KB, a.S);
            tv.load(vp, vpitch, (t + 1) * KB, a.S);
            load_weights((t + 1) * KB);
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            if (t * KB + 32 * j < w_end) {
                f32x16_v dp = zero16();
#pragma unroll
                for (int kk = 0; kk < 2 * ET; ++kk) dp = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fr.get(vc, 32 * j, kk), df[kk], dp, 0, 0, 0);
#pragma unroll
                for (int n = 0; n < 2; ++n) {
                    const bf16x8_v ds = __builtin_bit_cast(bf16x8_v, softmax_rule(reorder(pc[2 * j + n]), dp, n, dd, a.scale));
#pragma unroll
                    for (int e = 0; e < ET; ++e)
                        acc[e] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ft.get(kc, 32 * j + 16 * n, e), ds, acc[e], 0, 0, 0);
                }
            }
        }
        if (t + 1 < tiles) {
            tk.store(kt + ((t + 1) & 1) * TILE_BYTES, (t + 1) * KB, a.S);
            tv.store(vt + ((t + 1) & 1) * TILE_BYTES, (t + 1) * KB, a.S);
        }
        __syncthreads();
    }
    store_features<ET>(acc, a.dq + wh.h * a.qh + wh.b * a.qb + (int64_t)lc * a.qt, l < a.L, a.E);
}

// dk, dv: a wave owns 32 keys and walks the queries
constexpr int LB = 32;                                          // queries per tile
constexpr int LTILE = LB * PITCH;                               // 8 KiB: 32 queries x (128 features | 128 keys of the workgroup)
constexpr size_t DKV_LDS = 2 * (3 * LTILE + LB * 4);            // q, d_out, weights and d, two of each

template <int ET>
__global__ __launch_bounds__(THREADS, 2) void dkv_kernel(Args a) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    char* const qt = reinterpret_cast<char*>(lds_raw);
    char* const ot = qt + 2 * LTILE;
    char* const pt = ot + 2 * LTILE;
    float* const dt = reinterpret_cast<float*>(pt + 2 * LTILE);
    const Where wh(a, false);                                   // causal: the first block of keys is seen by every query
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5;
    const int s0 = wh.block * COLS, ws0 = s0 + 32 * w, s = ws0 + (lane & 31);
    const bf16_t* const qp = a.q + wh.h * a.qh + wh.b * a.qb;
    const bf16_t* const op = a.d_out + ((int64_t)wh.b * a.L * a.H + wh.h) * a.Ev;
    const bf16_t* const pp = a.probs + (int64_t)wh.head * a.L * a.S;
    const float* const dp_ = a.d + (int64_t)wh.head * a.L;
    const uint32_t qpitch = (uint32_t)(a.qt * 2), opitch = (uint32_t)(a.H * a.Ev * 2);
    const int first = a.causal ? s0 / LB : 0, tiles = (a.L + LB - 1) / LB;
    const int w_first = ws0 >= a.S ? tiles : a.causal ? ws0 / LB : 0;
    const FragRow fr;
    const FragT ft;
    bf16x8_v vf[2 * ET];
    load_columns<ET>(vf, a.v + wh.g * a.vh + wh.b * a.vb, (uint32_t)(a.vt * 2), s, a.S, a.Ev);
    f32x16_v ak[ET], av[ET];
#pragma unroll
    for (int t = 0; t < ET; ++t) { ak[t] = zero16(); av[t] = zero16(); }

    Tile<LB, ET> tq(a.E), to(a.Ev);
    // weights: 32 queries x 128 keys, two chunks of eight keys per thread
    raw16_t pw[2];
    float dv = 0.0f;
    const int prow = threadIdx.x >> 4, pch = threadIdx.x & 15;
    const uint32_t plds = prow * PITCH + ((pch ^ swz(prow)) << 4);
    auto load = [&](int t) {
        tq.load(qp, qpitch, t * LB, a.L);
        to.load(op, opitch, t * LB, a.L);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int r = t * LB + prow + 16 * i;
            pw[i] = load8(pp + (int64_t)min(r, a.L - 1) * a.S, s0 + 8 * pch, r < a.L ? a.S : 0);
        }
        if (threadIdx.x < LB) {                     // 0 past the end: a non-finite d must not reach the keys through absent queries
            const int r = t * LB + (int)threadIdx.x;
            dv = r < a.L ? dp_[r] : 0.0f;
        }
    };
    auto store = [&](int t) {
        const int b = t & 1;
        tq.store(qt + b * LTILE, t * LB, a.L);
        to.store(ot + b * LTILE, t * LB, a.L);
#pragma unroll
        for (int i = 0; i < 2; ++i) *reinterpret_cast<raw16_t*>(pt + b * LTILE + plds + i * 16 * PITCH) = pw[i];
        if (threadIdx.x < LB) dt[b * LB + threadIdx.x] = dv;
    };
    if (first < tiles) {
        load(first);
        store(first);
    }
    __syncthreads();
    for (int t = first; t < tiles; ++t) {
        const int b = t & 1;
        const char *qc = qt + b * LTILE, *oc = ot + b * LTILE, *pc = pt + b * LTILE;
        if (t + 1 < tiles) load(t + 1);
        if (t >= w_first) {
            f32x16_v dp = zero16();
#pragma unroll
            for (int kk = 0; kk < 2 * ET; ++kk) dp = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fr.get(oc, 0, kk), vf[kk], dp, 0, 0, 0);
#pragma unroll
            for (int n = 0; n < 2; ++n) {
                const bf16x8_v pb = ft.get(pc, 16 * n, w);       // the wave's 32 keys are "features" 32 w .. of the weights' tile
#pragma unroll
                for (int e = 0; e < ET; ++e) av[e] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ft.get(oc, 16 * n, e), pb, av[e], 0, 0, 0);
                float dd[8];
                const float4 d0 = *reinterpret_cast<const float4*>(dt + b * LB + 16 * n + 4 * h);
                const float4 d1 = *reinterpret_cast<const float4*>(dt + b * LB + 16 * n + 8 + 4 * h);
                dd[0] = d0.x; dd[1] = d0.y; dd[2] = d0.z; dd[3] = d0.w;
                dd[4] = d1.x; dd[5] = d1.y; dd[6] = d1.z; dd[7] = d1.w;
                const bf16x8_v ds = __builtin_bit_cast(bf16x8_v, softmax_rule(__builtin_bit_cast(raw16_t, pb), dp, n, dd, a.scale));
#pragma unroll
                for (int e = 0; e < ET; ++e) ak[e] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ft.get(qc, 16 * n, e), ds, ak[e], 0, 0, 0);
            }
        }
        if (t + 1 < tiles) store(t + 1);
        __syncthreads();
    }
    const int sc = min(s, a.S - 1);
    store_features<ET>(ak, a.dk + wh.i0 * a.dkr + wh.g * a.kh + wh.b * a.kb + (int64_t)sc * a.kt, s < a.S, a.E);
    store_features<ET>(av, a.dv + wh.i0 * a.dvr + wh.g * a.vh + wh.b * a.vb + (int64_t)sc * a.vt, s < a.S, a.Ev);
}

// ------------------------------------------------------------------------------------------------ host
template <int ET>
static int launch_fwd(hipStream_t s, Args& a) {
    static ResidentOnce ro;
    ro.get([&](hipError_t& err) {
        err = hipFuncSetAttribute(reinterpret_cast<const void*>(fwd_kernel<ET>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)FWD_LDS);
        return 1;
    });
    LUX_CHECK_HIP(ro.error);
    a.blocks = (int)ceil_div(a.L, COLS);
    ProfScope ps("attn_fwd_kernel", s);
    fwd_kernel<ET><<<dim3((unsigned)a.blocks * (unsigned)a.heads), dim3(THREADS), FWD_LDS, s>>>(a);
    LUX_CHECK_LAUNCH();
    return LUXHIP_OK;
}
template <int ET>
static int launch_bwd(hipStream_t s, Args& a) {
    static ResidentOnce ro;
    ro.get([&](hipError_t& err) {
        err = hipFuncSetAttribute(reinterpret_cast<const void*>(dq_kernel<ET>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)FWD_LDS);
        if (err == hipSuccess)
            err = hipFuncSetAttribute(reinterpret_cast<const void*>(dkv_kernel<ET>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)DKV_LDS);
        return 1;
    });
    LUX_CHECK_HIP(ro.error);
    a.blocks = (int)ceil_div(a.S, COLS);
    {
        ProfScope ps("attn_dkv_kernel", s);
        dkv_kernel<ET><<<dim3((unsigned)a.blocks * (unsigned)a.heads), dim3(THREADS), DKV_LDS, s>>>(a);
        LUX_CHECK_LAUNCH();
    }
    a.blocks = (int)ceil_div(a.L, COLS);
    ProfScope ps("attn_dq_kernel", s);
    dq_kernel<ET><<<dim3((unsigned)a.blocks * (unsigned)a.heads), dim3(THREADS), FWD_LDS, s>>>(a);
    LUX_CHECK_LAUNCH();
    return LUXHIP_OK;
}

// Offsets inside one head's operand are 32-bit bytes, a grid has fewer than 2^31 / 256 workgroups, loads are 16 bytes wide
static int check(const Args& a, int64_t batches) {
    const auto plane = [](int64_t tokens, int64_t stride) { return tokens * stride * 2 < (int64_t(1) << 31); };
    LUX_UNSUPPORTED_IF(!plane(a.L, a.qt) || !plane(a.S, a.kt) || !plane(a.S, a.vt) || !plane(a.L, (int64_t)a.H * a.Ev),
                       "attention: an operand of a head spans 2 GiB or more");
    LUX_UNSUPPORTED_IF((int64_t)a.H * batches >= (1 << 23) || ceil_div(std::max(a.L, a.S), COLS) * a.H * batches >= (1 << 23),
                       "attention: too many workgroups");
    return LUXHIP_OK;
}

}  // namespace attn
}  // namespace luxhip

using namespace luxhip;

// Fills the fields that both directions share; what the kernels assume of the operands is checked here
static int attention_args(attn::Args& a, int dtype, int64_t E, int64_t Ev, int64_t S, int64_t L, const int64_t* batch_dims, double scale,
                          int causal, const void* q, const int64_t* sq, const void* k, const int64_t* sk, const void* v, const int64_t* sv) {
    LUX_UNSUPPORTED_IF(dtype != LUXHIP_BF16, "fused attention exists for bf16 storage only");
    LUX_INVALID_IF(E < 0 || Ev < 0 || S < 0 || L < 0, "attention: negative dimension");
    LUX_INVALID_IF(batch_dims == nullptr || sq == nullptr || sk == nullptr || sv == nullptr, "attention: extents and strides must not be NULL");
    for (int i = 0; i < 3; ++i) {
        LUX_INVALID_IF(batch_dims[i] < 0, "attention: negative batch extent");
        LUX_UNSUPPORTED_IF(batch_dims[i] >= (1 << 23), "attention: batch extent too large");
        LUX_INVALID_IF(sq[i] < 0 || sk[i] < 0 || sv[i] < 0, "attention: negative stride");
        LUX_UNSUPPORTED_IF(sq[i] % 8 != 0 || sk[i] % 8 != 0 || sv[i] % 8 != 0, "fused attention: strides must be multiples of 8 elements");
    }
    LUX_UNSUPPORTED_IF(E == 0 || Ev == 0 || E > attn::MAX_E || Ev > attn::MAX_E || E % 8 != 0 || Ev % 8 != 0,
                       "fused attention: at most 128 features, in multiples of 8");
    LUX_UNSUPPORTED_IF(S >= (1ll << 30) || L >= (1ll << 30), "fused attention: too many tokens");
    a.H = (int)(batch_dims[0] * batch_dims[1]);
    LUX_UNSUPPORTED_IF(batch_dims[0] * batch_dims[1] >= (1 << 23), "attention: too many heads");
    a.q = (const bf16_t*)q; a.k = (const bf16_t*)k; a.v = (const bf16_t*)v;
    a.E = (int)E; a.Ev = (int)Ev; a.S = (int)S; a.L = (int)L;
    a.r = (int)batch_dims[0];
    a.qt = sq[0]; a.qh = sq[1]; a.qb = sq[2];
    a.kt = sk[0]; a.kh = sk[1]; a.kb = sk[2];
    a.vt = sv[0]; a.vh = sv[1]; a.vb = sv[2];
    a.causal = causal != 0;
    a.scale = (float)scale;
    a.c = (float)(scale * 1.4426950408889634);
    if (S == 0 || L == 0 || a.H == 0 || batch_dims[2] == 0) return LUXHIP_OK;
    LUX_INVALID_IF(q == nullptr || k == nullptr || v == nullptr, "attention: null operand");
    LUX_UNSUPPORTED_IF(!aligned16(q) || !aligned16(k) || !aligned16(v), "fused attention: operands must be 16-byte aligned");
    const int rc = attn::check(a, batch_dims[2]);
    if (rc != LUXHIP_OK) return rc;
    a.heads = (int)(a.H * batch_dims[2]);
    return LUXHIP_OK;
}

#define ATTN_DISPATCH(FN)                             \
    switch ((std::max(E, Ev) + 31) / 32) {            \
        case 1: return attn::FN<1>((hipStream_t)s, a); \
        case 2: return attn::FN<2>((hipStream_t)s, a); \
        case 3: return attn::FN<3>((hipStream_t)s, a); \
        default: return attn::FN<4>((hipStream_t)s, a); \
    }

extern "C" {

int luxhip_attention_fwd(luxhip_stream_t s, int dtype, int64_t E, int64_t Ev, int64_t S, int64_t L, const int64_t* batch_dims,
                         double scale, int causal, const void* q, const int64_t* strides_q, const void* k, const int64_t* strides_k,
                         const void* v, const int64_t* strides_v, void* probs, void* out, float* out_wide) {
    LUX_REQUIRE_INIT();
    attn::Args a = {};
    const int rc = attention_args(a, dtype, E, Ev, S, L, batch_dims, scale, causal, q, strides_q, k, strides_k, v, strides_v);
    if (rc != LUXHIP_OK) return rc;
    if (a.heads == 0) {
        LUX_UNSUPPORTED_IF(S == 0 && L > 0 && a.H > 0 && batch_dims[2] > 0, "fused attention: no keys");
        return LUXHIP_OK;
    }
    LUX_INVALID_IF(probs == nullptr || out == nullptr || out_wide == nullptr, "attention_fwd: null result");
    LUX_UNSUPPORTED_IF(!aligned16(out) || !aligned16(out_wide), "fused attention: results must be 16-byte aligned");
    a.probs = (bf16_t*)probs;
    a.out = (bf16_t*)out;
    a.out_wide = out_wide;
    ATTN_DISPATCH(launch_fwd)
}

int luxhip_attention_bwd(luxhip_stream_t s, int dtype, int64_t E, int64_t Ev, int64_t S, int64_t L, const int64_t* batch_dims,
                         double scale, int causal, const void* q, const int64_t* strides_q, const void* k, const int64_t* strides_k,
                         const void* v, const int64_t* strides_v, const void* probs, const float* out_wide, const void* d_out, void* dq,
                         void* dk, int64_t dk_repeat, void* dv, int64_t dv_repeat) {
    LUX_REQUIRE_INIT();
    attn::Args a = {};
    int rc = attention_args(a, dtype, E, Ev, S, L, batch_dims, scale, causal, q, strides_q, k, strides_k, v, strides_v);
    if (rc != LUXHIP_OK) return rc;
    LUX_UNSUPPORTED_IF(a.heads == 0, "fused attention: nothing to do");      // the caller's products write the zeros
    LUX_INVALID_IF(probs == nullptr || out_wide == nullptr || d_out == nullptr || dq == nullptr || dk == nullptr || dv == nullptr,
                   "attention_bwd: null operand");
    LUX_INVALID_IF(dk_repeat < 0 || dv_repeat < 0, "attention_bwd: negative stride");
    LUX_UNSUPPORTED_IF(!aligned16(d_out) || !aligned16(out_wide) || !aligned16(dq) || !aligned16(dk) || !aligned16(dv) || dk_repeat % 8 != 0 ||
                           dv_repeat % 8 != 0,
                       "fused attention: operands must be 16-byte aligned");
    Workspace ws;
    rc = get_workspace((hipStream_t)s, (size_t)a.heads * a.L * sizeof(float), &ws);
    if (rc != LUXHIP_OK) return rc;
    const int64_t so[3] = {a.Ev, (int64_t)a.Ev * a.r, (int64_t)a.Ev * a.H * a.L};
    rc = attention_rowdot((hipStream_t)s, (const bf16_t*)d_out, out_wide, reinterpret_cast<float*>(ws.data), a.Ev, a.L, (int64_t)a.Ev * a.H,
                          batch_dims, so);
    if (rc != LUXHIP_OK) return rc;
    a.d = reinterpret_cast<const float*>(ws.data);
    a.probs = const_cast<bf16_t*>((const bf16_t*)probs);
    a.d_out = (const bf16_t*)d_out;
    a.dq = (bf16_t*)dq;
    a.dk = (bf16_t*)dk;
    a.dv = (bf16_t*)dv;
    a.dkr = dk_repeat;
    a.dvr = dv_repeat;
    ATTN_DISPATCH(launch_bwd)
}

}  // extern "C"
