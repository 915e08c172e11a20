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
// Measured at 128 x 2048 x 32 x 4, causal (step-by-step path before): forward 1.15 ms -> 0.46 ms, pullback 0.85 ms -> 0.56 ms
// (dq 0.28, dk and dv 0.28; without the loads and stores of the weights 0.32, 0.21 and 0.26 of 0.48, 0.285 and 0.305).
//
// Layout of the work: a workgroup is four waves; a wave owns 32 columns (queries in the forward and dq kernels, keys in the
// dk / dv kernel) and walks the other dimension.  Every product is v_mfma_f32_32x32x16_bf16 with the walked dimension (or
// the features) as rows and the wave's columns as columns, so that
//   * a column of the softmax lies in two lanes (l and l + 32), its reductions are in-lane plus one exchange;
//   * the accumulator of one product is the B operand of the next without a shuffle: accumulator register r of half-wave h
//     holds row 8 (r / 4) + 4 h + r % 4, and the A operand's k slots are read in the same order (frag_t).
// Tiles of 32 rows go global -> registers -> LDS, double buffered with one barrier per tile.  An LDS row is 256 bytes in a
// pitch of 336 = 5 x 64 + 16: sixteen consecutive rows start in sixteen different 16-byte chunks of the 256-byte bank period
// (row-wise reads: no conflict), the four rows of a transposing read (ds_read_b64_tr_b16) 80 bytes apart (at most two lanes
// on a bank).  XOR-swizzled rows have no conflicts at all, but every fragment address is then an XOR and an addition where
// it is an immediate here: 234 vector instructions per 32 x 32 tile of the dk / dv kernel, which had become its bound.
#include <algorithm>
#include <cmath>

#include "common.h"
#include "gemm_core.h"

namespace luxhip {
namespace attn {

constexpr int WAVES = 4, THREADS = WAVES * 64, COLS = 32 * WAVES;      // columns of a workgroup
constexpr int ROWS = 32, PITCH = 336, TILE = ROWS * PITCH;              // a tile in LDS: rows, bytes of a row, bytes
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
    int negative;             // the sign of the scale, which the forward kernel moves to q
    float c, scale;           // |scale| log2(e), scale
    float* dsum;              // where the dq kernel leaves d for the dk / dv kernel
    int64_t qt, qh, qb, kt, kh, kb, vt, vh, vb, dkr, dvr;   // strides in elements: token, head, batch; repeat (dk, dv)
};

// ------------------------------------------------------------------------------------------------ who works on what
// Block by block over all heads: consecutive workgroups go to different XCDs, so with a multiple of eight heads all blocks
// of a head share one XCD's L2.  Under a causal mask the work grows with the query block and the masked part, which the
// forward kernel fills, shrinks:
//   REVERSE: the long blocks of all heads first (head by head, the last head's long blocks ran on while most compute units
//     were done: 70 % of the wave slots in use over the kernel);
//   ALTERNATE: last, first, second last, ...: blocks that compute and blocks that fill run side by side.
enum Order { FORWARD, REVERSE, ALTERNATE };
struct Where {
    int head, block, h, b, g, i0;
    __device__ __forceinline__ Where(const Args& a, Order order) {
        block = blockIdx.x / a.heads;
        head = blockIdx.x - block * a.heads;
        if (order == REVERSE) block = a.blocks - 1 - block;
        if (order == ALTERNATE) block = (block & 1) ? block >> 1 : a.blocks - 1 - (block >> 1);
        h = head % a.H;
        b = head / a.H;
        g = h / a.r;
        i0 = h - g * a.r;
    }
};

// ------------------------------------------------------------------------------------------------ tiles
// 32 rows of a (tokens x features) operand, one tile after the other; features past E and rows past the last as zeros.
// SETS tiles are on their way at a time, in register sets 0, 1 in turn.  Every load is issued unconditionally (past the end: the
// last row once more): a load under a condition, even a uniform one, makes the compiler's wait for an older load a wait for all.
template <int ET, int SETS>
struct Tile {
    static constexpr int NCH = ET == 1 ? 4 : ET == 2 ? 8 : 16;          // chunks of a row that are loaded
    static constexpr int STEP = THREADS / NCH;                           // rows per pass
    static constexpr int N = (ROWS + STEP - 1) / STEP;
    raw16_t reg[SETS][N];
    const char* p;
    uint32_t pitch, off, last, lds;      // off: this thread's chunk in its first row of the next tile; last: in the last row
    int row;
    bool live;
    __device__ __forceinline__ Tile(const bf16_t* p_, int64_t stride, int E, int rows, int first)
        : p(reinterpret_cast<const char*>(p_)), pitch((uint32_t)(stride * 2)) {
        const int ch = threadIdx.x % NCH;
        row = threadIdx.x / NCH;
        live = row < ROWS && ch * 8 < E;
        const uint32_t cb = ch * 8 < E ? ch * 16 : 0;
        off = (uint32_t)(ROWS * first + row) * pitch + cb;
        last = (uint32_t)(rows - 1) * pitch + cb;
        lds = row * PITCH + ch * 16;
    }
    // chunks that no tile fills
    __device__ __forceinline__ void clear(char* tile) const {
        const raw16_t zero = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int i = 0; i < N; ++i)
            if (row < ROWS && !live) *reinterpret_cast<raw16_t*>(tile + lds + i * STEP * PITCH) = zero;
    }
    __device__ __forceinline__ void load(int set) {
#pragma unroll
        for (int i = 0; i < N; ++i) reg[set][i] = *reinterpret_cast<const raw16_t*>(p + min(off + i * STEP * pitch, last));
        off += ROWS * pitch;
    }
    // tile t of an operand of `rows` rows
    __device__ __forceinline__ void store(char* tile, int set, int t, int rows) const {
        if (ROWS * (t + 1) <= rows) {      // uniform
#pragma unroll
            for (int i = 0; i < N; ++i)
                if (live) *reinterpret_cast<raw16_t*>(tile + lds + i * STEP * PITCH) = reg[set][i];
        } else {
            const raw16_t zero = {0u, 0u, 0u, 0u};
#pragma unroll
            for (int i = 0; i < N; ++i)
                if (live) *reinterpret_cast<raw16_t*>(tile + lds + i * STEP * PITCH) = ROWS * t + row + i * STEP < rows ? reg[set][i] : zero;
        }
    }
};

// Row-wise fragment (A operand): the tile's rows, features 16 kk .. 16 kk + 15
struct FragRow {
    uint32_t off;
    __device__ __forceinline__ FragRow() {
        const int l = threadIdx.x & 63;
        off = (l & 31) * PITCH + (l >> 5) * 16;
    }
    __device__ __forceinline__ bf16x8_v get(const char* tile, int kk) const {
        return __builtin_bit_cast(bf16x8_v, *reinterpret_cast<const raw16_t*>(tile + off + 32 * kk));
    }
};
// Transposed fragment (A operand): features 32 t .. 32 t + 31 as rows, tile rows r0 + {4h .. 4h + 3, 8 + 4h ..} as k slots
// (the order in which an accumulator holds its rows)
struct FragT {
    uint32_t off;
    __device__ __forceinline__ FragT() {
        const int l = threadIdx.x & 63, b = l >> 4, s = l & 15;
        off = (4 * (b >> 1) + (s >> 2)) * PITCH + (b & 1) * 32 + (s & 3) * 8;
    }
    __device__ __forceinline__ static s16x4_v tr(const char* p) {
        typedef __attribute__((address_space(3))) s16x4_v* lds_ptr;
        return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(p));
    }
    __device__ __forceinline__ bf16x8_v get(const char* tile, int r0, int t) const {
        const s16x4_v a = tr(tile + off + r0 * PITCH + 64 * t), b = tr(tile + off + (r0 + 8) * PITCH + 64 * t);
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

typedef uint32_t raw16_u __attribute__((ext_vector_type(4), aligned(2)));       // anywhere in a row of weights
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

// 32 columns (one per lane of a half-wave) x 64 keys of weights between the lanes that own a column and full lines of memory:
// a wave's own 4 KiB of LDS, 128 bytes per column, its eight chunks XORed with column % 8.  Straight from the lanes a store
// instruction touches 32 lines with 32 bytes each; this way eight whole ones.  No workgroup barrier is between the lanes that write
// and those that read: the LDS takes a wave's accesses in their order, and exchange() keeps the compiler to that order.
constexpr int PT_BYTES = 32 * 128;
struct WeightTile {
    char* lds;
    int lane;
    __device__ __forceinline__ WeightTile(void* p, int w) : lds((char*)p + w * PT_BYTES), lane(threadIdx.x & 63) {}
    // between one side's accesses and the other's
    __device__ __forceinline__ static void exchange() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
    }
    // keys 16 n + {4h .. 4h + 3, 8 + 4h ..} of this lane's column (accumulator order)
    __device__ __forceinline__ void put(int n, raw16_t w) const {
        const int c = lane & 31, h = lane >> 5;
        char* row = lds + c * 128 + 8 * h;
        *reinterpret_cast<uint2*>(row + (((2 * n) ^ (c & 7)) << 4)) = make_uint2(w[0], w[1]);
        *reinterpret_cast<uint2*>(row + (((2 * n + 1) ^ (c & 7)) << 4)) = make_uint2(w[2], w[3]);
    }
    __device__ __forceinline__ raw16_t get(int n) const {
        const int c = lane & 31, h = lane >> 5;
        const char* row = lds + c * 128 + 8 * h;
        const uint2 a = *reinterpret_cast<const uint2*>(row + (((2 * n) ^ (c & 7)) << 4));
        const uint2 b = *reinterpret_cast<const uint2*>(row + (((2 * n + 1) ^ (c & 7)) << 4));
        return raw16_t{a.x, a.y, b.x, b.y};
    }
    // line side, i < 4: column 8 i + lane / 8, keys 8 (lane % 8) ...
    __device__ __forceinline__ int column(int i) const { return 8 * i + (lane >> 3); }
    __device__ __forceinline__ int key() const { return 8 * (lane & 7); }
    __device__ __forceinline__ raw16_t* line(int i) const {
        return reinterpret_cast<raw16_t*>(lds + column(i) * 128 + (((lane & 7) ^ (lane >> 3)) << 4));
    }
};

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

// (32 rows of the tile) x (the wave's 32 columns), contracted over the features
// G: fragments that are on their way before the first product waits for one
template <int ET, int G>
__device__ __forceinline__ f32x16_v product(const FragRow& fr, const char* tile, const bf16x8_v (&cols)[2 * ET]) {
    f32x16_v z = zero16();
#pragma unroll
    for (int k0 = 0; k0 < 2 * ET; k0 += G) {
        bf16x8_v f[G];
#pragma unroll
        for (int i = 0; i < G; ++i)
            if (k0 + i < 2 * ET) f[i] = fr.get(tile, k0 + i);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < G; ++i)
            if (k0 + i < 2 * ET) z = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[i], cols[k0 + i], z, 0, 0, 0);
    }
    return z;
}

// ------------------------------------------------------------------------------------------------ forward
constexpr size_t FWD_LDS = 4 * TILE + WAVES * PT_BYTES;     // k and v, two tiles of each, and the waves' weights: 58 KiB

template <int ET>
__global__ __launch_bounds__(THREADS, 2) void fwd_kernel(Args a) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    char* const lds = reinterpret_cast<char*>(lds_raw);     // k 0, k 1, v 0, v 1, weights
    const Where wh(a, a.causal ? ALTERNATE : FORWARD);
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5;
    const int l0 = wh.block * COLS, wl0 = l0 + 32 * w, l = wl0 + (lane & 31);
    const bf16_t* const kp = a.k + wh.g * a.kh + wh.b * a.kb;
    const bf16_t* const vp = a.v + wh.g * a.vh + wh.b * a.vb;
    const int s_end = a.causal ? min(a.S, l0 + COLS) : a.S;                    // keys that any query of the workgroup sees
    const int tiles = 2 * ((s_end + 2 * ROWS - 1) / (2 * ROWS));               // in pairs; rows past the end are zeros
    const int w_end = wl0 >= a.L ? 0 : a.causal ? min(a.S, wl0 + 32) : a.S;    // ... of the wave
    const int limit = a.causal ? min(l, a.S - 1) : a.S - 1;
    const FragRow fr;
    const FragT ft;
    bf16x8_v qf[2 * ET];
    load_columns<ET>(qf, a.q + wh.h * a.qh + wh.b * a.qb, (uint32_t)(a.qt * 2), l, a.L, a.E);
    if (a.negative) {
#pragma unroll
        for (int kk = 0; kk < 2 * ET; ++kk) qf[kk] = __builtin_bit_cast(bf16x8_v, __builtin_bit_cast(raw16_t, qf[kk]) ^ 0x80008000u);
    }

    // unscaled logits of keys s0 .. s0 + 31: -inf where masked
    auto logits = [&](const char* tile, int s0) {
        f32x16_v z = product<ET, 2 * ET>(fr, tile, qf);
        if (s0 + 31 > (a.causal ? min(wl0, a.S - 1) : a.S - 1)) {
#pragma unroll
            for (int i = 0; i < 16; ++i)
                if (s0 + acc_row(i, h) > limit) z[i] = -INFINITY;
        }
        return z;
    };
    // Exponentials are exp2(c z - off), off = c m rounded (m: a maximum, 0 in place of -inf): any number near c m serves as long as the
    // sum and the weights mean the same one, and the exponent is rounded once.  From 2^20 on, where the rounding itself grows large, they are
    // exp2(c (z - m)).  rest: what the offset lacks of c m.  A weight is its exponential times 1 / sum: log2(sum) in the exponent, a
    // multiplication less, doubles the exponent and with it the error of a weight (of 64 features, 745 tokens 4.4e-5 of the weights rounded the
    // other way, 1.6e-5 now, 2.2e-5 in the step-by-step softmax; forward 88 -> 91 us for 12 heads of 11 batches, 474 -> 478 causal 128 x 2048 x 32 x 4).
    struct Offset { float m, off, rest; bool far; };
    auto offset = [&](float m) {
        Offset o;
        o.m = m == -INFINITY ? 0.0f : m;
        o.off = o.m * a.c;
        o.far = __any(fabsf(o.off) > 0x1p20f);
        o.rest = o.far ? 0.0f : fmaf(o.m, a.c, -o.off);
        return o;
    };
    auto exponentials = [&](f32x16_v& z, const Offset& o) {
        if (o.far) {
#pragma unroll
            for (int i = 0; i < 16; ++i) z[i] = __builtin_amdgcn_exp2f((z[i] - o.m) * a.c);
        } else {
#pragma unroll
            for (int i = 0; i < 16; ++i) z[i] = __builtin_amdgcn_exp2f(fmaf(z[i], a.c, -o.off));
        }
    };
    // the logarithm of maximum m's exponential, and what takes a sum from one offset to another
    auto height = [&](float m, const Offset& o) { return fmaf(m - o.m, a.c, o.rest); };
    auto factor = [&](const Offset& from, const Offset& to) { return __builtin_amdgcn_exp2f(fmaf(from.m - to.m, a.c, to.rest - from.rest)); };

    // sweep 1: maximum of the unscaled logits and sum of exponentials, per lane (half of the keys of its column).  A column of which
    // nothing but -inf has been seen keeps the sum 0.  The offset moves when a lane's maximum is further than 2^8 from it, which is seldom
    // after the first tile.  lost: what the last addition rounded off; without it a long column's sum carries a rounding per tile.
    float m = -INFINITY, sum = 0.0f, lost = 0.0f;
    Offset at = {0.0f, 0.0f, 0.0f, false};
    {
        Tile<ET, 2> tk(kp, a.kt, a.E, a.S, 0);
        tk.load(0);
        tk.load(1);                                         // past the end: the last row once more
        tk.clear(lds);
        tk.clear(lds + TILE);
        tk.store(lds, 0, 0, a.S);
        __syncthreads();
        for (int t0 = 0; t0 < tiles; t0 += 2) {
            static_for<2>([&](auto U) {
                constexpr int u = decltype(U)::value;
                const int t = t0 + u;
                tk.load(u);
                if (ROWS * t < w_end) {
                    f32x16_v z = logits(lds + u * TILE, ROWS * t);
#pragma unroll
                    for (int i = 0; i < 16; ++i) m = fmaxf(m, z[i]);
                    if (__any(fabsf(height(m, at)) > 8.0f && m != -INFINITY)) {
                        const Offset to = offset(m);
                        const float f = factor(at, to);
                        sum = sum == 0.0f ? 0.0f : sum * f;         // an empty sum may be as far away as it likes
                        lost = lost == 0.0f ? 0.0f : lost * f;
                        at = to;
                    }
                    exponentials(z, at);
                    float add = -lost;
#pragma unroll
                    for (int i = 0; i < 16; ++i) add += z[i];
                    const float old = sum;
                    sum += add;
                    lost = (sum - old) - add;
                }
                tk.store(lds + (1 - u) * TILE, 1 - u, t + 1, a.S);
                __syncthreads();
            });
        }
    }
    // weight = exponential * inv, inv = 1 / sum (infinite where no key counts: the weights are NaN)
    const Offset top = offset(fmaxf(m, __shfl_xor(m, 32)));
    const float half = sum == 0.0f ? 0.0f : sum * factor(at, top), inv = 1.0f / (half + __shfl_xor(half, 32));

    // sweep 2: the weights, rounded, to memory and into the product with v
    bf16_t* const wrow0 = a.probs + ((int64_t)wh.head * a.L + wl0) * a.S;        // row wl0 of this head
    const WeightTile pt(lds + 4 * TILE, w);
    f32x16_v o[ET];
#pragma unroll
    for (int t = 0; t < ET; ++t) o[t] = zero16();
    {
        Tile<ET, 2> tk(kp, a.kt, a.E, a.S, 0), tv(vp, a.vt, a.Ev, a.S, 0);
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            tk.load(b);
            tv.load(b);
            tv.clear(lds + (2 + b) * TILE);
        }
        tk.store(lds, 0, 0, a.S);
        tv.store(lds + 2 * TILE, 0, 0, a.S);
        __syncthreads();
        // the finished 64 keys (or the first 32 of them) from s0 on
        auto store_weights = [&](int s0) {
            const int end = min(w_end, s0 + 64);
            pt.exchange();
            if (end == s0 + 64 && wl0 + 32 <= a.L) {        // uniform
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    *reinterpret_cast<raw16_u*>(wrow0 + (int64_t)pt.column(i) * a.S + s0 + pt.key()) = *pt.line(i);
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (wl0 + pt.column(i) < a.L && s0 + pt.key() < end)
                        store8(wrow0 + (int64_t)pt.column(i) * a.S, s0 + pt.key(), end, *pt.line(i));
            }
        };
        for (int t0 = 0; t0 < tiles; t0 += 2) {
            static_for<2>([&](auto U) {
                constexpr int u = decltype(U)::value;
                const int t = t0 + u;
                tk.load(u);
                tv.load(u);
                if (ROWS * t < w_end) {
                    f32x16_v z = logits(lds + u * TILE, ROWS * t);
                    bf16x8_v vf[2][ET];                 // read while the exponentials are computed
#pragma unroll
                    for (int n = 0; n < 2; ++n)
#pragma unroll
                        for (int e = 0; e < ET; ++e) vf[n][e] = ft.get(lds + (2 + u) * TILE, 16 * n, e);
                    __builtin_amdgcn_sched_barrier(0);
                    exponentials(z, top);
#pragma unroll
                    for (int i = 0; i < 16; ++i) z[i] *= inv;
#pragma unroll
                    for (int n = 0; n < 2; ++n) {
                        const raw16_t pw = pack8(z, n);
                        pt.put(2 * u + n, pw);
#pragma unroll
                        for (int e = 0; e < ET; ++e)
                            o[e] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[n][e], __builtin_bit_cast(bf16x8_v, pw), o[e], 0, 0, 0);
                    }
                }
                // the next tile first: its wait must not include this tile's stores
                tk.store(lds + (1 - u) * TILE, 1 - u, t + 1, a.S);
                tv.store(lds + (3 - u) * TILE, 1 - u, t + 1, a.S);
                if (u == 1 && ROWS * t0 < w_end) store_weights(ROWS * t0);
                __syncthreads();                        // and an exchange(): the next weights go over these
            });
        }
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
    // the masked part of the columns, last: nothing waits for these stores.  0, or NaN where 1 / sum is no number.
    const int rows = min(32, a.L - wl0);
    if (w_end < a.S) {
        for (int i = 0; i < rows; ++i) {
            const float z0 = 0.0f * __shfl(inv, i);
            const uint32_t zz = f32x2_to_bf16x2(z0, z0);
            const raw16_t zw = {zz, zz, zz, zz};
            for (int s = w_end + 8 * lane; s < a.S; s += 512) store8(wrow0 + (int64_t)i * a.S, s, a.S, zw);
        }
    }
}

// ------------------------------------------------------------------------------------------------ pullback
// scale weights .* (dP - d) of 16 rows, as the B operand of the next product: pw as loaded (bf16 pairs in accumulator
// order), d of each row.  The difference first: it may cancel, and fma(dP, scale, -scale d), an instruction less, leaves the rounding of scale d.
__device__ __forceinline__ raw16_t softmax_rule(raw16_t pw, const f32x16_v& dp, int n, const float (&d)[8], float scale) {
    raw16_t out;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float p0 = __uint_as_float(pw[i] << 16), p1 = __uint_as_float(pw[i] & 0xffff0000u);
        out[i] = f32x2_to_bf16x2(scale * p0 * (dp[8 * n + 2 * i] - d[2 * i]), scale * p1 * (dp[8 * n + 2 * i + 1] - d[2 * i + 1]));
    }
    return out;
}

// dq: a wave owns 32 queries and walks the keys.  VEC: rows of weights are whole 16-byte vectors (S a multiple of 8).
template <int ET, bool VEC>
__global__ __launch_bounds__(THREADS, 2) void dq_kernel(Args a) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    char* const lds = reinterpret_cast<char*>(lds_raw);     // k 0, k 1, v 0, v 1, weights
    const Where wh(a, a.causal ? REVERSE : FORWARD);
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5;
    const int l0 = wh.block * COLS, wl0 = l0 + 32 * w, l = wl0 + (lane & 31);
    const int s_end = a.causal ? min(a.S, l0 + COLS) : a.S;
    const int tiles = 2 * ((s_end + 2 * ROWS - 1) / (2 * ROWS));               // in pairs; rows past the end are zeros
    const int w_end = wl0 >= a.L ? 0 : a.causal ? min(a.S, wl0 + 32) : a.S;
    const int lc = min(l, a.L - 1);
    const FragRow fr;
    const FragT ft;
    // the weights of 64 keys, as they lie in memory, one such step ahead of their use
    const WeightTile pt(lds + 4 * TILE, w);
    raw16_t pw[4];
    const bf16_t* const wplane = a.probs + (int64_t)wh.head * a.L * a.S;
    const bf16_t* wrow[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) wrow[i] = wplane + (int64_t)min(wl0 + pt.column(i), a.L - 1) * a.S;
    auto load_weights = [&](int s0) {
        const int key = s0 + pt.key();
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if constexpr (VEC) pw[i] = *reinterpret_cast<const raw16_u*>(wrow[i] + min(key, a.S - 8));     // past the end: masked below
            else pw[i] = load8(wrow[i], key, w_end);
        }
    };
    Tile<ET, 2> tk(a.k + wh.g * a.kh + wh.b * a.kb, a.kt, a.E, a.S, 0), tv(a.v + wh.g * a.vh + wh.b * a.vb, a.vt, a.Ev, a.S, 0);
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        tk.load(b);
        tv.load(b);
    }
    load_weights(0);
    bf16x8_v df[2 * ET];
    load_columns<ET>(df, a.d_out + ((int64_t)wh.b * a.L * a.H + wh.h) * a.Ev, (uint32_t)(a.H * a.Ev * 2), l, a.L, a.Ev);
    // d = sum over the features of d_out .* out, half of them in each of a query's two lanes
    float dl;
    {
        float part[8] = {};                             // a long chain of additions would round as often
        const float* orow = a.out_wide + (((int64_t)wh.b * a.L + lc) * a.H + wh.h) * a.Ev;
#pragma unroll
        for (int kk = 0; kk < 2 * ET; ++kk) {
            const int e = 16 * kk + 8 * h;
            const float* p = orow + (e < a.Ev ? e : 0);
            const float4 x = *reinterpret_cast<const float4*>(p), y = *reinterpret_cast<const float4*>(p + 4);
            const float ov[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
            float dv[8];
            Vec<bf16_t>::unpack(__builtin_bit_cast(raw16_t, df[kk]), dv);
            if (e < a.Ev) {
#pragma unroll
                for (int i = 0; i < 8; ++i) part[i] = fmaf(dv[i], ov[i], part[i]);
            }
        }
        dl = ((part[0] + part[1]) + (part[2] + part[3])) + ((part[4] + part[5]) + (part[6] + part[7]));
        dl += __shfl_xor(dl, 32);
        if (h == 0 && l < a.L) a.dsum[(int64_t)wh.head * a.L + l] = dl;
    }
    const float dd[8] = {dl, dl, dl, dl, dl, dl, dl, dl};
    f32x16_v acc[ET];
#pragma unroll
    for (int t = 0; t < ET; ++t) acc[t] = zero16();
    tk.clear(lds);
    tk.clear(lds + TILE);
    tv.clear(lds + 2 * TILE);
    tv.clear(lds + 3 * TILE);
    tk.store(lds, 0, 0, a.S);
    tv.store(lds + 2 * TILE, 0, 0, a.S);
    __syncthreads();
    for (int t0 = 0; t0 < tiles; t0 += 2) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const raw16_t zero = {0u, 0u, 0u, 0u};
            *pt.line(i) = !VEC || ROWS * t0 + pt.key() < w_end ? pw[i] : zero;
        }
        pt.exchange();
        static_for<2>([&](auto U) {
            constexpr int u = decltype(U)::value;
            const int t = t0 + u;
            tk.load(u);
            tv.load(u);
            if (u == 0) load_weights(ROWS * (t + 2));
            if (ROWS * t < w_end) {
                const f32x16_v dp = product<ET, 2 * ET>(fr, lds + (2 + u) * TILE, df);
                bf16x8_v kf[2][ET];                     // read while the softmax rule is computed
#pragma unroll
                for (int n = 0; n < 2; ++n)
#pragma unroll
                    for (int e = 0; e < ET; ++e) kf[n][e] = ft.get(lds + u * TILE, 16 * n, e);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int n = 0; n < 2; ++n) {
                    const bf16x8_v ds = __builtin_bit_cast(bf16x8_v, softmax_rule(pt.get(2 * u + n), dp, n, dd, a.scale));
#pragma unroll
                    for (int e = 0; e < ET; ++e) acc[e] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[n][e], ds, acc[e], 0, 0, 0);
                }
            }
            tk.store(lds + (1 - u) * TILE, 1 - u, t + 1, a.S);
            tv.store(lds + (3 - u) * TILE, 1 - u, t + 1, a.S);
            __syncthreads();                            // and an exchange(): the next weights go over these
        });
    }
    store_features<ET>(acc, a.dq + wh.h * a.qh + wh.b * a.qb + (int64_t)lc * a.qt, l < a.L, a.E);
}

// dk, dv: a wave owns 32 keys and walks the queries.  VEC as above.
constexpr size_t DKV_LDS = 2 * (3 * TILE + ROWS * 4);           // q, d_out, weights (32 queries x 128 keys) and d, two of each: 63 KiB

template <int ET, bool VEC>
__global__ __launch_bounds__(THREADS, 2) void dkv_kernel(Args a) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    char* const lds = reinterpret_cast<char*>(lds_raw);         // q 0, q 1, d_out 0, 1, weights 0, 1, d 0, 1
    float* const dt = reinterpret_cast<float*>(lds + 6 * TILE);
    const Where wh(a, FORWARD);                                 // causal: the first block of keys is seen by every query
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5;
    const int s0 = wh.block * COLS, ws0 = s0 + 32 * w, s = ws0 + (lane & 31);
    const int first = a.causal ? s0 / ROWS : 0, tiles = 2 * ((a.L + 2 * ROWS - 1) / (2 * ROWS));     // first is even
    const int w_first = ws0 >= a.S ? tiles : a.causal ? ws0 / ROWS : 0;
    const FragRow fr;
    const FragT ft;
    Tile<ET, 1> tq(a.q + wh.h * a.qh + wh.b * a.qb, a.qt, a.E, a.L, first);
    Tile<ET, 1> to(a.d_out + ((int64_t)wh.b * a.L * a.H + wh.h) * a.Ev, (int64_t)a.H * a.Ev, a.Ev, a.L, first);
    // weights: 32 queries x 128 keys, two chunks of eight keys per thread
    raw16_t pw[2][2];
    float dv[2] = {0.0f, 0.0f};
    const int prow = threadIdx.x >> 4, pch = threadIdx.x & 15;
    const bf16_t* const wplane = a.probs + (int64_t)wh.head * a.L * a.S;
    const float* const dplane = a.d + (int64_t)wh.head * a.L;
    const int pkey = s0 + 8 * pch;
    auto load_weights = [&](int t, int set) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int r = t * ROWS + prow + 16 * i;
            const bf16_t* row = wplane + (int64_t)min(r, a.L - 1) * a.S;
            if constexpr (VEC) pw[set][i] = *reinterpret_cast<const raw16_u*>(row + min(pkey, a.S - 8));    // past the end: masked below
            else pw[set][i] = load8(row, pkey, r < a.L ? a.S : 0);
        }
        dv[set] = dplane[min(t * ROWS + ((int)threadIdx.x & 31), a.L - 1)];
    };
    auto store = [&](int t, int b) {
        tq.store(lds + b * TILE, 0, t, a.L);
        to.store(lds + (2 + b) * TILE, 0, t, a.L);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const raw16_t zero = {0u, 0u, 0u, 0u};
            const bool in = !VEC || (pkey < a.S && t * ROWS + prow + 16 * i < a.L);
            *reinterpret_cast<raw16_t*>(lds + (4 + b) * TILE + (prow + 16 * i) * PITCH + pch * 16) = in ? pw[b][i] : zero;
        }
        // 0 past the end: a non-finite d must not reach the keys through absent queries
        if (threadIdx.x < ROWS) dt[b * ROWS + threadIdx.x] = t * ROWS + (int)threadIdx.x < a.L ? dv[b] : 0.0f;
    };
    tq.load(0);
    to.load(0);
    load_weights(first, 0);
    load_weights(first + 1, 1);
    bf16x8_v vf[2 * ET];
    load_columns<ET>(vf, a.v + wh.g * a.vh + wh.b * a.vb, (uint32_t)(a.vt * 2), s, a.S, a.Ev);
    f32x16_v ak[ET], av[ET];
#pragma unroll
    for (int t = 0; t < ET; ++t) { ak[t] = zero16(); av[t] = zero16(); }
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        tq.clear(lds + b * TILE);
        to.clear(lds + (2 + b) * TILE);
    }
    if (first < tiles) store(first, 0);
    __syncthreads();
    for (int t0 = first; t0 < tiles; t0 += 2) {
        static_for<2>([&](auto U) {
            constexpr int u = decltype(U)::value;
            const int t = t0 + u;
            const char *qc = lds + u * TILE, *oc = lds + (2 + u) * TILE, *pc = lds + (4 + u) * TILE;
            tq.load(0);
            to.load(0);
            load_weights(t + 2, u);             // these come from memory, the others mostly from caches
            if (t >= w_first) {
                const f32x16_v dp = product<ET, 2>(fr, oc, vf);
#pragma unroll
                for (int n = 0; n < 2; ++n) {
                    const bf16x8_v pb = ft.get(pc, 16 * n, w);       // the wave's 32 keys are "features" 32 w .. of the weights' tile
#pragma unroll
                    for (int e = 0; e < ET; ++e) av[e] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ft.get(oc, 16 * n, e), pb, av[e], 0, 0, 0);
                    const float4 d0 = *reinterpret_cast<const float4*>(dt + u * ROWS + 16 * n + 4 * h);
                    const float4 d1 = *reinterpret_cast<const float4*>(dt + u * ROWS + 16 * n + 8 + 4 * h);
                    const float dd[8] = {d0.x, d0.y, d0.z, d0.w, d1.x, d1.y, d1.z, d1.w};
                    const bf16x8_v ds = __builtin_bit_cast(bf16x8_v, softmax_rule(__builtin_bit_cast(raw16_t, pb), dp, n, dd, a.scale));
#pragma unroll
                    for (int e = 0; e < ET; ++e) ak[e] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ft.get(qc, 16 * n, e), ds, ak[e], 0, 0, 0);
                }
            }
            store(t + 1, 1 - u);
            __syncthreads();
        });
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
template <int ET, bool VEC>
static int launch_bwd_as(hipStream_t s, Args& a) {
    static ResidentOnce ro;
    ro.get([&](hipError_t& err) {
        err = hipFuncSetAttribute(reinterpret_cast<const void*>(dq_kernel<ET, VEC>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)FWD_LDS);
        if (err == hipSuccess)
            err = hipFuncSetAttribute(reinterpret_cast<const void*>(dkv_kernel<ET, VEC>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)DKV_LDS);
        return 1;
    });
    LUX_CHECK_HIP(ro.error);
    {
        a.blocks = (int)ceil_div(a.L, COLS);
        ProfScope ps("attn_dq_kernel", s);
        dq_kernel<ET, VEC><<<dim3((unsigned)a.blocks * (unsigned)a.heads), dim3(THREADS), FWD_LDS, s>>>(a);
        LUX_CHECK_LAUNCH();
    }
    a.blocks = (int)ceil_div(a.S, COLS);
    ProfScope ps("attn_dkv_kernel", s);
    dkv_kernel<ET, VEC><<<dim3((unsigned)a.blocks * (unsigned)a.heads), dim3(THREADS), DKV_LDS, s>>>(a);
    LUX_CHECK_LAUNCH();
    return LUXHIP_OK;
}
template <int ET>
static int launch_bwd(hipStream_t s, Args& a) {
    return a.S % 8 == 0 ? launch_bwd_as<ET, true>(s, a) : launch_bwd_as<ET, false>(s, a);
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
    // at least the smallest normal number: a masked logit is -inf before it is scaled
    a.negative = scale < 0;
    a.c = (float)(std::abs(scale) * 1.4426950408889634);
    if (a.c < 1.2e-38f) a.c = 1.2e-38f;
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
    a.dsum = reinterpret_cast<float*>(ws.data);
    a.d = a.dsum;
    a.out_wide = const_cast<float*>(out_wide);
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
