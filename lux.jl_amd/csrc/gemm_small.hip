// Products that are too small to fill the chip in tiles of 64 x 64: the contraction is divided among the waves of a workgroup, and the whole
// pullback of such a dense layer is one launch.
//
// What bounds them is latency and, in a program of small layers, the host: a launch costs it about 3 us.  A 64 x 64 tile of gemm_split.h
// takes a trip to memory, two barriers and an LDS round trip per stage and an epilogue of 16 values per lane; where K is cut over
// workgroups, another 3 us to hand partial sums over.  Here
//   * a workgroup of eight waves takes a tile of 32 x 32, and each wave an eighth of K for the whole tile: no LDS and no barrier
//     before the sums, and a wave requests its next 32 k before it multiplies the present ones;
//   * lanes load fragments of v_mfma_f32_32x32x2_f32 straight from memory: four k in one load along k, or one value of each k along m or n.
//     Any order of k does, if both operands agree on it: instruction j of eight k takes k0 + j in the lower and k0 + 4 + j in
//     the upper half of the wave.  bf16 values are widened; their products are exact in fp32 and are added in fp32 as everywhere;
//   * the eight sums meet in LDS, in wave order (the same sum on every run), and each thread finishes two values next to each other along m;
//   * the pullback forms dz = delta .* act'(y, pre) as it loads fragments, for either product, and the workgroups of the first
//     column of dW add it up for the bias gradient: no pass for dz, no partial sums.
// A tile that sticks out of the matrix clamps its rows.  The last eight k are moved back until they end with K, and what they repeat is
// zero in both operands.
//
// Measured (us in a captured graph, before / now): fp32 512 x 512 x 512 10.9 / 6.8, 256 x 64 x 128 5.8 / 3.6, 1024 x 512 x 256 9.2 / 7.2; pullback of 128 -> 256
// with 64 columns and tanh 12.2 / 5.5, of 256 -> 256 with 256 and gelu in bf16 13.0 / 7.3.
#include "act_vec.h"
#include "gemm_split_launch.h"

namespace luxhip {
namespace small {

constexpr int WAVES = 8, THREADS = WAVES * 64, TILE = 32;
constexpr int GROUP = 4;                                       // steps of eight k per trip to memory
constexpr int PITCH = TILE + 4;                                // floats between the columns of a tile in LDS

// Values of eight k of an operand as a lane has them: row r, k = k0 + 4 h + j of lane 32 h + r
template <typename T, bool KMAJOR>
struct Place {
    int64_t first, k_step;     // uniform, in elements: (r0, k = 0), and between k
    uint32_t voff;             // per thread, in bytes
    __device__ __forceinline__ Place(int64_t sr, int64_t sk, int rows, int r0) {
        const int l = threadIdx.x & 63, r = min(l & 31, rows - 1 - r0), h = l >> 5;
        first = KMAJOR ? (int64_t)r0 * sr : (int64_t)r0;
        k_step = KMAJOR ? 1 : sk;
        voff = (uint32_t)(((int64_t)r * (KMAJOR ? sr : 1) + (int64_t)(4 * h) * k_step) * (int64_t)sizeof(T));
    }
    __device__ __forceinline__ void load(const T* p, int k, float (&v)[4]) const {
        const char* base = reinterpret_cast<const char*>(p + first + k * k_step);
        if constexpr (KMAJOR && sizeof(T) == 4) {
            const u32x4_v x = *reinterpret_cast<const UnalignedVec<float>::type*>(base + voff);
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = __uint_as_float(x[j]);
        } else if constexpr (KMAJOR) {
            typedef uint32_t pair __attribute__((ext_vector_type(2), aligned(2)));
            const pair x = *reinterpret_cast<const pair*>(base + voff);
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = __uint_as_float((j & 1) ? x[j / 2] & 0xffff0000u : x[j / 2] << 16);
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = ld(reinterpret_cast<const T*>(base + (int64_t)j * k_step * (int64_t)sizeof(T) + voff));
        }
    }
};

// An operand as it is
template <typename T, bool KMAJOR>
struct Plain {
    struct Raw { float v[4]; };
    const T* p;
    Place<T, KMAJOR> at;
    __device__ __forceinline__ Plain(const Operand<T>& op, int r0) : p(op.p), at(op.sr, op.sk, op.rows, r0) {}
    __device__ __forceinline__ void load(int k, Raw& x) const { at.load(p, k, x.v); }
    __device__ __forceinline__ void value(Raw& x, float (&v)[4], int skip) const {
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = x.v[j];
        drop(v, skip);
    }
    // skip: leading k of the eight that are to count as zero
    __device__ __forceinline__ static void drop(float (&v)[4], int skip) {
        if (skip > 0) {
            const int h4 = (threadIdx.x & 32) >> 3;
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = h4 + j < skip ? 0.0f : v[j];
        }
    }
};

// dz = delta .* act'(y, pre), rounded to the storage type for the products and added up unrounded
template <typename T, int ACT, bool KMAJOR>
struct Cotangent {
    static constexpr bool AUX = ACT != LUXHIP_ACT_IDENTITY;
    struct Raw { float d[4], a[AUX ? 4 : 1]; };
    const T *delta, *aux;      // aux: the pre-activation where the derivative needs it, else y
    Place<T, KMAJOR> at;
    float sum;
    __device__ __forceinline__ Cotangent(const T* d, const T* a, int64_t M, int rows, int r0)
        : delta(d), aux(a), at(KMAJOR ? M : 1, KMAJOR ? 1 : M, rows, r0), sum(0.0f) {}
    __device__ __forceinline__ void load(int k, Raw& x) const {
        at.load(delta, k, x.d);
        if constexpr (AUX) at.load(aux, k, x.a);
    }
    __device__ __forceinline__ void value(Raw& x, float (&v)[4], int skip) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if constexpr (!AUX) v[j] = x.d[j];
            else if constexpr (Act<ACT>::needs_pre) v[j] = x.d[j] * Act<ACT>::d(Act<ACT>::f(x.a[j]), x.a[j]);
            else v[j] = x.d[j] * Act<ACT>::d(x.a[j], 0.0f);
        }
        Plain<T, KMAJOR>::drop(v, skip);
        sum += (v[0] + v[1]) + (v[2] + v[3]);
        if constexpr (sizeof(T) == 2 && AUX) {
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = bf16_to_f32(f32_to_bf16(v[j]));
        }
    }
};

// This wave's share of a tile: k [kbeg, kend) of K (at least 8)
template <class LA, class LB>
__device__ __forceinline__ void multiply(LA& la, LB& lb, int K, f32x16_v& acc) {
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kwave = ((K + WAVES * 8 - 1) / (WAVES * 8)) * 8, kbeg = w * kwave, kend = min(kbeg + kwave, K);
#pragma unroll
    for (int q = 0; q < 16; ++q) acc[q] = 0.0f;
    typename LA::Raw ra[2][GROUP];
    typename LB::Raw rb[2][GROUP];
    auto fetch_group = [&](int k0, auto BUF) {
#pragma unroll
        for (int g = 0; g < GROUP; ++g)
            if (k0 + 8 * g < kend) {                                    // uniform
                const int k = min(k0 + 8 * g, K - 8);
                la.load(k, ra[BUF][g]);
                lb.load(k, rb[BUF][g]);
            }
    };
    auto use_group = [&](int k0, auto BUF) {
#pragma unroll
        for (int g = 0; g < GROUP; ++g)
            if (k0 + 8 * g < kend) {
                const int skip = k0 + 8 * g + 8 - K;
                float fa[4], fb[4];
                la.value(ra[BUF][g], fa, skip);
                lb.value(rb[BUF][g], fb, skip);
#pragma unroll
                for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[j], fb[j], acc, 0, 0, 0);
            }
    };
    constexpr std::integral_constant<int, 0> even{};
    constexpr std::integral_constant<int, 1> odd{};
    constexpr int STEP = 8 * GROUP;
    fetch_group(kbeg, even);
    for (int k0 = kbeg; k0 < kend; k0 += 2 * STEP) {
        fetch_group(k0 + STEP, odd);
        use_group(k0, even);
        fetch_group(k0 + 2 * STEP, even);
        use_group(k0 + STEP, odd);
    }
}

// The eight waves' sums -> LDS -> done(m, n, values of m and m + 1)
template <class Done>
__device__ __forceinline__ void finish(const f32x16_v& acc, int M, int N, int m0, int n0, float* lds, Done&& done) {
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63, r = l & 31, h = l >> 5;
    // acc[q]: m = 8 (q / 4) + 4 h + q % 4, n = r
    float* mine = lds + w * TILE * PITCH + r * PITCH + 4 * h;
#pragma unroll
    for (int q = 0; q < 16; ++q) mine[8 * (q / 4) + q % 4] = acc[q];
    __syncthreads();
    const int e = threadIdx.x * 2, nl = e / TILE, ml = e % TILE;
    float v[2] = {0.0f, 0.0f};
#pragma unroll
    for (int s = 0; s < WAVES; ++s) {
        v[0] += lds[(s * TILE + nl) * PITCH + ml];
        v[1] += lds[(s * TILE + nl) * PITCH + ml + 1];
    }
    if (m0 + ml < M && n0 + nl < N) done(m0 + ml, n0 + nl, v);
}

template <typename T>
__device__ __forceinline__ void store_two(T* C, int64_t ldc, int M, int m, int n, const float (&v)[2]) {
    T* p = C + (int64_t)n * ldc + m;
    st(p, v[0]);
    if (m + 1 < M) st(p + 1, v[1]);
}

template <bool AK, bool BKM>
__global__ __launch_bounds__(THREADS) void small_gemm_kernel(DenseArgs<float> a) {
    __shared__ __align__(16) float lds[WAVES * TILE * PITCH];
    int tm, tn;
    tile_coords(blockIdx.x, a.tiles_m, a.tiles_n, tm, tn);
    const int m0 = tm * TILE, n0 = tn * TILE;
    Plain<float, AK> la(a.A, m0);
    Plain<float, BKM> lb(a.B, n0);
    f32x16_v acc;
    multiply(la, lb, a.K, acc);
    finish(acc, a.M, a.N, m0, n0, lds, [&](int m, int n, float (&v)[2]) {
        if (a.bias) {
            v[0] += ld(a.bias + m);
            v[1] += ld(a.bias + min(m + 1, a.M - 1));
        }
        if (a.pre) store_two(a.pre, a.ldc, a.M, m, n, v);
        act_vec(a.act, v);
        store_two(a.C, a.ldc, a.M, m, n, v);
    });
}

// The pullback of y (M x N) = act.(W (M x K) x (K x N) .+ b): workgroups [0, first) compute the product of the longer contraction, the rest the other.
template <typename T>
struct LayerArgs {
    const T *delta, *aux;
    Operand<T> W, x;           // W as K rows along m, x as K rows along n
    T *dW, *dx, *dbias;        // dbias may be null
    int M, K, N, first, weights_first;
};
template <typename T, int ACT>
__global__ __launch_bounds__(THREADS) void small_layer_bwd_kernel(LayerArgs<T> a) {
    __shared__ __align__(16) float lds[WAVES * TILE * PITCH];
    __shared__ float bsum[WAVES][TILE];
    const bool front = (int)blockIdx.x < a.first, weights = front == (a.weights_first != 0);
    const int id = front ? blockIdx.x : blockIdx.x - a.first;
    int tm, tn;
    f32x16_v acc;
    if (weights) {             // dW (M x K) = dz (M x N) * x'
        tile_coords(id, (a.M + TILE - 1) / TILE, (a.K + TILE - 1) / TILE, tm, tn);
        const int m0 = tm * TILE, n0 = tn * TILE;
        Cotangent<T, ACT, false> la(a.delta, a.aux, a.M, a.M, m0);
        Plain<T, false> lb(a.x, n0);
        multiply(la, lb, a.N, acc);
        if (tn == 0 && a.dbias != nullptr) {                            // uniform
            const float s = la.sum + __shfl_xor(la.sum, 32);
            if ((threadIdx.x & 63) < TILE) bsum[threadIdx.x >> 6][threadIdx.x & 63] = s;
        }
        finish(acc, a.M, a.K, m0, n0, lds, [&](int m, int n, float (&v)[2]) { store_two(a.dW, a.M, a.M, m, n, v); });
        if (tn == 0 && a.dbias != nullptr && (int)threadIdx.x < TILE && m0 + (int)threadIdx.x < a.M) {
            float t = 0.0f;
#pragma unroll
            for (int s = 0; s < WAVES; ++s) t += bsum[s][threadIdx.x];
            st(a.dbias + m0 + threadIdx.x, t);
        }
    } else {                   // dx (K x N) = W' * dz
        tile_coords(id, (a.K + TILE - 1) / TILE, (a.N + TILE - 1) / TILE, tm, tn);
        const int m0 = tm * TILE, n0 = tn * TILE;
        Plain<T, true> la(a.W, m0);
        Cotangent<T, ACT, true> lb(a.delta, a.aux, a.M, a.N, n0);
        multiply(la, lb, a.M, acc);
        finish(acc, a.K, a.N, m0, n0, lds, [&](int m, int n, float (&v)[2]) { store_two(a.dx, a.K, a.K, m, n, v); });
    }
}

// Time of one workgroup in microseconds: its ends, and k of a tile at `per_k` ns
static double tile_time(int64_t K, double per_k) { return 0.6 + (double)K * per_k * 1e-3; }

// Whether the product is faster here: by this estimate of its time against that of gemm_split.h, whose launch the 2.3 stand for.  A k of
// a tile costs 7 ns whether one workgroup or 256 are at work (its loads: 37 bytes per ns of a compute unit), and every further 256 tiles a round.
// Of 45 products of 16 to 2048 in every dimension (us, there / here): 112 x 1064 x 636 10.5 / 7.4, 363 x 438 x 1127 13.7 / 11.9, 48 x 752 x 128
// 7.6 / 3.7; on the other side 1024 x 1024 x 64 4.9 / 6.9, 256 x 128 x 2048 13.5 / 17.2.  bf16 products, half of whose loads along m or n would be two bytes a
// lane here, keep to gemm_split.h (512 x 512 x 128 3.6 / 4.0, 517 x 301 x 1023 8.7 / 13.3).
static bool product_pays(const DenseArgs<float>& a, bool ak) {
    const int64_t cus = num_cus() > 0 ? num_cus() : 256, tiles = ceil_div(a.M, TILE) * ceil_div(a.N, TILE);
    const split::Choice c = split::choose<float>(a.M, a.N, a.K);
    return 2.1 + (double)ceil_div(tiles, cus) * tile_time(a.K, ak ? 8.0 : 7.2) < split::estimate<float>(c.w, c.slices, a.M, a.N, a.K) + 2.3;
}

// Whether the whole pullback is one launch: up to a constant of its own estimated time, not by an estimate of the other way (past the constants some
// layers that would gain stay with the passes: 1023 -> 517 with 301 columns and gelu is 20.6 by this estimate, 25 in three launches).  The longer of
// the two contractions starts first, and where the tiles are more than the compute units its last ones end half a tile late.  Fitted to 60 layers of 16 to 2048 in every dimension with tanh and gelu (within 11 % rms).  Of those none below the limit was
// slower than the passes over delta and the pair of products in graphs, where the host does not count (us, there / here: fp32, gelu
// 301 x 77 x 560 14.0 / 6.6, 641 x 496 x 240 20.7 / 15.6, 1339 x 56 x 53 16.4 / 17.3; bf16 288 x 176 x 634 12.1 / 9.2, 567 x 67 x 178 12.9 / 13.2).
template <typename T>
static bool pullback_pays(int act, int64_t M, int64_t K, int64_t N) {
    const int64_t cus = num_cus() > 0 ? num_cus() : 256;
    const double per_k = sizeof(T) == 4 ? (act_needs_pre(act) ? 10.3 : 8.2) : (act_needs_pre(act) ? 12.0 : 9.0), limit = sizeof(T) == 4 ? 15.0 : 9.5;
    const int64_t tiles_w = ceil_div(M, TILE) * ceil_div(K, TILE), tiles_x = ceil_div(K, TILE) * ceil_div(N, TILE);
    const double longest = tile_time(std::max(M, N), per_k);
    double t = longest;
    if (tiles_w + tiles_x > cus)
        t = std::max(t, ((double)tiles_w * tile_time(N, per_k) + (double)tiles_x * tile_time(M, per_k)) / (double)cus + 0.5 * longest);
    return 2.4 + t <= limit;
}

}  // namespace small

bool launch_small(hipStream_t s, DenseArgs<float>& a, bool ak, bool bk, int* rc) {
    if (a.M < 1 || a.N < 1 || a.K < 8 || !small::product_pays(a, ak)) return false;
    a.tiles_m = (int)ceil_div(a.M, small::TILE);
    a.tiles_n = (int)ceil_div(a.N, small::TILE);
    const dim3 grid((unsigned)(a.tiles_m * a.tiles_n)), block(small::THREADS);
    ProfScope ps("small_gemm_kernel", s);
    if (ak && bk) small::small_gemm_kernel<true, true><<<grid, block, 0, s>>>(a);
    else if (ak) small::small_gemm_kernel<true, false><<<grid, block, 0, s>>>(a);
    else if (bk) small::small_gemm_kernel<false, true><<<grid, block, 0, s>>>(a);
    else small::small_gemm_kernel<false, false><<<grid, block, 0, s>>>(a);
    const hipError_t e = hipGetLastError();
    *rc = e == hipSuccess ? LUXHIP_OK : set_error(LUXHIP_HIP_ERROR, "kernel launch failed: %s", hipGetErrorString(e));
    return true;
}

template <typename T>
bool launch_small_layer_bwd(hipStream_t s, int act, int64_t M, int64_t K, int64_t N, const T* delta, const T* y, const T* pre, const T* W, int64_t ldw,
                            const T* x, int64_t ldx, T* dW, T* dx, T* dbias, int* rc) {
    // fragments lie up to 31 rows and 16 k apart in 32 bits
    if (M < 8 || N < 8 || K < 1 || std::max(ldw, ldx) >= (int64_t(1) << 24) || !small::pullback_pays<T>(act, M, K, N)) return false;
    const int64_t tk = ceil_div(K, small::TILE), tiles_w = ceil_div(M, small::TILE) * tk, tiles_x = tk * ceil_div(N, small::TILE);
    const bool weights_first = N >= M;
    small::LayerArgs<T> a{delta, act_needs_pre(act) ? pre : y, Operand<T>{W, ldw, 1, (int)K, 0}, Operand<T>{x, 1, ldx, (int)K, 0}, dW, dx, dbias,
                          (int)M, (int)K, (int)N, (int)(weights_first ? tiles_w : tiles_x), weights_first};
    const dim3 grid((unsigned)(tiles_w + tiles_x)), block(small::THREADS);
    ProfScope ps("small_layer_bwd_kernel", s);
#define LAUNCH_SMALL_BWD(A) small::small_layer_bwd_kernel<T, A><<<grid, block, 0, s>>>(a)
    LUX_DISPATCH_ACT(act, LAUNCH_SMALL_BWD);
#undef LAUNCH_SMALL_BWD
    const hipError_t e = hipGetLastError();
    *rc = e == hipSuccess ? LUXHIP_OK : set_error(LUXHIP_HIP_ERROR, "kernel launch failed: %s", hipGetErrorString(e));
    return true;
}
template bool launch_small_layer_bwd<float>(hipStream_t, int, int64_t, int64_t, int64_t, const float*, const float*, const float*, const float*, int64_t,
                                            const float*, int64_t, float*, float*, float*, int*);
template bool launch_small_layer_bwd<bf16_t>(hipStream_t, int, int64_t, int64_t, int64_t, const bf16_t*, const bf16_t*, const bf16_t*, const bf16_t*,
                                             int64_t, const bf16_t*, int64_t, bf16_t*, bf16_t*, bf16_t*, int*);

}  // namespace luxhip
