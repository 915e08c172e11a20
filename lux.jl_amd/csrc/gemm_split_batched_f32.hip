// Choice and launch of gemm_split_batched.h
#include "gemm_split_batched.h"

namespace luxhip {
namespace split {

// Slices of the contraction: as many as shorten the launch by the constants of estimate() (gemm_split_launch.h)
static int batched_slices(int64_t tiles, int64_t K, int structure) {
    const int64_t cus = num_cus() > 0 ? num_cus() : 256;
    int best = 1;
    double t_best = 1e30;
    for (int s = 1; s <= 8 && (s == 1 || K / s >= 64); ++s) {
        const double k = (double)ceil_div(K, s), work = structure >= 2 ? 0.5 : 1.0;
        double t = std::max(k * 24e-3, std::max(1.0, (double)tiles * s * work / (double)cus) * k * 19e-3);
        if (s > 1) t += 1.5 + 0.5 * s + (double)tiles * s * work * (64.0 * 64.0 * 8.0) / 5e6;
        if (t < t_best) { t_best = t; best = s; }
    }
    return best;
}

template <bool AK, bool BKM, bool EP>
static int launch_batched_as(hipStream_t s, DenseArgs<float>& a, int64_t units, const Plan& p) {
    using B = Body<float, 1, AK, BKM>;
    ProfScope ps(EP ? "split_batched_kernel+softmax_rule" : p.slices > 1 ? "split_batched_kernel+slices" : "split_batched_kernel", s);
    split_batched_kernel<float, AK, BKM, EP><<<dim3((unsigned)units), dim3(THREADS), B::LDS_BYTES, s>>>(a, p);
    LUX_CHECK_LAUNCH();
    return LUXHIP_OK;
}

}  // namespace split

// Everything but whole aligned 128 x 128 tiles that fill the chip once: those read each operand half as often (us, in such tiles / here: 512^3 x 16 48 / 52,
// 1024^3 x 8 154 / 174, 2048 x 2048 x 64 x 16 102 / 135; with fewer of them 1024^3 x 2 77 / 56, 128 x 2048 x 2048 x 8 144 / 93, 512^3 x 4 42 / 22).
// Ragged: 97 x 1001 x 1001 x 8 49 / 35, 1000 x 1000 x 100 x 4 24 / 19.  Attention of 128 features: 2 heads x 448 tokens x 7 254 / 108, 16 x 832 causal 486 / 207,
// 8 x 2048 causal 848 / 483.
bool launch_split_batched(hipStream_t s, DenseArgs<float>& a, bool ak, bool bk, int* rc) {
    using namespace split;
    using Tr = GemmTraits<float>;
    const bool ep = a.ep_probs != nullptr;
    if (a.M < Tr::VEC || a.N < Tr::VEC || a.K < Tr::BK || (ep && !(ak && bk))) return false;
    const int64_t lim = (int64_t(1) << 31) / (256 * (int64_t)sizeof(float));
    if (std::max(a.A.sr, a.A.sk) >= lim || std::max(a.B.sr, a.B.sk) >= lim) return false;
    const int64_t tiles = ceil_div(a.M, 64) * ceil_div(a.N, 64) * a.batch;
    const int64_t cus = num_cus() > 0 ? num_cus() : 256;
    if (whole_tiles<float, 128, 128>(a) && (int64_t)(a.M / 128) * (a.N / 128) * a.batch * 10 >= cus * 9) return false;
    a.tiles_m = (int)ceil_div(a.M, 64);
    a.tiles_n = (int)ceil_div(a.N, 64);
    int slices = ep || a.structure == 1 || tiles > (int64_t)kWorkspaceCounters ? 1 : batched_slices(tiles, a.K, a.structure);
    if (tiles * slices * THREADS >= kMostThreads) return false;
    Plan p{1, a.K, nullptr, nullptr};
    const size_t bytes = (size_t)tiles * slices * 64 * 64 * sizeof(float);
    if (slices > 1 && workspace_holds(s, bytes)) {
        Workspace ws;
        *rc = get_workspace(s, bytes, &ws);
        if (*rc != LUXHIP_OK) return true;
        p.kslice = (int)(ceil_div(ceil_div(a.K, slices), Tr::BK) * Tr::BK);
        p.slices = (int)ceil_div(a.K, p.kslice);
        p.partial = reinterpret_cast<float*>(ws.data);
        p.counters = ws.counters;
    }
    const int64_t units = tiles * p.slices;
    if (ep) *rc = launch_batched_as<true, true, true>(s, a, units, p);
    else if (ak && bk) *rc = launch_batched_as<true, true, false>(s, a, units, p);
    else if (ak) *rc = launch_batched_as<true, false, false>(s, a, units, p);
    else if (bk) *rc = launch_batched_as<false, true, false>(s, a, units, p);
    else *rc = launch_batched_as<false, false, false>(s, a, units, p);
    return true;
}

}  // namespace luxhip
