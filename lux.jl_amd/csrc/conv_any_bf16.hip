// Kernels of conv_any.h, storage bf16.
#include "conv_any_launch.h"
#include "conv_few.h"
namespace luxhip {
namespace cany {
template <int CPP>
static hipError_t run_few(hipStream_t s, const Args<bf16_t>& a, int tiles_a, int tiles_b, int tiles) {
    static ResidentOnce ro;
    ro.get([&](hipError_t& err) {
        err = hipFuncSetAttribute(reinterpret_cast<const void*>(conv_few_kernel<CPP>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)FEW_LDS);
        return 1;
    });
    if (ro.error != hipSuccess) return ro.error;
    const int cus = num_cus() > 0 ? num_cus() : 256;
    ProfScope ps("conv_dgrad_kernel<bf16>", s);
    conv_few_kernel<CPP><<<dim3((unsigned)std::min(tiles, cus)), dim3(FEW_THREADS), FEW_LDS, s>>>(a, tiles_a, tiles_b, tiles,
                                                                                                FastDiv((uint32_t)(FEW_A + a.sub[0].TW - 1)));
    return hipGetLastError();
}

// True if the problem is this kernel's, and then launched (*rc).  Fewer tiles than a quarter of the compute units stay on the
// gathers, which cut the contraction.
bool launch_few(hipStream_t s, const Args<bf16_t>& a, int* rc) {
    const Sub& q = a.sub[0];
    const int64_t cus = num_cus() > 0 ? num_cus() : 256;
    if (!a.merged || a.subs != 1 || a.Ncols > 32 || a.Cp > 64 || a.Cp % 16 != 0 || q.TW > FEW_TAPS || q.TH > FEW_TAPS || q.wstep != -1 || q.hstep != -1 ||
        q.K != q.TW * q.TH * a.Cp)
        return false;
    const int RB = q.RAB / q.RA, N = q.M / q.RAB, ta = (int)ceil_div(q.RA, FEW_A), tb = (int)ceil_div(RB, FEW_B);
    const int64_t tiles = (int64_t)ta * tb * N;
    if (tiles * 4 < cus || tiles >= (int64_t(1) << 31)) return false;
    // 32-bit offsets inside an image's planes
    if ((int64_t)a.Cch * a.PQ + (int64_t)a.os_h * a.P >= (int64_t(1) << 31) || a.os_w >= 32768 || a.os_h >= 32768) return false;
    hipError_t e;
    switch (a.Cp / 16) {
        case 1: e = run_few<2>(s, a, ta, tb, (int)tiles); break;
        case 2: e = run_few<4>(s, a, ta, tb, (int)tiles); break;
        case 3: e = run_few<6>(s, a, ta, tb, (int)tiles); break;
        default: e = run_few<8>(s, a, ta, tb, (int)tiles); break;
    }
    *rc = e == hipSuccess ? LUXHIP_OK : set_error(LUXHIP_HIP_ERROR, "conv: kernel launch failed: %s", hipGetErrorString(e));
    return true;
}

template Choice choose_any<bf16_t>(Sub*, int, int, int, bool);
template int launch_any<bf16_t>(hipStream_t, Args<bf16_t>&, int, size_t, bool, bool);
template int launch_any_wgrad<bf16_t>(hipStream_t, WgradArgs<bf16_t>&, int, bool);
}
}
