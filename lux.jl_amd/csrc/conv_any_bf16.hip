// Kernels of conv_any.h, storage bf16.
#include "conv_any_launch.h"
namespace luxhip {
namespace cany {
template Choice choose_any<bf16_t>(Sub*, int, int, int, bool);
template int launch_any<bf16_t>(hipStream_t, Args<bf16_t>&, int, size_t, bool, bool);
template int launch_any_wgrad<bf16_t>(hipStream_t, WgradArgs<bf16_t>&, int, bool);
}
}
