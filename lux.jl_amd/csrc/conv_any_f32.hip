// Kernels of conv_any.h, storage f32.
#include "conv_any_launch.h"
namespace luxhip {
namespace cany {
template Choice choose_any<float>(Sub*, int, int, int, bool);
template int launch_any<float>(hipStream_t, Args<float>&, int, size_t, bool, bool);
template int launch_any_wgrad<float>(hipStream_t, WgradArgs<float>&, int, bool);
}
}
