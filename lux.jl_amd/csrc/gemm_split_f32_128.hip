// 128 x 128 tiles of gemm_split.h, storage f32.
#include "gemm_split_launch.h"
namespace luxhip {
namespace split {
template int launch_layouts<float, 2>(hipStream_t, DenseArgs<float>&, bool, bool, int);
}
}
