// Products with few tiles or ragged operands, storage f32: kernels of gemm_split.h and their launch.
#include "gemm_split_launch.h"
namespace luxhip {
template bool launch_split<float>(hipStream_t, DenseArgs<float>&, bool, bool, int*);
template bool launch_split_pair<float>(hipStream_t, DenseArgs<float>&, DenseArgs<float>&, int*);
}
