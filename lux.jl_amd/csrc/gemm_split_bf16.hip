// Products with few tiles or ragged operands, storage bf16: kernels of gemm_split.h and their launch.
#include "gemm_split_launch.h"
namespace luxhip {
template bool launch_split<bf16_t>(hipStream_t, DenseArgs<bf16_t>&, bool, bool, int*);
template bool launch_split_pair<bf16_t>(hipStream_t, DenseArgs<bf16_t>&, DenseArgs<bf16_t>&, int*);
}
