// Products with few tiles or ragged operands, storage bf16: kernels of gemm_split.h and their launch.
#include "gemm_split_launch.h"
namespace luxhip {
template bool launch_split<bf16_t>(hipStream_t, DenseArgs<bf16_t>&, bool, bool, int*);
template bool launch_split_pair<bf16_t>(hipStream_t, DenseArgs<bf16_t>&, DenseArgs<bf16_t>&, int*);
double split_time_bf16(int64_t M, int64_t N, int64_t K) {
    const split::Choice c = split::choose<bf16_t>(M, N, K);
    return split::estimate<bf16_t>(c.w, c.slices, M, N, K);
}
}
