// Explicit instantiation: storage bf16, A K-major, B K-major; and the 256 x 256 kernel of gemm_kk256.h.
#include "gemm_dense.h"
#include "gemm_kk256.h"
namespace luxhip {
bool launch_kk256_if_applicable(hipStream_t s, DenseArgs<bf16_t>& a, int* rc) {
    if (!kk256::applicable(a)) return false;
    *rc = kk256::launch(s, a);
    return true;
}
size_t kk256_partial_bytes(int64_t M, int64_t N, int slices) { return kk256::partial_bytes(M, N, slices); }
int launch_kk256_sliced(hipStream_t s, DenseArgs<bf16_t>& a, int slices, float* partial) {
    if (!kk256::applicable(a) || slices < 1 || a.K / kk256::BK < 2 * slices)
        return set_error(LUXHIP_INVALID, "launch_kk256_sliced: not a problem of the 256 x 256 kernel");
    return kk256::launch(s, a, slices, partial);
}
template int launch_layout<bf16_t, true, true>(hipStream_t, DenseArgs<bf16_t>&);
template int launch_batched_layout<bf16_t, true, true>(hipStream_t, DenseArgs<bf16_t>&);
}
