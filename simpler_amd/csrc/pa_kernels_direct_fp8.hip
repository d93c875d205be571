// Short-context decode kernels with fp8 E4M3FN caches (bf16 query, head dim 128).
#include "pa_kernels_direct.h"

namespace simpler_hip {
namespace pa {

DirectFn pick_direct_fp8(int bs, int d, int out_dtype) {
    if (d != 128) return DirectFn{};
    if (out_dtype == SIMPLER_HIP_DT_FLOAT32) return direct_by_block<128, float, true, __bf16>(bs);
    if (out_dtype == SIMPLER_HIP_DT_BFLOAT16) return direct_by_block<128, __bf16, true, __bf16>(bs);
    return DirectFn{};
}

}  // namespace pa
}  // namespace simpler_hip
