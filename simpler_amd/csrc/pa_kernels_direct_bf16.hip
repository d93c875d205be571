// Short-context decode kernels with bf16 query and caches (fp32 or bf16 output).
#include "pa_kernels_direct.h"

namespace simpler_hip {
namespace pa {

DirectFn pick_direct_bf16(int bs, int d, int out_dtype) {
    if (out_dtype == SIMPLER_HIP_DT_FLOAT32) return direct_by_dim<float, __bf16>(bs, d);
    if (out_dtype == SIMPLER_HIP_DT_BFLOAT16) return direct_by_dim<__bf16, __bf16>(bs, d);
    return DirectFn{};
}

}  // namespace pa
}  // namespace simpler_hip
