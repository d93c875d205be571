// Short-context decode kernels with f16 query and caches (fp32 or f16 output).
#include "pa_kernels_direct.h"

namespace simpler_hip {
namespace pa {

DirectFn pick_direct_f16(int bs, int d, int out_dtype) {
    if (out_dtype == SIMPLER_HIP_DT_FLOAT32) return direct_by_dim<float, _Float16>(bs, d);
    if (out_dtype == SIMPLER_HIP_DT_FLOAT16) return direct_by_dim<_Float16, _Float16>(bs, d);
    return DirectFn{};
}

}  // namespace pa
}  // namespace simpler_hip
