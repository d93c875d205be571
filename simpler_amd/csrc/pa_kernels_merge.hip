// Split-merge kernels (pa_merge_kernel) for every output width and dtype the
// decode kernels produce.
#include "pa_kernels.h"

namespace simpler_hip {
namespace pa {
namespace {

template <int DV, typename OutT>
MergeFn merge_set() {  // a tile of 16 rows has 4 DV units
    if constexpr (DV > 256)
        return {{pa_merge_kernel<DV, OutT, 1>, pa_merge_kernel<DV, OutT, 2>, pa_merge_kernel<DV, OutT, 4>}};
    else if constexpr (DV > 128)
        return {{pa_merge_kernel<DV, OutT, 1>, pa_merge_kernel<DV, OutT, 2>, nullptr}};
    else
        return {{pa_merge_kernel<DV, OutT, 1>, nullptr, nullptr}};
}

template <int DV>
MergeFn merge_for(int out_dtype) {
    switch (out_dtype) {
        case SIMPLER_HIP_DT_FLOAT32: return merge_set<DV, float>();
        case SIMPLER_HIP_DT_BFLOAT16: return merge_set<DV, __bf16>();
        case SIMPLER_HIP_DT_FLOAT16: return merge_set<DV, _Float16>();
        default: return MergeFn{};
    }
}

}  // namespace

MergeFn pick_merge(int dv, int out_dtype) {
    switch (dv) {
        case 16: return merge_for<16>(out_dtype);
        case 32: return merge_for<32>(out_dtype);
        case 64: return merge_for<64>(out_dtype);
        case 128: return merge_for<128>(out_dtype);
        case 256: return merge_for<256>(out_dtype);
        case kMlaDv: return merge_for<kMlaDv>(out_dtype);
        default: return MergeFn{};
    }
}

}  // namespace pa
}  // namespace simpler_hip
