// MLA decode kernels (Dk 576, Dv 512, V a prefix of K; bf16): block sizes 32
// and 64, fp32 or bf16 output. The fused KV append runs as a launch of its own
// ahead of these (simpler_hip_pa_decode_append).
#include "pa_kernels.h"

namespace simpler_hip {
namespace pa {

namespace {

template <int BS, typename OutT>
KernelPair mla_set() {
    return {pa_mla_kernel<BS, kMlaDk, kMlaDv, OutT>, pa_mla_kernel<BS, kMlaDk, kMlaDv, OutT, 1>, true, false,
            pa_mla_kernel<BS, kMlaDk, kMlaDv, OutT, 2>};
}

}  // namespace

KernelPair pick_mla(int bs, int out_dtype) {
    const bool f32 = out_dtype == SIMPLER_HIP_DT_FLOAT32, b16 = out_dtype == SIMPLER_HIP_DT_BFLOAT16;
    if (bs == 32 && f32) return mla_set<32, float>();
    if (bs == 32 && b16) return mla_set<32, __bf16>();
    if (bs == 64 && f32) return mla_set<64, float>();
    if (bs == 64 && b16) return mla_set<64, __bf16>();
    return KernelPair{};
}

}  // namespace pa
}  // namespace simpler_hip
