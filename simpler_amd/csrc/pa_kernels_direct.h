// GQA decode of short contexts: one workgroup per 16-row tile (batch, kv head,
// row tile), its KV blocks shared out among the workgroup's waves in
// contiguous runs, which meet in LDS. There is no work list and no merge
// launch: a small decode is bound by latency, i.e. by launches and by the
// chain of dependent loads, and here the chain is the length and the block
// table (both at addresses known from the block index), K and V, the store.
// The waves run the decode kernel's own segments (run_segment).
#pragma once

#include "pa_kernels.h"

namespace simpler_hip {
namespace pa {

// LDS of one wave: its K buffer (K staged through LDS), reused for its partial
// (O of 16 rows, then m and l).
template <int BS, int D, bool KV8>
constexpr int direct_wave_lds() {
    constexpr int part = 16 * D * 4 + 32 * 4, k = (!KV8 && D == 128) ? BS * 256 : 0;
    return part > k ? part : k;
}

// Most waves per workgroup: what the segment's registers leave room for.
template <int BS, int D>
constexpr int direct_max_waves() {
    if (BS == 16) return D <= 64 ? 16 : 8;
    return (BS == 32 && D <= 128) || (BS == 64 && D <= 64) ? 8 : 4;
}

template <int BS, int D, typename OutT, bool KV8, typename ET>
__global__ void __launch_bounds__((64 * direct_max_waves<BS, D>())) pa_direct_kernel(const KernelParams P) {
    constexpr bool KLDS = !KV8 && D == 128;
    constexpr int LW = direct_wave_lds<BS, D, KV8>();
    extern __shared__ __attribute__((aligned(16))) char direct_lds[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
    const int per_seq = P.kv_heads * P.row_tiles;
    const int b = blockIdx.x / per_seq, jr = blockIdx.x - b * per_seq;
    const int kvh = jr / P.row_tiles, rt = jr - kvh * P.row_tiles;
    const int rows_here = min(16, P.rows - rt * 16);
    const int len = P.context_lens[b];
    const int cap = P.max_blocks * BS;
    // every workgroup of a sequence checks its length (see flag_bad_lengths)
    if (threadIdx.x == 0 && (len < (P.causal ? P.q_len : 0) || len > cap)) atomicOr(P.error_flag, kErrBadLength);
    const int ctx = __builtin_amdgcn_readfirstlane(min(max(len, 0), cap));
    const int nb = (ctx + BS - 1) / BS;
    const int per = (nb + waves - 1) / waves;  // blocks per wave
    const int units = rows_here * (D / 4);     // 16-byte units of the tile's output
    if (nb == 0) {                             // empty context: defined as a zero output
        for (int u = threadIdx.x; u < units; u += blockDim.x) {
            const int row = u / (D / 4);
            OutStore<OutT>::store4(P.out, out_row_offset(P, b, kvh, rt * 16 + row, D) + 4 * (u - row * (D / 4)),
                                   (f32x4_t){0.f, 0.f, 0.f, 0.f});
        }
        return;
    }
    char *const lds = direct_lds + wave * LW;
    float *const part = reinterpret_cast<float *>(lds);
    const int lo = wave * per, hi = min(nb, lo + per);
    if (lo < hi) {
        if constexpr (BS * D > 16384)
            run_segment_big<BS, D, D, OutT, ET>(P, b, kvh, rt, ctx, nb, lo, hi, part, part + 16 * D);
        else
            run_segment<BS, D, D, OutT, false, KV8, KLDS, ET>(P, b, kvh, rt, ctx, nb, lo, hi, part, part + 16 * D,
                                                              false, lds);
    }
    const int pieces = (nb + per - 1) / per;
    if (pieces == 1) return;  // wave 0 stored the output
    __syncthreads();
    // log-sum-exp merge of the waves' pieces, in the arithmetic of the merge
    // kernel: the weights are normalised first and the sums run in piece order,
    // so a tile cut into the same pieces by the work lists has the same bits
    auto merge = [&](auto most) {  // every LDS read of a unit in flight at once
        constexpr int N = decltype(most)::value;
        for (int u = threadIdx.x; u < units; u += blockDim.x) {
            const int row = u / (D / 4), c = 4 * (u - row * (D / 4));
            float m[N], l[N];
            f32x4_t piece[N];
#pragma unroll
            for (int w = 0; w < N; ++w) {
                const float *const p = reinterpret_cast<const float *>(direct_lds + min(w, pieces - 1) * LW);
                m[w] = p[16 * D + row];
                l[w] = p[16 * D + 16 + row];
                piece[w] = *reinterpret_cast<const f32x4_t *>(p + row * D + c);
            }
            float M = m[0];
#pragma unroll
            for (int w = 1; w < N; ++w) M = fmaxf(M, m[w]);
            float L = 0.f;
#pragma unroll
            for (int w = 0; w < N; ++w)
                if (w < pieces) {
                    m[w] = __expf(m[w] - M);
                    L += m[w] * l[w];
                }
            const float inv = L > 0.f ? 1.f / L : 0.f;
            f32x4_t o = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int w = 0; w < N; ++w)
                if (w < pieces) o += (m[w] * inv) * piece[w];
            OutStore<OutT>::store4(P.out, out_row_offset(P, b, kvh, rt * 16 + row, D) + c, o);
        }
    };
    constexpr int MAXW = direct_max_waves<BS, D>();
    if (MAXW <= 4 || pieces <= 4)
        merge(std::integral_constant<int, 4>{});
    else if (MAXW <= 8 || pieces <= 8)
        merge(std::integral_constant<int, MAXW < 8 ? MAXW : 8>{});
    else
        merge(std::integral_constant<int, MAXW>{});
}

template <int BS, int D, typename OutT, bool KV8, typename ET>
DirectFn direct_fn() {
    return {pa_direct_kernel<BS, D, OutT, KV8, ET>, direct_max_waves<BS, D>(), direct_wave_lds<BS, D, KV8>()};
}

template <int D, typename OutT, bool KV8, typename ET>
DirectFn direct_by_block(int bs) {
    switch (bs) {
        case 16: return direct_fn<16, D, OutT, KV8, ET>();
        case 32: return direct_fn<32, D, OutT, KV8, ET>();
        case 64: return direct_fn<64, D, OutT, KV8, ET>();
        case 128: return direct_fn<128, D, OutT, KV8, ET>();
        default: return DirectFn{};
    }
}

template <typename OutT, typename ET>
DirectFn direct_by_dim(int bs, int d) {
    switch (d) {
        case 16: return direct_by_block<16, OutT, false, ET>(bs);
        case 32: return direct_by_block<32, OutT, false, ET>(bs);
        case 64: return direct_by_block<64, OutT, false, ET>(bs);
        case 128: return direct_by_block<128, OutT, false, ET>(bs);
        case 256: return direct_by_block<256, OutT, false, ET>(bs);
        default: return DirectFn{};
    }
}

}  // namespace pa
}  // namespace simpler_hip
