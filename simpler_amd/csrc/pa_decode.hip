// Host side of the paged-attention decode: argument validation, the work
// plan (worker count, work lists, workspace layout), kernel selection and the
// C entry points of include/simpler_hip/pa_decode.h. The kernels themselves
// are in pa_kernels.h, instantiated by the pa_kernels_*.hip translation units.

#include <hip/hip_runtime.h>

#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <mutex>
#include <vector>

#include "simpler_hip/pa_decode.h"
#include "pa_decode_internal.h"
#include "pa_kernels.h"

namespace simpler_hip {
namespace {

using namespace pa;

// ----------------------------------------------------------------------------
// Host side: validation, worker count, dispatch
// ----------------------------------------------------------------------------

constexpr int kZeroOffset = 128;  // workspace bytes [128, 256) are never written after init
constexpr int kMaxAppendTokens = 16;  // fused append: new tokens per sequence (one per residue mod 16)
constexpr size_t kMaxZeroPageBytes = 1 << 20;  // larger token strides read the padding tiles as they are
constexpr int kMlaSegTokens = 256;  // MLA: work charged for each sequence a slice starts, in tokens

struct Plan {
    int workers;
    int row_tiles;
    int rows;
    int tiles_per_worker;
    int row_groups;
    int threads;  // per worker workgroup
    size_t lds;   // dynamic LDS per workgroup (sibling waves' K buffers)
    int groups;   // workgroups per worker (MLA row groups), else 1
    int lanes;    // work lists (KernelParams::lanes)
    int seg_cost; // KernelParams::seg_cost
    int64_t grid;
    KernelFn main;
    size_t flag_bytes, zero_bytes, part_ml_bytes, part_o_bytes;
    size_t total;
};

inline size_t align_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

int validate(const SimplerHipPaDecodeArgs *a) {
    if (!a) return SIMPLER_HIP_ERR_INVALID;
    if (!a->query || !a->key_cache || !a->value_cache || !a->block_table || !a->context_lens || !a->out)
        return SIMPLER_HIP_ERR_INVALID;
    if (a->batch < 0 || a->q_len < 1 || a->num_kv_heads < 1 || a->num_heads < 1) return SIMPLER_HIP_ERR_INVALID;
    if (a->num_heads % a->num_kv_heads) return SIMPLER_HIP_ERR_INVALID;
    if (a->head_dim_k < 8 || a->head_dim_v < 8 || a->head_dim_k % 8 || a->head_dim_v % 8)
        return SIMPLER_HIP_ERR_INVALID;
    if (a->block_size < 1 || a->max_blocks_per_seq < 1 || a->num_blocks < 1) return SIMPLER_HIP_ERR_INVALID;
    const int64_t strides[6] = {a->k_block_stride, a->k_token_stride, a->k_head_stride,
                                a->v_block_stride, a->v_token_stride, a->v_head_stride};
    if (a->kv_format != SIMPLER_HIP_KV_BF16 && a->kv_format != SIMPLER_HIP_KV_FP8_E4M3 &&
        a->kv_format != SIMPLER_HIP_KV_FP16)
        return SIMPLER_HIP_ERR_INVALID;
    const bool fp8 = a->kv_format == SIMPLER_HIP_KV_FP8_E4M3;
    const int esz = fp8 ? 1 : 2;
    for (int64_t s : strides)
        if (s <= 0 || (s * esz) % 16) return SIMPLER_HIP_ERR_INVALID;  // 16-byte aligned rows
    if (a->k_token_stride * esz * a->block_size >= (int64_t)1 << 31 ||
        a->v_token_stride * esz * a->block_size >= (int64_t)1 << 31)
        return SIMPLER_HIP_ERR_INVALID;  // per-lane 32-bit byte offsets within a block
    if (fp8 && (!a->k_scale || !a->v_scale || ((uintptr_t)a->k_scale & 3) || ((uintptr_t)a->v_scale & 3)))
        return SIMPLER_HIP_ERR_INVALID;
    if (a->out_dtype != SIMPLER_HIP_DT_FLOAT32 && a->out_dtype != SIMPLER_HIP_DT_BFLOAT16 &&
        a->out_dtype != SIMPLER_HIP_DT_FLOAT16)
        return SIMPLER_HIP_ERR_UNSUPPORTED;
    if (!(a->scale == a->scale)) return SIMPLER_HIP_ERR_INVALID;
    if (a->num_workers < 0) return SIMPLER_HIP_ERR_INVALID;
    if (((uintptr_t)a->query | (uintptr_t)a->key_cache | (uintptr_t)a->value_cache | (uintptr_t)a->out) & 15)
        return SIMPLER_HIP_ERR_INVALID;
    const int group = a->num_heads / a->num_kv_heads;
    const int64_t row_tiles = ((int64_t)group * a->q_len + 15) / 16;
    // the flattened (tile, block) work list is indexed with 32-bit integers
    if ((int64_t)a->batch * a->num_kv_heads * row_tiles * a->max_blocks_per_seq >= (int64_t)1 << 31)
        return SIMPLER_HIP_ERR_UNSUPPORTED;
    if ((int64_t)a->batch * a->num_kv_heads * row_tiles >= (int64_t)1 << 31) return SIMPLER_HIP_ERR_UNSUPPORTED;
    return SIMPLER_HIP_OK;
}

// MLA: V is the first head_dim_v dims of K (same buffer, same strides).
bool is_mla_shape(const SimplerHipPaDecodeArgs *a) { return a->head_dim_k == kMlaDk && a->head_dim_v == kMlaDv; }

bool v_is_k_prefix(const SimplerHipPaDecodeArgs *a) {
    return a->value_cache == a->key_cache && a->v_block_stride == a->k_block_stride &&
           a->v_token_stride == a->k_token_stride && a->v_head_stride == a->k_head_stride;
}

// The main kernel(s) and the merge kernel a decode with these args runs;
// main is null when the combination is not supported. With `append`, ka holds
// the fused-append variants of k (same launch shapes; the plan is made from k).
struct Kernels {
    KernelPair k;
    KernelPair ka;
    DirectFn direct;
    MergeFn merge;
};

Kernels pick_kernel(const SimplerHipPaDecodeArgs *a, bool append = false) {
    Kernels s{};
    const int bs = a->block_size, dk = a->head_dim_k, dv = a->head_dim_v, out = a->out_dtype;
    const bool f16 = a->kv_format == SIMPLER_HIP_KV_FP16;
    if (a->kv_format == SIMPLER_HIP_KV_FP8_E4M3) {
        if (dk == dv && !append) {  // no fused append for fp8 caches
            s.k = pick_gqa_fp8(bs, dk, out);
            s.direct = pick_direct_fp8(bs, dk, out);
        }
    } else if (is_mla_shape(a)) {
        // (the kernel's fill offsets use 24-bit multiplies: token rows below 8 MB)
        if (v_is_k_prefix(a) && a->kv_format == SIMPLER_HIP_KV_BF16 && a->k_token_stride * 2 < (1 << 23)) {
            s.k = pick_mla(bs, out);  // no fused form: the append runs as its own launch
        }
    } else if (dk == dv) {
        s.k = f16 ? pick_gqa_f16(bs, dk, out) : pick_gqa_bf16(bs, dk, out);
        s.direct = f16 ? pick_direct_f16(bs, dk, out) : pick_direct_bf16(bs, dk, out);
        if (append) s.ka = f16 ? pick_gqa_f16_append(bs, dk, out) : pick_gqa_bf16_append(bs, dk, out);
    }
    s.merge = pick_merge(dv, out);
    if (!s.merge.fn[0] || (append && !s.ka.main)) s.k.main = nullptr;
    return s;
}

int current_device() {
    int dev = -1;
    return hipGetDevice(&dev) == hipSuccess ? dev : -1;
}

// Compute units of the current device; without one an MI355X is assumed.
int cu_count() {
    constexpr int kDevices = 64;
    static std::atomic<int> known[kDevices];
    const int dev = current_device();
    if (dev < 0) return 256;
    int n = dev < kDevices ? known[dev].load(std::memory_order_relaxed) : 0;
    if (n > 0) return n;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) {
        (void)hipGetLastError();
        return 256;
    }
    if (dev < kDevices) known[dev].store(n, std::memory_order_relaxed);
    return n;
}

// Default worker count: compute units x the requested workgroups per CU
// (workers_per_cu), capped by what the kernel's register footprint allows.
int wave_slots(KernelFn fn, int threads, int want_per_cu, size_t lds = 0) {
    struct Entry {
        KernelFn fn;
        int device;
        int threads;
        int want;
        size_t lds;
        int slots;
    };
    static std::mutex mu;
    static std::vector<Entry> cache;
    const int dev = current_device();
    std::lock_guard<std::mutex> lk(mu);
    for (const Entry &e : cache)
        if (e.fn == fn && e.device == dev && e.threads == threads && e.want == want_per_cu && e.lds == lds)
            return e.slots;
    int per_cu = want_per_cu;
    const int cus = cu_count();
    // Without a device: the kernels use the whole register file of a SIMD
    // (one wave per SIMD, four SIMDs per CU), the MLA kernel most of the LDS.
    if (dev < 0) per_cu = std::max(1, std::min(per_cu, 256 / threads));
    if (dev >= 0) {
        int n = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, reinterpret_cast<const void *>(fn),
                                                         threads, lds) == hipSuccess &&
            n > 0 && n < per_cu)
            per_cu = n;
    }
    (void)hipGetLastError();
    const int slots = cus * per_cu;
    cache.push_back({fn, dev, threads, want_per_cu, lds, slots});
    return slots;
}

// Workers per CU of the GQA kernels (wave_slots lowers it to what fits).
// - K in whole rows through LDS, one row tile: one per SIMD (108.9 us at four,
//   108.2 at three on the Qwen3-8B bs=32 shape, but 164.5 against 165.5 on
//   long contexts).
// - Two-tile waves, whose blocks take twice the math per byte: three (the
//   verify shape 134.2 us against 142.9 with four).
// - Waves that keep K and V in registers and read rows of 128 bytes or less
//   (head dims to 64, fp8 caches): a wave has one block of K and one of V in
//   flight, 4 KB with 16-token blocks of 64 dims, so the smaller the block
//   the more waves a CU needs. us per main launch, 37 sequences of 300 to 5000
//   tokens, 8 kv heads of 64 dims, at 2 / 4 / 6 / 8 per CU: 16-token blocks
//   104.4 / 60.1 / 43.5 / 36.2; 32: 71.8 / 42.3 / 34.5 / 36.3; 64: 55.9 / 37.2
//   / 37.8 / 37.1; 128: 58.6 / 37.8 / 49.5 / 43.3. fp8 (32 sequences to 8192)
//   at 3 / 4 / 8: 101.4 / 79.6 / 54.2; 66.8 / 54.9 / 57.8; 54.2 / 57.1 / 58.2.
//   128-token fp8 blocks: three; four was up to 4% faster with some lengths and
//   up to 3% slower with others (steps of 32 sequences of 1024-8192 tokens at
//   3 / 4, three draws: 62.7 / 60.5, 63.0 / 64.1, 58.3 / 59.4).
// - 256-dim heads: two (four and more measured 2-8% slower), but four where a
//   block exceeds the registers and runs unpipelined (151.6 against 170.7).
// - Sibling waves (several row tiles per worker): the same by waves, since
//   the siblings' loads meet in the caches. us per main launch, 16 sequences of
//   4 kv heads (122 MB), 2 / 3 / 4 tiles, against two, one and one workgroups
//   per CU: 64 dims x 16 tokens 35.5 / 48.7 / 59.5 against 63.0 / 108 / 115,
//   x 32 31.5 / 42.3 / 51.9 against 44.0 / 73.3 / 75.2; 128 dims x 16 tokens,
//   3 / 4 tiles, 35.7 / 40.0 against 49.9 / 52.6 (at 64 and 128 tokens one
//   workgroup is best); fp8, 2 tiles, 16 / 32 / 64 tokens 42.7 / 35.3 / 34.1
//   against 75.1 / 51.4 / 41.0.
// A plan made without a device (which can launch nothing) reports `nominal`
// counts that do not depend on the block size.
int workers_per_cu(const SimplerHipPaDecodeArgs *a, const KernelPair &k, const Plan &p, bool pair, bool nominal) {
    if (pair) return kWorkersThreePerCu;
    const int bs = a->block_size, d = a->head_dim_k, tiles = p.tiles_per_worker;
    const bool fp8 = a->kv_format == SIMPLER_HIP_KV_FP8_E4M3;
    if (tiles > 1) {
        if (nominal) return kWorkersPerCu;
        const int waves = (d <= 64 || fp8) ? (bs <= 16 ? 12 : bs <= 32 ? 9 : bs <= 64 ? 6 : 4)
                          : d <= 128       ? (bs <= 16 ? 8 : bs <= 32 ? 6 : 4)
                                           : 4;
        return std::max(1, waves / tiles);
    }
    if (k.klds) return kWorkersPerSimdCu;
    if (nominal) return fp8 ? kWorkersThreePerCu : kWorkersPerCu;
    if (fp8) return bs <= 16 ? 8 : bs <= 32 ? 4 : 3;
    if (d <= 64) return bs <= 16 ? 8 : bs <= 32 ? 6 : 4;
    return bs * d > 16384 ? 4 : kWorkersPerCu;
}

Plan make_plan(const SimplerHipPaDecodeArgs *a, const KernelPair &k) {  // k: the main kernels of pick_kernel
    Plan p{};
    const int group = a->num_heads / a->num_kv_heads;
    p.rows = group * a->q_len;
    p.row_tiles = (p.rows + 15) / 16;
    p.lanes = 1;
    if (k.mla) {
        // A work slice runs as `groups` sibling workgroups of 128 rows (8 row
        // tiles of 16) each; `workers` counts slices.
        p.groups = (p.rows + kMlaRowsPerGroup - 1) / kMlaRowsPerGroup;
        p.tiles_per_worker = kMlaRowsPerGroup / 16 * p.groups;
        p.row_groups = 1;
        p.threads = 256;
        // At most 64 rows: the kernels whose four waves share the rows. us per
        // step against the 128-row form: 32 sequences of 32 rows, 200-6000
        // tokens 35.4 against 42.2; 16 of 16 rows, 1000-30000 68 against 105;
        // 32 of 64 rows, 500-8000 59 against 72 (32-token blocks alike).
        p.main = p.rows <= 32 ? k.main_multi : p.rows <= 64 ? k.main_pair : k.main;
        if (a->num_workers > 0) {
            p.workers = a->num_workers;
        } else {
            // One workgroup per CU: its two blocks fill half the LDS or more
            // (a 32-token form whose registers let two run would double the
            // partials, beyond the fixed scratch of the no-alloc entry).
            const int wgs = wave_slots(p.main, p.threads, 1);
            p.workers = wgs / p.groups > 0 ? wgs / p.groups : 1;
        }
        p.grid = (int64_t)p.workers * p.groups;
        // A slice that starts another sequence pays for its set-up: 147 KB of
        // query rows, a first block fetched without prefetch and a 256 KB
        // partial or output store, about 23 us per extra sequence on cfg4
        // (per-workgroup timestamps: 228 / 252 / 275 us for slices of one,
        // two and three sequences with equal blocks), so each sequence is
        // charged kMlaSegTokens tokens of work ahead of its blocks.
        p.seg_cost = (kMlaSegTokens + a->block_size - 1) / a->block_size;
    } else {
        // Row tiles of one kv head run as sibling waves of one worker workgroup
        // (up to four), so K/V of a block is fetched once for all of them;
        // two row tiles with K through LDS run in one wave instead.
        const bool pair = k.main_pair && p.row_tiles == 2;
        p.tiles_per_worker = pair ? 2 : (p.row_tiles < kMaxWavesPerWorker ? p.row_tiles : kMaxWavesPerWorker);
        p.threads = pair ? 64 : 64 * p.tiles_per_worker;
        p.main = pair ? k.main_pair : p.tiles_per_worker > 1 ? k.main_multi : k.main;
        if (!pair && k.klds && p.tiles_per_worker > 1) p.lds = (size_t)p.tiles_per_worker * a->block_size * 256;
        p.groups = 1;
        p.row_groups = (p.row_tiles + p.tiles_per_worker - 1) / p.tiles_per_worker;
        const int per_cu = workers_per_cu(a, k, p, pair, current_device() < 0);
        p.workers = a->num_workers > 0 ? a->num_workers : wave_slots(p.main, p.threads, per_cu, p.lds);
        // Work lists (the tiles of a batch shared out among them, rotating with
        // the batch). 16-bit caches: one list per tile of a batch when the
        // worker count allows it, so the kv heads' workers walk the same blocks
        // side by side (cfg3-like long contexts: 167.7 us against 173.4 us
        // with one list, and 176 with two tiles per list). fp8 caches, whose
        // heads are single 128-byte lines of a 1 KB token row: four lists
        // (60.5 us against 61.4 with one list and 62.4 with one per tile on
        // the Qwen3-8B bs=32 shape).
        const int tpb = a->num_kv_heads * p.row_groups;
        const bool fp8 = a->kv_format == SIMPLER_HIP_KV_FP8_E4M3;
        const int want_lanes = fp8 ? (tpb % 4 == 0 ? 4 : 1) : tpb;
        if (want_lanes > 1) {
            if (a->num_workers > 0) {
                if (p.workers % want_lanes == 0) p.lanes = want_lanes;
            } else if (p.workers >= 4 * want_lanes) {
                p.workers -= p.workers % want_lanes;
                p.lanes = want_lanes;
            }
        }
        p.grid = p.workers;
    }
    const int dv = a->head_dim_v;
    // Layout: [error word] [zero page] [m,l partials] [O partials]; two
    // partial slots per worker wave. The zero page covers the lane offsets of
    // one 16-token tile (16 token strides of K or V, plus the dims): tiles past
    // a context's end read it instead of the cache. Its contents do not affect
    // results (those tokens are masked and their V rows zeroed), so calls of
    // other shapes may overwrite it.
    const int esz = a->kv_format == SIMPLER_HIP_KV_FP8_E4M3 ? 1 : 2;
    const size_t tok_bytes = (size_t)std::max(a->k_token_stride, a->v_token_stride) * esz;
    const size_t zero_bytes = align_up(16 * tok_bytes + 512, 256);
    p.zero_bytes = (!k.mla && zero_bytes <= kMaxZeroPageBytes) ? zero_bytes : 0;
    const size_t pieces = (size_t)p.workers * p.tiles_per_worker * 2;
    p.flag_bytes = 256;  // error word at 0, zeros at [kZeroOffset, 256)
    p.part_ml_bytes = align_up(pieces * 32 * sizeof(float), 256);
    p.part_o_bytes = align_up(pieces * 16 * dv * sizeof(float), 256);
    p.total = p.flag_bytes + p.zero_bytes + p.part_ml_bytes + p.part_o_bytes;
    return p;
}

// Waves per workgroup of the short-context kernels (pa_kernels_direct.h), or 0
// where the work lists run: the caller forced a worker count, or a context may
// be long (the host knows the table's width, not the lengths). One workgroup
// per tile saves the merge launch and the work scan, but does not balance
// lengths and has fewer waves for a tile, so it is taken where the longest
// possible tile is short. us per step, this form / work lists, all sequences
// as long as the table is wide or 10-30% to 100% of it:
// - From 32 tiles: up to 384 KB of K and V per tile (16 to 100 sequences of 8
//   kv heads, 128 dims, 0.55 to 0.92 of the lists' time; at 512 KB, 40 of 1024
//   tokens 37.8 / 36.6, 100 of 102-1024 50.2 / 48.4). 256 KB with head dims to
//   64 and fp8 caches (0.97 at most; 4 x 8 of 200-2000 tokens, 64 dims, 17.8 /
//   15.4) and with 256 dims, there 384 KB from 128 tiles (0.96 at most) unless
//   blocks exceed the registers (200 x 4, 51-512 tokens in 128-token blocks,
//   512 KB, 72.8 / 65.1).
// - Fewer tiles, whose chains the lists cut finer: 192 KB with head dims to 64
//   and fp8 caches (0.97 at most; one sequence of 64 dims in 16-token blocks
//   10.2 / 9.9 at 256 KB, 16.1 / 10.3 at 512), else 256 KB (128 dims 0.84 at
//   most; 9.8 / 9.6 at 384), with 256 dims one block per wave (1.005 at most;
//   with two 12.2 / 9.4).
// - To 128 tiles one block per wave or 48 KB (two 64 KB blocks 16.2 / 13.5).
// - A sequence as long as the table among short ones is one chain here, and cut
//   among all workers by the lists: to 511 tiles six blocks per wave to 32
//   tokens, four of 64, three of 128, from 512 tiles ten, ten, six and three.
//   With one such sequence and 10 tokens in the others 0.96 at most (512 tiles
//   of 16 dims, 64-token blocks: 6 blocks 0.9, 8 15.7 / 14.1, 32 51.6 / 15.0;
//   2048 of 64 dims, 32-token blocks: 8 0.73, 16 23.3 / 18.9, 32 42.3 / 19.4).
// - Every row tile of a kv head reads K and V again: with several of them up to
//   64 KB per tile (0.93 at most, to 8192 tiles) or 48 MB in all (0.92 at most;
//   128 x 8 kv heads, 64 rows of 64 dims, 1000 tokens in 32-token blocks, 1 GB,
//   174 / 127; 15 x 8 of 380 tokens, 64 rows of 128 dims, 90 MB, 23.5 / 20.9).
//   Above 64 dims, 768 KB over the row tiles of a kv head at most.
// Waves per tile: enough for workers_per_cu waves on every CU, at least four.
int direct_waves(const SimplerHipPaDecodeArgs *a, const Kernels &s, const Plan &p) {
    if (!s.direct.fn || a->num_workers > 0) return 0;
    const int bs = a->block_size, d = a->head_dim_k;
    const bool fp8 = a->kv_format == SIMPLER_HIP_KV_FP8_E4M3, narrow = fp8 || d <= 64;
    const int64_t blocks = a->max_blocks_per_seq, block = (int64_t)bs * 2 * d * (fp8 ? 1 : 2);
    const int64_t tile = blocks * block;
    const int64_t tiles = std::max<int64_t>((int64_t)a->batch * a->num_kv_heads * p.row_tiles, 1);
    constexpr int64_t KB = 1 << 10;
    if (!narrow && p.row_tiles > 1 && tile * p.row_tiles > 768 * KB) return 0;
    Plan one = p;
    one.tiles_per_worker = 1;
    const int64_t want = (int64_t)cu_count() * std::max(kWorkersPerSimdCu, workers_per_cu(a, s.k, one, false, false));
    const int64_t waves = std::min<int64_t>({(want + tiles - 1) / tiles, s.direct.max_waves, blocks});
    const int64_t per_wave = (blocks + waves - 1) / waves;
    if (per_wave > (bs > 64 ? 3 : bs > 32 ? (tiles < 512 ? 4 : 6) : (tiles < 512 ? 6 : 10))) return 0;
    if (tiles < 128 && per_wave > 1 && per_wave * block > 48 * KB) return 0;
    if (tiles < 32 && per_wave > 1 && d > 128) return 0;
    const int64_t most = narrow    ? (tiles < 32 ? 192 : 256)
                         : d > 128 ? (tiles < 128 || bs * d > 16384 ? 256 : 384)
                                   : (tiles < 32 ? 256 : 384);
    if (tile > most * KB) return 0;
    if (p.row_tiles > 1 && tile > 64 * KB && tiles * tile > 48 * KB * KB) return 0;
    return (int)waves;
}

// MLA: whether each tile runs whole, in a launch of one workgroup per (tile,
// 128 rows), without the work lists and the merge. Short contexts only, as the
// host knows the table's width and not the lengths: with few workgroups a tile
// cut into blocks ends earlier. us per step against the work lists, 16 / 64 /
// 128 rows, 64-token blocks:
// - to 128 tokens any: one sequence 10.6 / 15.5 / 21.1 against 13.5 / 18.1 /
//   23.0, 128 of them 11.7 / 17.6 / 23.9 against 19.8 / 27.9 / 35.6;
// - to 256 from 32 workgroups: 32 of 128-256 tokens 14.5 / 20.3 / 28.9 against
//   15.3 / 26.3 / 31.6 (8 of them 14.5 / 20.0 / 28.1 against 14.0 / 20.0 / 26.5);
// - to 512 from 128 workgroups: 128 of 64-512 tokens 23.3 / 31.0 / 43.9 against
//   26.7 / 38.8 / 52.4 (64 of 256-512 22.9 / 30.3 / 43.1 against 20.5 / 31.5 /
//   41.7; 300 of 256-1024 73 / 87 / 120 against 69 / 88 / 121).
// These are with lengths near each other; one sequence as long as the table
// among sequences of 10 tokens is a chain of blocks here, hence 384 tokens from
// 128 workgroups (128 rows 42.1 against 38.0 at 512) and 192 below 64 (128 rows
// 27.8 against 26.6 at 256). 32-token blocks are twice the steps: 256 tokens from
// 128 workgroups (128 of 128 rows 52.0 against 40.2 at 512), 192 from 64 (64 of
// 16 rows 15.9 against 15.3 at 256), 160 from 32, else 96 (one sequence of 128
// tokens, 96 rows, 20.4 against 19.2). 0.98 of the lists' time at most, 1.00 for
// 64 rows with 32-token blocks.
bool mla_whole_tiles(const SimplerHipPaDecodeArgs *a, const Kernels &s, const Plan &p) {
    if (!s.k.mla || a->num_workers > 0) return false;
    const int64_t groups = (int64_t)a->batch * a->num_kv_heads * p.groups;
    const int64_t tokens = (int64_t)a->max_blocks_per_seq * a->block_size;
    if (a->block_size == 32) return tokens <= (groups >= 128 ? 256 : groups >= 64 ? 192 : groups >= 32 ? 160 : 96);
    return tokens <= (groups >= 128 ? 384 : groups >= 64 ? 256 : groups >= 32 ? 192 : 128);
}

// How a plain decode runs: one workgroup of `waves` waves per tile
// (pa_direct_kernel), an MLA workgroup per whole tile and row group, or, with
// neither, the work lists.
struct Route {
    int waves;
    bool whole;
};

Route pick_route(const SimplerHipPaDecodeArgs *a, const Kernels &s, const Plan &p) {
    return {direct_waves(a, s, p), mla_whole_tiles(a, s, p)};
}

// Writes the error word into the host's mirror, after everything before it on
// the stream.
__global__ void mirror_kernel(const unsigned *flag, unsigned *mirror) {
    __hip_atomic_store(mirror, *flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The merge's launch: workgroups per tile (grid y), each with `units` of the
// tile's 16-byte units. A tile is cut into about workers / tiles + 1 pieces,
// at most one per block.
// It is shared out among workgroups (down to 8 units, a 128-byte line, each)
// until a thread has one unit and reads kMergeAhead of its pieces at most,
// as long as the grid stays within kMergeGrid workgroups: with more, every
// workgroup's own set-up costs more than its shorter chain saves. us of the
// merge alone, launched in a row: 128 sequences of 128 MLA heads, 1024 tiles,
// 18.9 with one per tile and 30.9 with four; 32 of them, 256 tiles, 15.4 with
// four, 16.2 with one, 17.8 with sixteen; one sequence of 16 heads and 32000
// tokens, one tile, 7.2 in 128 workgroups and 444 in one. Small tiles of few
// pieces take smaller workgroups.
struct MergePlan {
    KernelFn fn;
    int units, groups, threads;
};
constexpr int64_t kMergeGrid = 1024;

MergePlan plan_merge(const MergeFn &m, const SimplerHipPaDecodeArgs *a, const Plan &p) {
    const int64_t all = (int64_t)std::min(16, p.rows) * (a->head_dim_v / 4);
    const int64_t lists = (int64_t)a->batch * a->num_kv_heads;
    const int64_t tiles = std::max<int64_t>(lists * p.row_tiles, 1);
    const int64_t pieces = std::min<int64_t>(p.workers / std::max<int64_t>(lists * p.row_groups, 1) + 1,
                                             a->max_blocks_per_seq);
    MergePlan r{};
    int64_t units = all, groups = 1;
    while (units >= 16 && tiles * groups * 2 <= kMergeGrid &&
           (units > kMergeThreads || units * pieces > kMergeThreads * kMergeAhead)) {
        units = (units + 1) / 2;
        groups = (all + units - 1) / units;
    }
    r.units = (int)units;
    r.groups = (int)groups;
    r.threads = kMergeThreads;
    while (r.threads > 128 && units <= r.threads / 2 && units * pieces <= r.threads / 2 * kMergeAhead) r.threads /= 2;
    r.fn = m.fn[units <= kMergeThreads ? 0 : units <= 2 * kMergeThreads ? 1 : 2];
    return r;
}

}  // namespace
}  // namespace simpler_hip

using namespace simpler_hip;

extern "C" size_t simpler_hip_pa_decode_workspace_size(const SimplerHipPaDecodeArgs *args) {
    if (validate(args) != SIMPLER_HIP_OK) return 0;
    const Kernels s = pick_kernel(args);
    if (!s.k.main) return 0;
    return make_plan(args, s.k).total;
}

namespace simpler_hip {
namespace {
// Zeroes [p, p + bytes): 16-byte stores over the aligned body, byte stores for
// the tail. A kernel rather than hipMemsetAsync, so that callers may enqueue it
// inside a HIP graph capture (memset nodes are avoided in captured work).
__global__ void __launch_bounds__(256) zero_fill_kernel(char *p, size_t bytes) {
    const size_t n16 = bytes / 16;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += stride)
        reinterpret_cast<u32x4_t *>(p)[i] = (u32x4_t){0u, 0u, 0u, 0u};
    if (blockIdx.x == 0 && threadIdx.x < bytes % 16) p[n16 * 16 + threadIdx.x] = 0;
}
}  // namespace

int zero_fill(void *p, size_t bytes, void *stream) {
    if (bytes == 0) return SIMPLER_HIP_OK;
    const size_t units = (bytes + 15) / 16;
    const unsigned grid = (unsigned)std::min<size_t>((units + 255) / 256, 2048);
    hipLaunchKernelGGL(zero_fill_kernel, dim3(grid), dim3(256), 0, (hipStream_t)stream, (char *)p, bytes);
    return hipGetLastError() == hipSuccess ? SIMPLER_HIP_OK : SIMPLER_HIP_ERR_LAUNCH;
}
}  // namespace simpler_hip

extern "C" int simpler_hip_pa_decode_workspace_init(void *workspace, size_t workspace_bytes, void *stream) {
    if (!workspace) return SIMPLER_HIP_ERR_WORKSPACE;
    return simpler_hip::zero_fill(workspace, workspace_bytes, stream);
}

extern "C" int simpler_hip_pa_decode_plan(const SimplerHipPaDecodeArgs *args, int32_t *num_workers) {
    const int rc = validate(args);
    if (rc != SIMPLER_HIP_OK) return rc;
    const Kernels s = pick_kernel(args);
    if (!s.k.main) return SIMPLER_HIP_ERR_UNSUPPORTED;
    const Plan plan = make_plan(args, s.k);
    const Route route = pick_route(args, s, plan);
    if (num_workers)
        *num_workers = route.waves   ? args->batch * args->num_kv_heads * plan.row_tiles
                       : route.whole ? args->batch * args->num_kv_heads
                                     : plan.workers;
    return SIMPLER_HIP_OK;
}

extern "C" const char *simpler_hip_pa_decode_kernel_name(const SimplerHipPaDecodeArgs *args) {
    if (validate(args) != SIMPLER_HIP_OK) return "";
    const Kernels s = pick_kernel(args);
    if (!s.k.main) return "";
    if (s.k.mla) return "pa_mla_kernel";
    return pick_route(args, s, make_plan(args, s.k)).waves ? "pa_direct_kernel" : "pa_decode_kernel";
}

extern "C" int simpler_hip_pa_decode(const SimplerHipPaDecodeArgs *a, void *workspace, size_t workspace_bytes,
                                     void *stream) {
    return simpler_hip_pa_decode_phase(a, workspace, workspace_bytes, stream,
                                       SIMPLER_HIP_PHASE_MAIN | SIMPLER_HIP_PHASE_MERGE);
}

namespace simpler_hip {
namespace {
// k_new / v_new: the fused append's new tokens (null: plain decode).
int pa_decode_launch(const SimplerHipPaDecodeArgs *a, void *workspace, size_t workspace_bytes, void *stream,
                     int phases, unsigned *err_mirror, const void *k_new = nullptr, const void *v_new = nullptr) {
    if (phases & ~(SIMPLER_HIP_PHASE_MAIN | SIMPLER_HIP_PHASE_MERGE)) return SIMPLER_HIP_ERR_INVALID;
    int rc = validate(a);
    if (rc != SIMPLER_HIP_OK) return rc;
    const bool append = k_new != nullptr;
    const Kernels s = pick_kernel(a, append);
    if (!s.k.main) return SIMPLER_HIP_ERR_UNSUPPORTED;
    Plan plan = make_plan(a, s.k);
    if (append)
        plan.main = plan.main == s.k.main_multi ? s.ka.main_multi : plan.main == s.k.main_pair ? s.ka.main_pair : s.ka.main;
    if (!workspace || workspace_bytes < plan.total || ((uintptr_t)workspace & 255)) return SIMPLER_HIP_ERR_WORKSPACE;
    if (a->batch == 0) return SIMPLER_HIP_OK;

    KernelParams P{};
    P.q = (const uint16_t *)a->query;
    P.k = (const uint16_t *)a->key_cache;
    P.v = (const uint16_t *)a->value_cache;
    P.block_table = a->block_table;
    P.context_lens = a->context_lens;
    P.out = a->out;
    char *ws = (char *)workspace;
    P.error_flag = (unsigned *)ws;
    P.zeros = ws + kZeroOffset;
    P.zero_page = plan.zero_bytes ? ws + plan.flag_bytes : nullptr;
    P.part_ml = (float *)(ws + plan.flag_bytes + plan.zero_bytes);
    P.part_o = (float *)(ws + plan.flag_bytes + plan.zero_bytes + plan.part_ml_bytes);
    P.k_block_stride = a->k_block_stride;
    P.k_token_stride = a->k_token_stride;
    P.k_head_stride = a->k_head_stride;
    P.v_block_stride = a->v_block_stride;
    P.v_token_stride = a->v_token_stride;
    P.v_head_stride = a->v_head_stride;
    P.batch = a->batch;
    P.q_len = a->q_len;
    P.num_heads = a->num_heads;
    P.kv_heads = a->num_kv_heads;
    P.group = a->num_heads / a->num_kv_heads;
    P.rows = plan.rows;
    P.row_tiles = plan.row_tiles;
    P.tiles_per_worker = plan.tiles_per_worker;
    P.row_groups = plan.row_groups;
    P.block_size = a->block_size;
    P.max_blocks = a->max_blocks_per_seq;
    P.num_pool_blocks = a->num_blocks;
    P.workers = plan.workers;
    P.lanes = plan.lanes;
    P.seg_cost = plan.seg_cost;
    P.scale = a->scale;
    P.causal = (a->causal && a->q_len > 1) ? 1 : 0;
    P.k_scale = a->k_scale;
    P.v_scale = a->v_scale;
    P.err_mirror = (phases & SIMPLER_HIP_PHASE_MERGE) ? err_mirror : nullptr;
    P.k_new = (const uint16_t *)k_new;
    P.v_new = (const uint16_t *)v_new;

    const int64_t tiles = (int64_t)a->batch * a->num_kv_heads * plan.row_tiles;
    const Route route = append ? Route{} : pick_route(a, s, plan);
    P.whole_tiles = route.whole;
    if (route.waves || route.whole) {  // one launch; the mirror's, if any, follows
        if (phases & SIMPLER_HIP_PHASE_MAIN) {
            if (route.waves)
                hipLaunchKernelGGL(s.direct.fn, dim3((unsigned)tiles), dim3(64u * route.waves),
                                   (unsigned)(route.waves * s.direct.wave_lds), (hipStream_t)stream, P);
            else
                hipLaunchKernelGGL(plan.main, dim3((unsigned)(a->batch * a->num_kv_heads * plan.groups)),
                                   dim3((unsigned)plan.threads), 0, (hipStream_t)stream, P);
            if (hipGetLastError() != hipSuccess) return SIMPLER_HIP_ERR_LAUNCH;
        }
        if (P.err_mirror) {
            hipLaunchKernelGGL(mirror_kernel, dim3(1), dim3(1), 0, (hipStream_t)stream, P.error_flag, P.err_mirror);
            if (hipGetLastError() != hipSuccess) return SIMPLER_HIP_ERR_LAUNCH;
        }
        return SIMPLER_HIP_OK;
    }
    const MergePlan merge = plan_merge(s.merge, a, plan);
    P.merge_units = merge.units;
    if (phases & SIMPLER_HIP_PHASE_MAIN) {
        hipLaunchKernelGGL(plan.main, dim3((unsigned)plan.grid), dim3((unsigned)plan.threads), (unsigned)plan.lds,
                           (hipStream_t)stream, P);
        if (hipGetLastError() != hipSuccess) return SIMPLER_HIP_ERR_LAUNCH;
    }
    if (phases & SIMPLER_HIP_PHASE_MERGE) {
        hipLaunchKernelGGL(merge.fn, dim3((unsigned)tiles, (unsigned)merge.groups), dim3((unsigned)merge.threads), 0,
                           (hipStream_t)stream, P);
        if (hipGetLastError() != hipSuccess) return SIMPLER_HIP_ERR_LAUNCH;
    }
    return SIMPLER_HIP_OK;
}
}  // namespace

int pa_decode_with_mirror(const SimplerHipPaDecodeArgs *a, void *workspace, size_t workspace_bytes, void *stream,
                          unsigned *err_mirror) {
    return pa_decode_launch(a, workspace, workspace_bytes, stream, SIMPLER_HIP_PHASE_MAIN | SIMPLER_HIP_PHASE_MERGE,
                            err_mirror);
}
}  // namespace simpler_hip

extern "C" int simpler_hip_pa_decode_phase(const SimplerHipPaDecodeArgs *a, void *workspace, size_t workspace_bytes,
                                           void *stream, int phases) {
    return simpler_hip::pa_decode_launch(a, workspace, workspace_bytes, stream, phases, nullptr);
}

extern "C" int simpler_hip_pa_decode_append(const SimplerHipPaDecodeArgs *a, const void *key_new,
                                            const void *value_new, void *workspace, size_t workspace_bytes,
                                            void *stream) {
    const int rc = validate(a);
    if (rc != SIMPLER_HIP_OK) return rc;
    if (a->kv_format == SIMPLER_HIP_KV_FP8_E4M3 || a->q_len > kMaxAppendTokens) return SIMPLER_HIP_ERR_UNSUPPORTED;
    const bool mla = is_mla_shape(a) && v_is_k_prefix(a);
    if (!key_new || ((uintptr_t)key_new & 15)) return SIMPLER_HIP_ERR_INVALID;
    if (mla ? value_new != nullptr : (!value_new || ((uintptr_t)value_new & 15))) return SIMPLER_HIP_ERR_INVALID;
    {
        // Two or more row tiles per worker (the two-tile wave, sibling waves,
        // MLA's 128-row workgroups): the append runs as its own launch ahead
        // of the plain decode. There the fused form's unpipelined new-token
        // blocks measured slower (the verify shape: 155.2 against 140.2 us per
        // step), and MLA's register budget has no room for the new rows; with
        // one tile per worker the fused form is the faster one (cfg2: 113.3
        // against 114.5). Ahead of the short-context kernel as well: both
        // launches together against the fused work lists, on the device alone,
        // 2 sequences of 153-512 tokens and one kv head 9.9 against 13.2 us, 16
        // of 90-300 and 8 heads 9.2 against 12.3, 32 of 153-512 in 16-token
        // blocks 13.3 against 18.3; 128 of 153-512, called in a row, 37.9
        // against 42.8.
        const Kernels s = pick_kernel(a);
        if (s.k.main) {
            const Plan plan = make_plan(a, s.k);
            if (plan.tiles_per_worker > 1 || s.k.mla || pick_route(a, s, plan).waves) {
                if (!workspace || workspace_bytes < plan.total || ((uintptr_t)workspace & 255))
                    return SIMPLER_HIP_ERR_WORKSPACE;
                if (a->batch == 0) return SIMPLER_HIP_OK;
                const int rc2 =
                    launch_paged_append(a, key_new, value_new, (unsigned *)workspace, kErrBadLength, stream);
                if (rc2 != SIMPLER_HIP_OK) return rc2;
                return pa_decode_launch(a, workspace, workspace_bytes, stream,
                                        SIMPLER_HIP_PHASE_MAIN | SIMPLER_HIP_PHASE_MERGE, nullptr);
            }
        }
    }
    return simpler_hip::pa_decode_launch(a, workspace, workspace_bytes, stream,
                                         SIMPLER_HIP_PHASE_MAIN | SIMPLER_HIP_PHASE_MERGE, nullptr, key_new,
                                         value_new);
}

namespace {

// simpler_hip_pa_decode_prelude's workspace after the decode's: the bf16
// query rows the prelude writes.
size_t prelude_query_bytes(const SimplerHipPaDecodeArgs *a) {
    return align_up((size_t)a->batch * a->q_len * a->num_heads * a->head_dim_k * 2, 256);
}

// The prelude entry's checks beyond validate(); a->query is not read.
int check_prelude(const SimplerHipPaDecodeArgs *a, const SimplerHipDecodePreludeArgs *pre) {
    if (a->kv_format != SIMPLER_HIP_KV_BF16 || a->head_dim_k != 128 || a->head_dim_v != 128 ||
        a->q_len > kMaxAppendTokens || (is_mla_shape(a) && v_is_k_prefix(a)))
        return SIMPLER_HIP_ERR_UNSUPPORTED;
    if (!pre) return SIMPLER_HIP_OK;
    const void *ptrs[8] = {pre->q_proj,        pre->k_proj,        pre->v_proj,   pre->inv_rms,
                           pre->q_norm_weight, pre->k_norm_weight, pre->rope_cos, pre->rope_sin};
    for (const void *p : ptrs)
        if (!p || ((uintptr_t)p & 15)) return SIMPLER_HIP_ERR_INVALID;
    if (pre->max_position < 1 || !(pre->eps >= 0.f)) return SIMPLER_HIP_ERR_INVALID;
    return SIMPLER_HIP_OK;
}

}  // namespace

extern "C" size_t simpler_hip_pa_decode_prelude_workspace_size(const SimplerHipPaDecodeArgs *a) {
    if (!a) return 0;
    SimplerHipPaDecodeArgs args = *a;
    if (!args.query) args.query = (const void *)(uintptr_t)256;  // not read: any aligned stand-in validates
    if (validate(&args) != SIMPLER_HIP_OK || check_prelude(&args, nullptr) != SIMPLER_HIP_OK) return 0;
    const Kernels s = pick_kernel(&args);
    if (!s.k.main) return 0;
    return make_plan(&args, s.k).total + prelude_query_bytes(&args);
}

extern "C" int simpler_hip_pa_decode_prelude(const SimplerHipPaDecodeArgs *a, const SimplerHipDecodePreludeArgs *pre,
                                             void *workspace, size_t workspace_bytes, void *stream) {
    if (!a || !pre) return SIMPLER_HIP_ERR_INVALID;
    // the query is computed: validate the rest with q_proj standing in for it
    SimplerHipPaDecodeArgs args = *a;
    args.query = pre->q_proj;
    int rc = validate(&args);
    if (rc != SIMPLER_HIP_OK) return rc;
    rc = check_prelude(&args, pre);
    if (rc != SIMPLER_HIP_OK) return rc;
    const Kernels s = pick_kernel(&args);
    if (!s.k.main) return SIMPLER_HIP_ERR_UNSUPPORTED;
    const size_t total = make_plan(&args, s.k).total;
    if (!workspace || workspace_bytes < total + prelude_query_bytes(&args) || ((uintptr_t)workspace & 255))
        return SIMPLER_HIP_ERR_WORKSPACE;
    if (args.batch == 0) return SIMPLER_HIP_OK;
    // The prelude as a launch of its own (query rows into the workspace after
    // the decode's part, new K/V rows into the caches), then the plain
    // decode on that query. Computing the prelude inside the decode's workers
    // measured slower on every shape tried (cfg2 117.4 against 115.6 us per
    // step, the verify shape 161.0 against 142.6, cfg1 17.5 against 14.3).
    void *const q = (char *)workspace + total;
    rc = launch_paged_prelude(&args, pre, q, (unsigned *)workspace, kErrBadLength, stream);
    if (rc != SIMPLER_HIP_OK) return rc;
    args.query = q;
    return simpler_hip::pa_decode_launch(&args, workspace, total, stream,
                                         SIMPLER_HIP_PHASE_MAIN | SIMPLER_HIP_PHASE_MERGE, nullptr);
}

// ---------------------------------------------------------------------------
// The entry point that allocates nothing: simpler_hip_pa_decode with the
// workspace replaced by a fixed device array of this library.
// ---------------------------------------------------------------------------

namespace simpler_hip {
namespace {

// Every decode of the direct entry fits here at the default worker count on
// MI355X (256 CUs): a GQA plan has at most 12 waves per CU, 6144 partial slots
// of 16 rows x Dv fp32, with head dims to 64 and fp8 caches (48 MiB at Dv 128),
// and 2048 with 256 dims (32 MiB); the MLA plan 4096 slots of 16 x 512 fp32 (256
// slices x 8 row tiles x 2: 128 MiB), plus (m, l) pairs, the error word and the
// zero page.
constexpr size_t kScratchBytes = (size_t)SIMPLER_HIP_PA_NOALLOC_SCRATCH_BYTES;
static_assert(kScratchBytes % 256 == 0, "scratch size");

// One copy per GPU the library runs on, held until the process ends. In host
// code `scratch` is only a stand-in for the symbol: its device address comes
// from hipGetSymbolAddress, per device.
static __device__ __align__(256) char scratch[kScratchBytes];

constexpr int kMaxScratchDevices = 64;
std::mutex g_scratch_mu;
void *g_scratch_ptr[kMaxScratchDevices] = {};

// This device's address of `scratch`, looked up once per device (with that
// device current) and kept; nullptr if the lookup fails.
void *scratch_on_current_device() {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxScratchDevices) return nullptr;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) {
            (void)hipGetLastError();
            return nullptr;
        }
        g_scratch_ptr[dev] = p;
    }
    return g_scratch_ptr[dev];
}

}  // namespace
}  // namespace simpler_hip

extern "C" int simpler_hip_pa_decode_noalloc(const SimplerHipPaDecodeArgs *a, void *stream) {
    int rc = validate(a);
    if (rc != SIMPLER_HIP_OK) return rc;
    const Kernels s = pick_kernel(a);
    if (!s.k.main) return SIMPLER_HIP_ERR_UNSUPPORTED;
    const size_t need = make_plan(a, s.k).total;
    if (need > kScratchBytes) {
        fprintf(stderr,
                "[simpler_hip] simpler_hip_pa_decode_noalloc: this decode needs %zu bytes of scratch, above the "
                "fixed %zu (use fewer workers or simpler_hip_pa_decode with a workspace)\n",
                need, kScratchBytes);
        return SIMPLER_HIP_ERR_WORKSPACE;
    }
    void *ws = scratch_on_current_device();
    if (!ws) return SIMPLER_HIP_ERR_LAUNCH;
    // Nothing in the scratch has to start at zero: every partial slot the
    // merge reads is written by the same call's main kernel, and the zero
    // page's contents never reach a result. The error word only accumulates.
    return simpler_hip::pa_decode_launch(a, ws, kScratchBytes, stream, SIMPLER_HIP_PHASE_MAIN | SIMPLER_HIP_PHASE_MERGE,
                                         nullptr);
}

extern "C" int simpler_hip_pa_decode_check(void *workspace, size_t workspace_bytes, void *stream) {
    if (!workspace || workspace_bytes < sizeof(unsigned)) return SIMPLER_HIP_ERR_WORKSPACE;
    unsigned flag = 0;
    if (hipStreamSynchronize((hipStream_t)stream) != hipSuccess) return SIMPLER_HIP_ERR_LAUNCH;
    if (hipMemcpy(&flag, workspace, sizeof(flag), hipMemcpyDeviceToHost) != hipSuccess) return SIMPLER_HIP_ERR_LAUNCH;
    if (flag == 0) return SIMPLER_HIP_OK;
    const unsigned zero = 0;
    if (hipMemcpy(workspace, &zero, sizeof(zero), hipMemcpyHostToDevice) != hipSuccess) return SIMPLER_HIP_ERR_LAUNCH;
    return (flag & kErrBadBlock) ? SIMPLER_HIP_ERR_BAD_BLOCK : SIMPLER_HIP_ERR_BAD_LENGTH;
}
