"""The short-context decode (one workgroup per tile, no merge launch) at the
edges of its shapes: fewer blocks than waves, one more, several per wave, a last
partial block, empty contexts, row tiles past the first, causal rows, the table widths on
both sides of the rule that selects it, and its error reports."""

from __future__ import annotations

import pytest
import torch

from oracle import pa_oracle as po
from simpler_amd import paged_attention as pa
from simpler_amd.workloads import make_custom_case, quantize_kv_fp8
from tests.pa_helpers import assert_close, oracle_numpy

pytestmark = pytest.mark.gpu


def run(case, device, **kw):
    d = case.to(device)
    if d.k_scale is not None:
        kw.update(k_scale=d.k_scale, v_scale=d.v_scale)
    out = pa.paged_attention_decode(d.query, d.key_cache, d.value_cache, d.block_table, d.context_lens,
                                    scale=case.scale, causal=case.config.causal, **kw)
    torch.cuda.synchronize(device)
    return out.cpu().numpy()


# (heads, kv heads, dim, block, lengths, q_len, table width in blocks)
@pytest.mark.parametrize("hq,hkv,dim,bs,lens,q_len,width", [
    (4, 1, 16, 16, [1, 0, 16, 17, 255, 256], 1, 16),      # one block per wave at most
    (16, 2, 64, 16, [0, 300, 511], 1, 32),                # two blocks for some waves
    (8, 8, 128, 128, [512, 385, 1, 0], 1, 4),             # one row, four waves
    (10, 2, 128, 64, [130, 64], 1, 4),
    (8, 1, 128, 32, [31, 33, 255], 1, 8),
    (4, 2, 256, 64, [200, 1], 1, 4),
    (4, 2, 256, 128, [128, 77], 1, 1),                    # blocks larger than the registers
    (40, 2, 128, 16, [97, 20], 1, 8),                     # a second row tile of 4 rows
    (32, 4, 64, 32, [8, 100, 64], 8, 4),                  # causal, four row tiles
    (32, 32, 64, 64, [1024, 3, 700, 0, 65], 1, 16),       # many tiles: one wave or two each
    (16, 1, 128, 128, [512, 400], 1, 5),                  # a table one block wider: the work lists
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_short_contexts(hq, hkv, dim, bs, lens, q_len, width, dtype, device):
    print(f"[case] {hq}/{hkv} d{dim} bs{bs} {lens} q{q_len} width {width} {dtype}", flush=True)
    case = make_custom_case(batch=len(lens), num_heads=hq, kv_heads=hkv, head_dim=dim, block_size=bs, q_len=q_len,
                            causal=q_len > 1, context_lens=lens, seed=1200 + hq + dim + bs, dtype=dtype,
                            max_blocks=width)
    assert_close(run(case, device), oracle_numpy(case), what=f"d{dim} bs{bs}")
    pa.check_errors(device)


@pytest.mark.parametrize("bs", [16, 32, 64, 128])
def test_short_fp8_contexts(bs, device):
    case = make_custom_case(batch=3, num_heads=8, kv_heads=2, head_dim=128, block_size=bs, context_lens=[5, 130, 256],
                            seed=1300 + bs)
    case.key_cache, case.k_scale = quantize_kv_fp8(case.key_cache, pow2=False)
    case.value_cache, case.v_scale = quantize_kv_fp8(case.value_cache, pow2=False)
    k = po.dequantize_kv(case.key_cache.view(torch.uint8).numpy(), case.k_scale.numpy())
    v = po.dequantize_kv(case.value_cache.view(torch.uint8).numpy(), case.v_scale.numpy())
    ref = po.paged_attention_decode(case.query.float().numpy(), k, v, case.block_table.numpy(),
                                    case.context_lens.numpy(), case.scale)
    assert_close(run(case, device), ref, what=f"fp8 bs{bs}")


def test_errors_are_reported(device):
    case = make_custom_case(batch=2, num_heads=8, kv_heads=2, head_dim=128, block_size=64, context_lens=[100, 128],
                            seed=1400, max_blocks=2)
    base = run(case, device)
    pa.check_errors(device)
    case.context_lens[1] = 129  # past the table: clamped to 128 and reported
    got = run(case, device)
    assert (got == base).all()
    with pytest.raises(pa.PagedAttentionError) as e:
        pa.check_errors(device)
    assert e.value.rc == -7
    case.context_lens[1] = 128
    case.block_table[0, 1] = 99  # outside the pool: skipped and reported
    run(case, device)
    with pytest.raises(pa.PagedAttentionError) as e:
        pa.check_errors(device)
    assert e.value.rc == -6
    pa.check_errors(device)


# (heads, kv heads, dim, block, table width, lengths); several blocks per wave, so
# a wave's K buffer is written block after block with the next one's loads in
# flight, then holds its partial; waves of shorter sequences end early or idle
@pytest.mark.parametrize("hq,hkv,dim,bs,width,lens", [
    (8, 1, 128, 16, 24, [380, 17, 250]),                             # three blocks for a wave
    (8, 2, 128, 16, 17, [272, 129]),
    (32, 8, 128, 32, 24, [768, 500, 33, 97]),
    (32, 8, 128, 128, 6, [768, 650, 257, 1] + [100 + 40 * i for i in range(12)]),  # 128 tiles, two blocks for a wave
    (32, 8, 128, 16, 48, [768, 250, 641, 0] + [60 * i + 5 for i in range(12)]),
    (8, 4, 256, 16, 16, [256, 241, 100, 129, 17, 1, 255, 64]),
    (4, 2, 256, 128, 2, [206, 100, 130, 256]),                       # blocks larger than the registers, merged
    (32, 8, 256, 128, 2, [206, 100] + [16 * i + 3 for i in range(14)]),
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_several_blocks_per_wave(hq, hkv, dim, bs, width, lens, dtype, device):
    print(f"[case] {hq}/{hkv} d{dim} bs{bs} width {width} {lens} {dtype}", flush=True)
    case = make_custom_case(batch=len(lens), num_heads=hq, kv_heads=hkv, head_dim=dim, block_size=bs,
                            context_lens=lens, seed=1480 + dim + bs + width, dtype=dtype, max_blocks=width)
    d = case.to(device)
    out = torch.full(case.out_shape(), float("nan"), dtype=torch.float32, device=device)
    args = pa.make_args(d.query, d.key_cache, d.value_cache, d.block_table, d.context_lens, out, case.scale)
    assert pa.kernel_name(args) == "pa_direct_kernel"
    pa.launch(args, device)
    assert_close(out.cpu().numpy(), oracle_numpy(case), what=f"d{dim} bs{bs} width {width}")
    pa.check_errors(device)


# (heads, kv heads, dim, block, lengths, cache format); one block per wave
@pytest.mark.parametrize("hq,hkv,dim,bs,lens,kv", [
    (16, 1, 128, 128, [512, 512], "bf16"),
    (8, 2, 128, 128, [500, 129, 384], "bf16"),
    (5, 1, 128, 16, [128, 3, 100], "fp16"),
    (16, 4, 64, 32, [255, 64, 17], "fp16"),
    (16, 2, 256, 64, [256, 70], "bf16"),
    (4, 1, 256, 128, [256, 130], "bf16"),
    (8, 1, 128, 64, [256, 200], "fp8"),
])
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
def test_same_bits_as_the_work_lists(hq, hkv, dim, bs, lens, kv, out_dtype, device):
    """A tile cut into the same pieces (a block each) by the work lists: the
    pieces are the same and are merged in the same order, so the output is too."""
    if kv == "fp16" and out_dtype == torch.bfloat16:
        out_dtype = torch.float16
    print(f"[case] {hq}/{hkv} d{dim} bs{bs} {lens} {kv} {out_dtype}", flush=True)
    case = make_custom_case(batch=len(lens), num_heads=hq, kv_heads=hkv, head_dim=dim, block_size=bs,
                            context_lens=lens, seed=1450 + dim + bs,
                            dtype=torch.float16 if kv == "fp16" else torch.bfloat16)
    if kv == "fp8":
        case.key_cache, case.k_scale = quantize_kv_fp8(case.key_cache, pow2=False)
        case.value_cache, case.v_scale = quantize_kv_fp8(case.value_cache, pow2=False)
    a_worker_per_block = hkv * sum((n + bs - 1) // bs for n in lens)
    d = case.to(device)
    direct, lists = (pa.paged_attention_decode(d.query, d.key_cache, d.value_cache, d.block_table, d.context_lens,
                                               scale=case.scale, out_dtype=out_dtype, num_workers=w,
                                               k_scale=d.k_scale, v_scale=d.v_scale) for w in (0, a_worker_per_block))
    assert torch.equal(direct, lists)
