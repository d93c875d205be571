"""MLA decode with at most 64 query rows (the waves of a workgroup share the
rows): one and two row tiles of 32, partly filled, both block sizes, causal
rows, partial and whole contexts, scales of either sign, and the first row
count of the 128-row form; and short contexts (a workgroup per whole tile)."""

from __future__ import annotations

import pytest
import torch

from simpler_amd import paged_attention as pa
from simpler_amd.workloads import make_custom_case
from tests.pa_helpers import assert_close, oracle_numpy

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bs", [32, 64])
@pytest.mark.parametrize("heads,q_len,lens,workers,scale", [
    (1, 1, [1, 63, 64, 65], 0, None),
    (16, 1, [700, 0, 129], 0, None),
    (16, 2, [2, 33, 500], 1, None),      # one slice: whole tiles
    (16, 4, [4, 64, 900], 7, None),      # 64 rows, causal, cut tiles
    (33, 1, [96, 640], 3, None),         # a second row tile of one row
    (32, 2, [1000], 5, -0.05),
    (16, 1, [300], 2, 0.0),
    (65, 1, [200], 2, None),             # the 128-row form
])
def test_few_rows(bs, heads, q_len, lens, workers, scale, device):
    print(f"[case] heads={heads} q={q_len} bs={bs} lens={lens} w={workers} scale={scale}", flush=True)
    case = make_custom_case(batch=len(lens), num_heads=heads, kv_heads=1, head_dim=576, head_dim_v=512, block_size=bs,
                            q_len=q_len, causal=q_len > 1, context_lens=lens, seed=1500 + heads + bs, mla=True,
                            scale=scale, pool_extra=1)
    d = case.to(device)
    got = pa.paged_attention_decode(d.query, d.key_cache, d.value_cache, d.block_table, d.context_lens,
                                    scale=case.scale, causal=case.config.causal, num_workers=workers)
    assert_close(got.cpu().numpy(), oracle_numpy(case), what=f"mla h{heads} q{q_len} bs{bs}")
    pa.check_errors(device)


@pytest.mark.parametrize("heads,kv_heads,q_len,bs,batch,width,longest", [
    (16, 1, 1, 64, 1, 2, 128),       # the smallest launch
    (16, 1, 2, 64, 3, 2, 128),
    (65, 1, 2, 32, 5, 4, 128),       # two row groups, the second partly filled
    (16, 1, 1, 64, 2, 3, 192),       # too long for two workgroups: work lists
    (33, 1, 1, 64, 32, 4, 256),      # 32 workgroups
    (4, 2, 4, 32, 16, 8, 256),       # two kv heads
    (128, 1, 2, 64, 64, 8, 512),     # 128 workgroups
    (16, 1, 1, 64, 129, 8, 512),
    # the longest whole tiles of each range (those above are just past it)
    (65, 1, 2, 32, 5, 3, 96),
    (33, 1, 1, 64, 32, 3, 192),
    (16, 1, 1, 64, 64, 4, 256),
    (4, 2, 4, 32, 16, 5, 160),
    (128, 1, 2, 64, 64, 6, 384),
    (16, 1, 1, 64, 129, 6, 384),
    (16, 1, 1, 32, 128, 8, 256),
])
def test_whole_tiles(heads, kv_heads, q_len, bs, batch, width, longest, device):
    """Against the oracle and the work lists (a forced worker count)."""
    lens = [max(q_len, longest - 37 * i % longest) for i in range(batch)]
    if batch > 2:
        lens[1] = 0
    lens[0] = longest
    if q_len > 1:
        lens = [max(n, q_len) for n in lens]
    print(f"[case] h={heads} kvh={kv_heads} q={q_len} bs={bs} b={batch} w={width}", flush=True)
    case = make_custom_case(batch=batch, num_heads=heads, kv_heads=kv_heads, head_dim=576, head_dim_v=512,
                            block_size=bs, q_len=q_len, causal=q_len > 1, context_lens=lens, seed=1700 + heads,
                            mla=True)
    assert case.block_table.shape[1] == width
    d = case.to(device)
    outs = []
    for workers in (0, 300):
        out = torch.full((*d.query.shape[:-1], 512), float("nan"), device=device, dtype=torch.float32)
        pa.paged_attention_decode(d.query, d.key_cache, d.value_cache, d.block_table, d.context_lens, out=out,
                                  scale=case.scale, causal=case.config.causal, num_workers=workers)
        outs.append(out)
    assert_close(outs[0].cpu().numpy(), oracle_numpy(case), what=f"whole tiles h{heads} b{batch}")
    # the same block frames, summed in another order
    assert torch.allclose(outs[0], outs[1], rtol=1e-4, atol=1e-5)
    pa.check_errors(device)
    d.context_lens[0] = longest + 1  # past the table: clamped, and reported
    pa.paged_attention_decode(d.query, d.key_cache, d.value_cache, d.block_table, d.context_lens, out=outs[1],
                              scale=case.scale, causal=case.config.causal)
    with pytest.raises(pa.PagedAttentionError):
        pa.check_errors(device)
    assert torch.equal(outs[0], outs[1])


def test_bad_blocks_and_garbage_past_the_context(device):
    case = make_custom_case(batch=2, num_heads=16, kv_heads=1, head_dim=576, head_dim_v=512, block_size=64,
                            context_lens=[200, 70], seed=1600, mla=True, pool_extra=1)
    base = None
    for garbage in (False, True):
        if garbage:
            for b, n in enumerate((200, 70)):
                case.key_cache[int(case.block_table[b, (n - 1) // 64]), n % 64:] = float("nan")
        d = case.to(device)
        got = pa.paged_attention_decode(d.query, d.key_cache, d.value_cache, d.block_table, d.context_lens,
                                        scale=case.scale).cpu()
        assert base is None or torch.equal(got, base)
        base = got
    case.block_table[0, 1] = 1000
    d = case.to(device)
    pa.paged_attention_decode(d.query, d.key_cache, d.value_cache, d.block_table, d.context_lens, scale=case.scale)
    with pytest.raises(pa.PagedAttentionError):
        pa.check_errors(device)
    pa.check_errors(device)
