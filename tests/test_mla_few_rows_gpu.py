"""MLA decode with at most 64 query rows (the waves of a workgroup share the
rows): one and two row tiles of 32, partly filled, both block sizes, causal
rows, partial and whole contexts, scales of either sign, and the first row
count of the 128-row form."""

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
