"""The split merge at the edges of its launch shapes: tiles of one row up to a
full 16, every output width, and contexts cut into few pieces (one workgroup
per tile), many (several workgroups and groups of threads per tile) and more
than its LDS table of weights holds (1024 per workgroup)."""

from __future__ import annotations

import pytest
import torch

from simpler_amd import paged_attention as pa
from simpler_amd.workloads import make_custom_case
from tests.pa_helpers import assert_close, oracle_numpy

pytestmark = pytest.mark.gpu


# (group, dim, lengths in 16-token blocks, workers)
@pytest.mark.parametrize("group,dim,blocks,workers", [
    (1, 16, [40, 0, 3], 9),        # one row, few pieces; an empty sequence
    (1, 128, [300], 300),          # one row, 300 pieces: 16 groups of threads
    (5, 64, [130, 1], 131),        # an odd row count
    (16, 128, [9, 8], 17),         # as many pieces as are read ahead, one more
    (16, 128, [200], 100),         # a full tile in several workgroups
    (16, 256, [64, 5], 30),
    (16, 256, [130, 7, 1], 3),     # more units than threads, few pieces
    (16, 32, [2300], 5000),        # above the LDS table: 16 rows x 2300 pieces
    (20, 64, [50, 33], 40),        # a second row tile of 4 rows
    # above the LDS table in a batch whose mean is short: one workgroup per tile
    (16, 64, [300] + [1] * 69, 369),
    (16, 16, [300] + [1] * 69, 369),   # several groups of threads
    (5, 128, [2, 500, 0, 1] + [1] * 60, 570),
    (16, 256, [200] + [1] * 599, 799),  # two units per thread
])
def test_pieces_and_rows(group, dim, blocks, workers, device):
    print(f"[case] group={group} dim={dim} blocks={blocks} workers={workers}", flush=True)
    lens = [max(0, 16 * n - 5) for n in blocks]
    case = make_custom_case(batch=len(lens), num_heads=group, kv_heads=1, head_dim=dim, block_size=16,
                            context_lens=lens, seed=900 + group + dim + workers)
    d = case.to(device)
    got = pa.paged_attention_decode(d.query, d.key_cache, d.value_cache, d.block_table, d.context_lens,
                                    scale=case.scale, num_workers=workers)
    assert_close(got.cpu().numpy(), oracle_numpy(case), what=f"g{group} d{dim} w{workers}")
    pa.check_errors(device)


@pytest.mark.parametrize("heads,lens,workers", [
    (16, [3000], 90), (33, [700, 0, 64], 12), (128, [500] * 3, 6),
    (16, [9000] + [32] * 40, 800),    # above the LDS table
    (128, [4800] + [32] * 66, 760),   # the same with four units per thread
])
def test_mla_pieces(heads, lens, workers, device):
    print(f"[case] mla heads={heads} lens={lens} workers={workers}", flush=True)
    case = make_custom_case(batch=len(lens), num_heads=heads, kv_heads=1, head_dim=576, head_dim_v=512, block_size=32,
                            context_lens=lens, seed=950 + heads, mla=True)
    d = case.to(device)
    got = pa.paged_attention_decode(d.query, d.key_cache, d.value_cache, d.block_table, d.context_lens,
                                    scale=case.scale, num_workers=workers)
    assert_close(got.cpu().numpy(), oracle_numpy(case), what=f"mla h{heads} w{workers}")
    pa.check_errors(device)
