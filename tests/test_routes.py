"""Which way a decode runs, as the kernel name and the plan report it: work
lists, or one workgroup per tile for short contexts (GQA: pa_direct_kernel; MLA:
whole tiles), on both sides of the rules that decide."""

from __future__ import annotations

import pytest

from simpler_amd import paged_attention as pa
from tests.test_abi import _args, _mla_args

# (heads, kv heads, dim, block size, batch, q_len, table width): the shapes of
# test_direct_gpu.py, and whether they are short enough
GQA = [
    (4, 1, 16, 16, 6, 1, 16, True),
    (16, 2, 64, 16, 3, 1, 32, True),
    (8, 8, 128, 128, 4, 1, 4, True),
    (10, 2, 128, 64, 2, 1, 4, True),
    (8, 1, 128, 32, 3, 1, 8, True),
    (4, 2, 256, 64, 2, 1, 4, True),
    (4, 2, 256, 128, 2, 1, 1, True),
    (40, 2, 128, 16, 2, 1, 8, True),
    (32, 4, 64, 32, 3, 8, 4, True),
    (32, 32, 64, 64, 5, 1, 16, True),
    (16, 1, 128, 128, 2, 1, 5, False),  # two 64 KB blocks for a wave
    (32, 8, 128, 128, 32, 1, 64, False),
    # below 32 tiles: bytes per tile
    (4, 1, 64, 16, 1, 1, 48, True),     # 192 KB, three blocks for a wave
    (4, 1, 64, 16, 1, 1, 49, False),
    (4, 1, 64, 64, 31, 1, 12, True),
    (4, 1, 64, 64, 31, 1, 13, False),
    (4, 1, 128, 16, 31, 1, 32, True),   # 256 KB
    (4, 1, 128, 16, 31, 1, 33, False),
    (16, 4, 256, 16, 4, 1, 8, True),    # one block for a wave
    (16, 4, 256, 16, 4, 1, 9, False),
    (4, 1, 256, 128, 1, 1, 2, True),
    (4, 1, 256, 128, 1, 1, 3, False),
    # from 32 tiles
    (4, 1, 64, 64, 32, 1, 16, True),    # 256 KB
    (4, 1, 64, 64, 32, 1, 17, False),
    (4, 1, 128, 16, 32, 1, 48, True),   # 384 KB
    (4, 1, 128, 16, 32, 1, 49, False),
    (32, 8, 128, 64, 8, 1, 4, True),    # one block for a wave, or 48 KB
    (32, 8, 128, 64, 8, 1, 5, False),
    (16, 4, 256, 16, 8, 1, 16, True),
    (16, 4, 256, 16, 8, 1, 17, False),
    # from 128 tiles
    (32, 8, 128, 128, 16, 1, 6, True),  # 384 KB
    (32, 8, 128, 128, 16, 1, 7, False),
    (32, 8, 64, 16, 16, 1, 64, True),   # 256 KB
    (32, 8, 64, 16, 16, 1, 65, False),
    (32, 8, 256, 64, 16, 1, 6, True),
    (32, 8, 256, 64, 16, 1, 7, False),
    (32, 8, 256, 128, 16, 1, 2, True),  # blocks larger than the registers
    (32, 8, 256, 128, 16, 1, 3, False),
    # the blocks of one wave
    (32, 8, 16, 16, 16, 1, 96, True),   # six of 16 waves
    (32, 8, 16, 16, 16, 1, 97, False),
    (4, 1, 16, 64, 1, 1, 32, True),     # four of 8
    (4, 1, 16, 64, 1, 1, 33, False),
    (4, 1, 16, 128, 1, 1, 12, True),    # three of 4
    (4, 1, 16, 128, 1, 1, 13, False),
    (32, 8, 64, 32, 64, 1, 30, True),   # 512 tiles: ten of 3
    (32, 8, 64, 32, 64, 1, 31, False),
    (32, 8, 128, 64, 256, 1, 6, True),  # 2048 tiles: six of one
    (32, 8, 128, 64, 256, 1, 7, False),
    # several row tiles: 64 KB per tile or 48 MB over all of them
    (128, 8, 64, 32, 32, 4, 8, True),
    (128, 8, 64, 32, 32, 4, 9, False),
    (32, 2, 64, 32, 16, 4, 32, True),
    (128, 8, 64, 128, 24, 4, 2, True),
    (128, 8, 64, 128, 24, 4, 3, False),
    (128, 8, 64, 128, 16, 4, 3, True),
    (16, 1, 128, 16, 1, 4, 24, True),   # 768 KB over four row tiles
    (16, 1, 128, 16, 1, 4, 25, False),
]


def gqa(hq, hkv, d, bs, batch, q_len, width, **kw):
    token = hkv * d
    return _args(num_heads=hq, num_kv_heads=hkv, head_dim_k=d, head_dim_v=d, block_size=bs, batch=batch, q_len=q_len,
                 causal=int(q_len > 1), max_blocks_per_seq=width, k_block_stride=bs * token, v_block_stride=bs * token,
                 k_token_stride=token, v_token_stride=token, k_head_stride=d, v_head_stride=d, **kw)


def check_gqa(hq, hkv, d, bs, batch, q_len, width, short, **kw):
    a = gqa(hq, hkv, d, bs, batch, q_len, width, **kw)
    assert pa.kernel_name(a) == ("pa_direct_kernel" if short else "pa_decode_kernel")
    if short:  # a workgroup per tile
        assert pa.plan(a) == batch * hkv * ((hq // hkv * q_len + 15) // 16)
    a.num_workers = 9  # a forced count keeps the work lists
    assert pa.kernel_name(a) == "pa_decode_kernel" and pa.plan(a) == 9


# (heads, kv heads, batch, q_len, block size, width, whole tiles)
MLA = [
    (16, 1, 1, 1, 64, 2, True),
    (16, 1, 2, 1, 64, 3, False),
    (33, 1, 32, 1, 64, 3, True),     # 192 tokens from 32 workgroups
    (33, 1, 32, 1, 64, 4, False),
    (33, 1, 31, 1, 64, 3, False),
    (16, 1, 64, 1, 64, 4, True),     # 256 from 64
    (16, 1, 64, 1, 64, 5, False),
    (128, 1, 64, 2, 64, 6, True),    # 384 from 128
    (128, 1, 63, 2, 64, 6, False),
    (16, 1, 129, 1, 64, 6, True),
    (16, 1, 129, 1, 64, 7, False),
    # 32-token blocks
    (65, 1, 5, 2, 32, 3, True),
    (96, 1, 7, 1, 32, 4, False),
    (4, 2, 16, 4, 32, 5, True),
    (16, 1, 32, 1, 32, 6, False),
    (16, 1, 64, 1, 32, 6, True),
    (16, 1, 127, 1, 32, 7, False),
    (16, 1, 128, 1, 32, 8, True),
    (16, 1, 128, 1, 32, 9, False),
]


def check_mla(heads, hkv, batch, q_len, bs, width, whole):
    a = _mla_args(num_heads=heads, num_kv_heads=hkv, batch=batch, q_len=q_len, causal=int(q_len > 1), block_size=bs,
                  max_blocks_per_seq=width)
    assert pa.kernel_name(a) == "pa_mla_kernel"
    groups = (heads // hkv * q_len + 127) // 128
    assert pa.plan(a) == (batch * hkv if whole else 256 // groups)
    a.num_workers = 9
    assert pa.plan(a) == 9


@pytest.mark.parametrize("row", GQA)
@pytest.mark.parametrize("kv_format", [pa.KV_BF16, pa.KV_FP16])
def test_gqa(row, kv_format):
    check_gqa(*row, kv_format=kv_format, out_dtype=0)


@pytest.mark.parametrize("row", [
    (8, 1, 128, 16, 1, 1, 48, True), (8, 1, 128, 16, 1, 1, 49, False),   # few tiles: 192 KB
    (64, 8, 128, 32, 16, 1, 32, True), (64, 8, 128, 32, 16, 1, 33, False),  # many: 256 KB
    (128, 8, 128, 64, 128, 8, 4, True), (128, 8, 128, 64, 128, 8, 5, False),  # eight row tiles: 64 KB
])
def test_fp8(row):
    check_gqa(*row, kv_format=pa.KV_FP8_E4M3, out_dtype=0, k_scale=0x7000, v_scale=0x8000)


@pytest.mark.parametrize("row", MLA)
def test_mla(row):
    check_mla(*row)


@pytest.mark.gpu
def test_on_the_device(device):
    """The same with the device's own CU and occupancy figures."""
    for row in GQA:
        check_gqa(*row)
    for row in MLA:
        check_mla(*row)


@pytest.mark.gpu
def test_fp8_workers_by_block_size(device):
    """Eight, four, three and three waves per CU (the default plan of long contexts)."""
    import torch

    cus = torch.cuda.get_device_properties(device).multi_processor_count
    for bs, per_cu in ((16, 8), (32, 4), (64, 3), (128, 3)):
        a = gqa(32, 8, 128, bs, 32, 1, 8192 // bs, kv_format=pa.KV_FP8_E4M3, k_scale=0x7000, v_scale=0x8000)
        assert pa.plan(a) == cus * per_cu
