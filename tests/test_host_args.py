"""The one-pass argument packing of the decode, prelude and append calls
against their checked form: the same bytes for every layout both accept, and
whatever the checks refuse is left to them."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from simpler_amd import kv_cache
from simpler_amd import paged_attention as pa


class OnDevice(torch.Tensor):
    """A CPU tensor that says it is on the device (nothing here reads it)."""

    is_cuda = True
    device = torch.device("cuda", 0)


def dev(*shape, dtype=torch.float32):
    return torch.empty(shape, dtype=dtype).as_subclass(OnDevice)


def decode(dtype=torch.bfloat16, kv=None, out=torch.float32, q_len=1, layout="bsnd", **kw):
    b, hq, hkv, d, bs, n = 3, 8, 2, 64, 16, 5
    kv = kv or dtype
    if layout == "bsnd":
        k, v = dev(n, bs, hkv, d, dtype=kv), dev(n, bs, hkv, d, dtype=kv)
    elif layout == "fused":  # K and V side by side in each block
        both = dev(n, 2, bs, hkv, d, dtype=kv)
        k, v = both[:, 0], both[:, 1]
    elif layout == "head_major":
        k, v = (dev(n, hkv, bs, d, dtype=kv).transpose(1, 2) for _ in range(2))
    else:  # MLA: V is a prefix of K
        k = dev(n, bs, hkv, d, dtype=kv)
        v = k[..., :48]
    q = dev(b, hq, d, dtype=dtype) if q_len == 1 else dev(b, q_len, hq, d, dtype=dtype)
    a = dict(query=q, key_cache=k, value_cache=v, block_table=dev(b, 7, dtype=torch.int32),
             context_lens=dev(b, dtype=torch.int32), out=dev(*q.shape[:-1], v.shape[-1], dtype=out), scale=0.125)
    if kv in (torch.float8_e4m3fn, torch.uint8):
        a.update(k_scale=dev(n, hkv), v_scale=dev(n, hkv))
    a.update(kw)
    return a


def both(fn, module, plain, monkeypatch, args):
    """fn's result by its one-pass form and, with that switched off, by its checks."""
    fast = fn(**args)
    with monkeypatch.context() as m:
        m.setattr(module, plain, lambda *a: None)
        slow = fn(**args)
    return bytes(fast), bytes(slow)


@pytest.mark.parametrize("args", [
    dict(), dict(dtype=torch.float16, out=torch.float16), dict(out=torch.bfloat16, q_len=4, causal=True),
    dict(layout="fused"), dict(layout="head_major", num_workers=7), dict(layout="mla"),
    dict(kv=torch.float8_e4m3fn), dict(kv=torch.uint8, q_len=2), dict(scale=np.float64(0.5)), dict(scale=-1),
    dict(scale=torch.tensor(0.25)), dict(num_workers=np.int32(5)),
])
def test_decode_args_pack_like_the_checked_form(args, monkeypatch):
    a = decode(**args)
    named = dict(causal=False, num_workers=0, k_scale=None, v_scale=None)
    assert pa._plain_args(**{**named, **a}) is not None  # the one-pass form takes it
    fast, slow = both(pa.make_args, pa, "_plain_args", monkeypatch, a)
    assert fast == slow


@pytest.mark.parametrize("change,error", [
    (dict(query=torch.empty(3, 8, 64, dtype=torch.bfloat16)), ValueError),  # on the host
    (dict(query=None), (TypeError, AttributeError)),
    (dict(query=dev(3, 8, 64)), ValueError),
    (dict(query=dev(3, 8, 32, dtype=torch.bfloat16)), ValueError),
    (dict(out=dev(3, 8, 64, dtype=torch.float16)), ValueError),
    (dict(out=dev(3, 64, 8).transpose(1, 2)), ValueError),
    (dict(block_table=dev(3, 7, dtype=torch.int64)), ValueError),
    (dict(block_table=dev(4, 7, dtype=torch.int32)), ValueError),
    (dict(context_lens=dev(6, dtype=torch.int32)[::2]), ValueError),
    (dict(key_cache=dev(5, 16, 64, 2, dtype=torch.bfloat16).transpose(2, 3)), ValueError),
    (dict(value_cache=dev(5, 16, 4, 64, dtype=torch.bfloat16)), ValueError),
    (dict(k_scale=dev(5, 2)), ValueError),
])
def test_decode_args_refuse_what_they_refused(change, error):
    with pytest.raises(error):
        pa.make_args(**{**decode(), **change})


@pytest.mark.parametrize("value", [True, False])
@pytest.mark.parametrize("strided", [True, False])
@pytest.mark.parametrize("err", [True, False])
def test_append_args_pack_like_the_checked_form(value, strided, err, monkeypatch):
    bf = torch.bfloat16
    rows = dev(9, 2, 3, 64, dtype=bf)  # [token, k or v, head, dim]
    key, val = (rows[:, 0], rows[:, 1]) if strided else (dev(9, 3, 64, dtype=bf), dev(9, 3, 64, dtype=bf))
    a = dict(key=key, value=val if value else None, slot_mapping=dev(9, dtype=torch.int32),
             key_cache=dev(4, 16, 3, 64, dtype=bf), value_cache=dev(4, 16, 3, 64, dtype=bf) if value else None,
             error_count=dev(1, dtype=torch.int32) if err else None)
    assert kv_cache._plain_append(**a) is not None
    fast, slow = both(kv_cache.append_args, kv_cache, "_plain_append", monkeypatch, a)
    assert fast == slow


@pytest.mark.parametrize("q_len", [1, 4])
def test_prelude_args_pack_like_the_checked_form(q_len, monkeypatch):
    b, hq, hkv, d, bs, n = 3, 8, 2, 128, 16, 5
    lead = (b,) if q_len == 1 else (b, q_len)
    a = dict(q_proj=dev(*lead, hq, d), k_proj=dev(*lead, hkv, d), v_proj=dev(*lead, hkv, d),
             inv_rms=dev(b * q_len), q_norm_weight=dev(d), k_norm_weight=dev(d), rope_cos=dev(99, d),
             rope_sin=dev(99, d), key_cache=dev(n, bs, hkv, d, dtype=torch.bfloat16),
             value_cache=dev(n, bs, hkv, d, dtype=torch.bfloat16), block_table=dev(b, 7, dtype=torch.int32),
             context_lens=dev(b, dtype=torch.int32), out=dev(*lead, hq, d), scale=0.5, causal=q_len > 1)
    plain = dict(a, num_workers=0)
    args = pa._plain_prelude(**plain)
    assert args is not None
    got, pre = pa.prelude_args(**a)
    assert bytes(got) == bytes(args)
    # the checked form's query view needs device storage: compare with the decode args over a query of that shape
    q = a["q_proj"]
    ref = pa.make_args(dev(*q.shape, dtype=torch.bfloat16), a["key_cache"], a["value_cache"], a["block_table"],
                       a["context_lens"], a["out"], a["scale"], causal=a["causal"])
    ref.query = q.data_ptr()
    assert bytes(got) == bytes(ref)
    assert (pre.q_proj, pre.inv_rms, pre.rope_sin, pre.max_position) == (
        q.data_ptr(), a["inv_rms"].data_ptr(), a["rope_sin"].data_ptr(), 99)
    for name, bad in (("k_proj", dev(*lead, hq, d)), ("rope_sin", dev(98, d)), ("inv_rms", dev(b * q_len + 1)),
                      ("q_norm_weight", dev(d, dtype=torch.float16)), ("v_proj", dev(*lead, d, hkv).transpose(-1, -2))):
        assert pa._plain_prelude(**dict(plain, **{name: bad})) is None
        with pytest.raises(ValueError):
            pa.prelude_args(**dict(a, **{name: bad}))
