"""The measured workloads of this framework: what a serving program has it do.

Six kinds of call, each through a public entry point:

* ``decode``  - one decode step over paged 16-bit or fp8 caches
  (``paged_attention.paged_attention_decode``), also with several causal query
  tokens per sequence (speculative verify);
* ``worker``  - the same step submitted as the reference's paged-attention
  callable (``Worker.register`` / ``Worker.run``) on device-resident tensors;
* ``mla``     - the decode of latent caches (Dk 576, V the first 512 dims of K);
* ``prelude`` - q/k RMS norm, RoPE, KV append and decode in one call
  (``paged_attention.paged_attention_decode_prelude``);
* ``append``  - the KV append of a prefill (``kv_cache.kv_append``).

A case's sizes are plain values; its context lengths are spread evenly at
random over ``len_min .. len_max`` by ``len_draw``, so the work of a case does
not depend on the seed of its values. Values are N(0, 1), scale 1/sqrt(Dk), as
in ``simpler_amd.workloads``.
"""

import ctypes
import math
import random

import torch

from simpler_amd import Worker, kv_cache
from simpler_amd import paged_attention as pa
from simpler_amd.task_interface import ChipStorageTaskArgs, ChipTensor
from simpler_amd.torch_interop import torch_dtype_to_datatype
from simpler_amd.workloads import FP8_MAX, rope_tables

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
MLA_DK, MLA_DV = 576, 512


def _decode(name, batch, heads, kv_heads, dim, block, len_min, len_max, q_len=1, dtype="bf16", kv="16bit", out="bf16",
            pool="one", kind="decode", len_draw=1):
    return {"name": name, "kind": kind, "batch": batch, "heads": heads, "kv_heads": kv_heads, "dim": dim,
            "block": block, "len_min": len_min, "len_max": len_max, "len_draw": len_draw, "q_len": q_len,
            "dtype": dtype, "kv": kv, "out": out, "pool": pool}


def listed():
    return [
        # the smallest call: two short sequences, bound by latency, launches and the call itself
        _decode("decode_small", 2, 16, 1, 128, 128, 512, 512),
        # the flagship: a GQA model of 32 query and 8 KV heads serving 32 sequences, one decode step of a layer
        _decode("decode_serving", 32, 32, 8, 128, 128, 1024, 8192),
        # the same heads in a server that pages its caches in 16 tokens, with caches allocated one by one
        _decode("decode_page16", 24, 32, 8, 128, 16, 150, 6000, pool="two", out="fp32"),
        # the largest: the reference's own timed scene (256 sequences of 8192 tokens, one KV head) through Worker.run
        _decode("worker_unroll", 256, 16, 1, 128, 128, 8192, 8192, out="fp32", pool="two", kind="worker"),
        # a fp16 model with small heads, pages of 32 tokens and an odd batch
        _decode("decode_d64_fp16", 37, 32, 8, 64, 32, 300, 5000, dtype="fp16", out="fp16"),
        # a model with large heads, few sequences
        _decode("decode_d256", 11, 16, 4, 256, 64, 500, 7000),
        # the flagship's step over fp8 caches
        _decode("decode_fp8", 32, 32, 8, 128, 128, 1024, 8192, kv="fp8"),
        # speculative verify: 8 causal query tokens per sequence over long prefixes
        _decode("verify_q8", 16, 32, 8, 128, 128, 2056, 16392, q_len=8),
        # latent attention with all 128 query heads on one GPU (data-parallel attention), a full batch
        _decode("mla_heads128", 128, 128, 1, MLA_DK, 64, 512, 8192, kind="mla"),
        # latent attention with the heads split over 8 GPUs and two query tokens (one speculated)
        _decode("mla_heads16", 32, 16, 1, MLA_DK, 64, 200, 6000, q_len=2, kind="mla"),
        # a whole decode step after the projections: norm, RoPE, cache write and attention in one call
        _decode("prelude_step", 16, 32, 8, 128, 64, 100, 3000, kind="prelude"),
        # the cache write of a prefill of odd length
        _append("prefill_append", 16001, 8, 128, 128),
    ]


def _append(name, tokens, kv_heads, dim, block):
    return {"name": name, "kind": "append", "tokens": tokens, "kv_heads": kv_heads, "dim": dim, "block": block}


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: batches of 1 to 256, lengths of 16 to 32768, every block size, at most 1 GB of cache read."""
    kind = rng.choice(["decode"] * 8 + ["worker", "mla", "mla", "prelude", "append"])
    if kind == "append":
        c = _append("", _log(rng, 1, 32768), rng.choice([1, 2, 4, 8]), rng.choice([64, 128, 256]),
                    rng.choice([16, 32, 64, 128]))
    elif kind == "mla":
        heads, q_len, batch = rng.choice([16, 32, 64, 128]), rng.choice([1, 1, 2, 4]), _log(rng, 1, 128)
        most = min(8192, int(130e9 / (batch * heads * q_len * 2 * (MLA_DK + MLA_DV))))
        c = _lens(rng, _decode("", batch, heads, 1, MLA_DK, rng.choice([32, 64]), 0, 0, q_len, kind="mla",
                               out=rng.choice(["bf16", "fp32"])), most)
    elif kind == "prelude":
        batch, kv_heads = _log(rng, 1, 64), rng.choice([1, 2, 4, 8])
        most = min(8192, int(100e6 / (batch * kv_heads * 256)))  # the caches are among the outputs
        c = _lens(rng, _decode("", batch, kv_heads * rng.choice([1, 2, 4, 5, 8]), kv_heads, 128,
                               rng.choice([16, 32, 64, 128]), 0, 0, rng.choice([1, 1, 2, 4]), kind="prelude"), most)
    else:
        kv_heads, batch = rng.choice([1, 2, 4, 8]), _log(rng, 1, 256)
        heads, dim = kv_heads * rng.choice([1, 2, 4, 5, 7, 8, 16]), rng.choice([64, 128, 128, 128, 256])
        dtype, kv, q_len = rng.choice(["bf16", "bf16", "fp16"]), "16bit", rng.choice([1, 1, 1, 1, 2, 4, 8])
        if kind == "worker":
            q_len = 1
        elif dim == 128 and dtype == "bf16" and rng.random() < 0.25:
            kv = "fp8"
        most = min(32768, int(900e6 / (batch * kv_heads * dim * (2 if kv == "fp8" else 4))))
        c = _lens(rng, _decode("", batch, heads, kv_heads, dim, rng.choice([16, 32, 64, 128]), 0, 0, q_len, dtype, kv,
                               rng.choice([dtype, "fp32"]), rng.choice(["one", "two"]), kind), most)
    del c["name"]
    return c


def _lens(rng, c, most):
    c["len_max"] = _log(rng, 16, max(16, most))
    c["len_min"] = max(c["q_len"], int(c["len_max"] * rng.uniform(0.05, 1.0)))
    c["len_draw"] = rng.randrange(1 << 20)
    return c


def _lengths(c):
    r = random.Random(c["len_draw"])
    return [r.randint(c["len_min"], c["len_max"]) for _ in range(c["batch"])]


def _table(c, lens, gen):
    """A block table whose sequences take blocks all over the pool, as a server's do after a while."""
    per = [(n + c["block"] - 1) // c["block"] for n in lens]
    perm = torch.randperm(sum(per), generator=gen, device="cuda").to(torch.int32)
    table = torch.zeros((c["batch"], max(per)), dtype=torch.int32, device="cuda")
    at = 0
    for b, n in enumerate(per):
        table[b, :n] = perm[at:at + n]
        at += n
    return table, sum(per)


def _randn(shape, gen, dtype=torch.float32):
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32).to(dtype)


def _fill(cache, gen):
    """N(0, 1) into a cache, a part of its blocks at a time."""
    for part in cache.split(max(1, (1 << 27) // max(1, cache[0].numel()))):
        part.copy_(_randn(part.shape, gen))


def _quantized(cache):
    """E4M3FN blocks with one fp32 scale per (block, kv head) that maps the block's largest value to the format's."""
    scale = cache.abs().amax(dim=(1, 3)).float() / FP8_MAX
    return (cache.float() / scale[:, None, :, None]).to(torch.float8_e4m3fn), scale.contiguous()


class _Program:
    """The worker and the registered callable that a program on the reference's API keeps."""

    worker = None

    @classmethod
    def get(cls):
        if cls.worker is None:
            cls.worker = Worker(level=2, platform="mi355x", device_id=torch.cuda.current_device()).init()
            cls.handle = cls.worker.register(pa.reference_callable("paged_attention_unroll"))
        return cls.worker, cls.handle


def prepare(case, seed):
    c, gen = dict(case), torch.Generator("cuda").manual_seed(seed)
    if c["kind"] == "append":
        blocks = (c["tokens"] + c["block"] - 1) // c["block"] + 3
        k, v = kv_cache.alloc_kv_pools(blocks, c["block"], c["kv_heads"], c["dim"])
        k.zero_(), v.zero_()
        # a prefill's positions in order, its blocks anywhere in the pool
        order = torch.randperm(blocks, generator=gen, device="cuda")
        pos = torch.arange(c["tokens"], device="cuda")
        slots = (order[pos // c["block"]] * c["block"] + pos % c["block"]).to(torch.int32)
        shape = (c["tokens"], c["kv_heads"], c["dim"])
        return {"kind": "append", "key": _randn(shape, gen, torch.bfloat16), "value": _randn(shape, gen, torch.bfloat16),
                "slots": slots, "k": k, "v": v}
    lens = _lengths(c)
    table, blocks = _table(c, lens, gen)
    dtype, q_len, dim = DTYPES[c["dtype"]], c["q_len"], c["dim"]
    s = {"kind": c["kind"], "table": table, "lens": torch.tensor(lens, dtype=torch.int32, device="cuda"),
         "scale": 1.0 / math.sqrt(dim), "causal": q_len > 1, "k_scale": None, "v_scale": None}
    rows = (c["batch"], q_len, c["heads"]) if q_len > 1 else (c["batch"], c["heads"])
    if c["kind"] == "mla":
        s["k"] = torch.empty((blocks, c["block"], 1, dim), dtype=dtype, device="cuda")
        _fill(s["k"], gen)
        s["v"] = s["k"][..., :MLA_DV]
    else:
        if c["pool"] == "one":
            s["k"], s["v"] = kv_cache.alloc_kv_pools(blocks, c["block"], c["kv_heads"], dim, dtype)
        else:
            s["k"], s["v"] = (torch.empty((blocks, c["block"], c["kv_heads"], dim), dtype=dtype, device="cuda")
                              for _ in range(2))
        _fill(s["k"], gen), _fill(s["v"], gen)
        if c["kv"] == "fp8":
            (k8, s["k_scale"]), (v8, s["v_scale"]) = _quantized(s["k"]), _quantized(s["v"])
            s["k"], s["v"] = kv_cache.alloc_kv_pools(blocks, c["block"], c["kv_heads"], dim, torch.float8_e4m3fn)
            s["k"].copy_(k8), s["v"].copy_(v8)
    s["out"] = torch.empty((*rows, s["v"].shape[-1]), dtype=DTYPES[c["out"]], device="cuda")
    if c["kind"] == "prelude":
        kv_rows = (*rows[:-1], c["kv_heads"], dim)
        s["q_proj"], s["k_proj"], s["v_proj"] = _randn((*rows, dim), gen), _randn(kv_rows, gen), _randn(kv_rows, gen)
        s["inv_rms"] = 0.5 + torch.rand(c["batch"] * q_len, generator=gen, device="cuda")
        s["q_w"], s["k_w"] = 1 + 0.1 * _randn((dim,), gen), 1 + 0.1 * _randn((dim,), gen)
        s["cos"], s["sin"] = (t.cuda() for t in rope_tables(c["len_max"] + 1, dim))
        return s
    s["q"] = _randn((*rows, dim), gen, dtype)
    if c["kind"] == "worker":
        s["worker"], s["handle"] = _Program.get()
        s["args"] = ChipStorageTaskArgs()
        for t in (s["q"], s["k"], s["v"], s["table"], s["lens"], s["out"]):
            s["args"].add_tensor(ChipTensor.make(t.data_ptr(), tuple(t.shape), torch_dtype_to_datatype(t.dtype),
                                                 child_memory=True, strides=tuple(t.stride())))
        s["args"].add_scalar(ctypes.c_float(s["scale"]))
    return s


def run(s):
    if s["kind"] == "append":
        kv_cache.kv_append(s["key"], s["value"], s["slots"], s["k"], s["v"])
        return {"k": s["k"], "v": s["v"]}
    if s["kind"] == "worker":
        s["worker"].run(s["handle"], s["args"])
        return s["out"]
    if s["kind"] == "prelude":
        pa.paged_attention_decode_prelude(s["q_proj"], s["k_proj"], s["v_proj"], s["inv_rms"], s["q_w"], s["k_w"],
                                          s["cos"], s["sin"], s["k"], s["v"], s["table"], s["lens"], s["out"],
                                          s["scale"], causal=s["causal"])
        return {"out": s["out"], "k": s["k"], "v": s["v"]}
    return pa.paged_attention_decode(s["q"], s["k"], s["v"], s["table"], s["lens"], s["out"], s["scale"],
                                     causal=s["causal"], k_scale=s["k_scale"], v_scale=s["v_scale"])


def work(case):
    c = case
    if c["kind"] == "append":
        return {"bytes": c["tokens"] * (8 * c["kv_heads"] * c["dim"] + 4), "flops": 0}
    lens, mla = _lengths(c), c["kind"] == "mla"
    dv = MLA_DV if mla else c["dim"]
    tokens, blocks = sum(lens), sum((n + c["block"] - 1) // c["block"] for n in lens)
    rows = c["batch"] * c["q_len"] * c["heads"]
    if c["kv"] == "fp8":
        kv = tokens * c["kv_heads"] * 2 * c["dim"] + 8 * c["kv_heads"] * blocks
    else:
        kv = tokens * c["kv_heads"] * 2 * (c["dim"] if mla else 2 * c["dim"])
    q = rows * c["dim"] * 2
    if c["kind"] == "prelude":  # fp32 projections and RoPE rows; the new rows are written to the caches besides
        new = c["batch"] * c["q_len"]
        q = 4 * (rows * c["dim"] + new * (2 * c["kv_heads"] * c["dim"] + 2 * c["dim"] + 1))
    pairs = sum(c["q_len"] * n - c["q_len"] * (c["q_len"] - 1) // 2 for n in lens)  # causal
    return {"bytes": kv + q + rows * dv * DTYPES[c["out"]].itemsize + 4 * (blocks + c["batch"]),
            "flops": pairs * c["heads"] * 2 * (c["dim"] + dv)}


def tolerance(case):
    """About four times the error measured against ``exact``: p and the output are rounded to the input's type (8
    bits of mantissa: 0.0010 with fp32 output to 0.0022; 11 bits: 0.00025), the prelude's query and keys too (0.0027)."""
    if case["kind"] == "append":
        return "exact"
    return {"rel": 0.001 if case["dtype"] == "fp16" else 0.011 if case["kind"] == "prelude" else 0.009}


def _norm_rope(x, inv_rms, w, cos, sin):
    """x [..., heads, D] float64 (inv_rms, cos and sin per token): RMS norm with weight w, half-split RoPE."""
    x = x * inv_rms[..., None, None]
    x = x / torch.sqrt((x * x).mean(-1, keepdim=True) + kv_cache.EPS) * w
    lo, hi = x.chunk(2, dim=-1)
    return x * cos[..., None, :] + torch.cat([-hi, lo], dim=-1) * sin[..., None, :]


def exact(case, seed):
    """What ``run`` returns, in plain torch and 64 bits."""
    c, s = case, prepare(dict(case, kind="decode") if case["kind"] == "worker" else case, seed)
    if c["kind"] == "append":
        at = s["slots"].long()
        for cache, new in ((s["k"], s["key"]), (s["v"], s["value"])):
            cache.view(-1, c["kv_heads"], c["dim"])[at] = new
        return {"k": s["k"], "v": s["v"]}
    lens, block, q_len, hkv = s["lens"].tolist(), c["block"], c["q_len"], c["kv_heads"]
    group = c["heads"] // hkv
    k_all, v_all = s["k"], s["v"]
    if c["kind"] == "prelude":
        k_all, v_all = k_all.double(), v_all.double()
        shape = (c["batch"], q_len)
        pos = s["lens"].long()[:, None] - q_len + torch.arange(q_len, device="cuda")
        inv, cos, sin = s["inv_rms"].double().view(shape), s["cos"].double()[pos], s["sin"].double()[pos]
        q_all = _norm_rope(s["q_proj"].double().view(*shape, c["heads"], -1), inv, s["q_w"].double(), cos, sin)
        blk, off = torch.gather(s["table"].long(), 1, pos // block), pos % block
        k_all[blk, off] = _norm_rope(s["k_proj"].double().view(*shape, hkv, -1), inv, s["k_w"].double(), cos, sin)
        v_all[blk, off] = s["v_proj"].double().view(*shape, hkv, -1) * inv[..., None, None]
    else:
        q_all = s["q"].double().view(c["batch"], q_len, c["heads"], -1)
    dv = v_all.shape[-1]
    out = torch.empty((c["batch"], q_len, c["heads"], dv), dtype=torch.float64, device="cuda")
    for b, n in enumerate(lens):
        ids = s["table"][b, :(n + block - 1) // block].long()
        k, v = k_all[ids].double(), v_all[ids].double()
        if c["kv"] == "fp8":
            k, v = k * s["k_scale"][ids].double()[:, None, :, None], v * s["v_scale"][ids].double()[:, None, :, None]
        k = k.reshape(-1, hkv, k.shape[-1])[:n].transpose(0, 1).contiguous()
        v = v.reshape(-1, hkv, dv)[:n].transpose(0, 1).contiguous()
        q = q_all[b].view(q_len, hkv, group, -1).transpose(0, 1).reshape(hkv, q_len * group, -1)
        x = torch.matmul(q, k.transpose(1, 2).contiguous()) * s["scale"]
        seen = n - (q_len - 1) + torch.arange(q_len, device="cuda").repeat_interleave(group)  # tokens row r sees
        x = x.masked_fill(torch.arange(n, device="cuda")[None, None, :] >= seen[None, :, None], -math.inf)
        o = torch.matmul(torch.softmax(x, dim=-1), v)
        out[b] = o.view(hkv, q_len, group, dv).transpose(0, 1).reshape(q_len, c["heads"], dv)
    out = out.view(s["out"].shape)
    return {"out": out, "k": k_all, "v": v_all} if c["kind"] == "prelude" else out
