"""What a user of this framework has it do, as cases that can be timed and compared.

A case is one layer's share of an engine step, through the calls the model's attention layer makes: the cache update
of the step's new tokens and the attention over the paged cache (``Int8AttentionImpl``, ``Int8MLAImpl`` with
``Int8MLADecodeCaller``), or the movement of cache blocks between the GPU and pinned host memory (``swap_blocks``).
What an engine keeps from step to step or shares between the layers of a step -- the cache with its context, the
weights, the metadata of the batch -- is made in ``prepare``.

Sequence lengths are drawn from the case's own ``lengths`` number, values from the seed, so every input of one case
has the same shape.  Keys have a hundredth of their channels twenty times larger, as trained models have.
"""
from __future__ import annotations

import math
import os
import random
import sys
import types

import torch

sys.path.insert(1, os.path.abspath("vllm-metax_amd"))

from vllm_metax_amd import _custom_ops as ops  # noqa: E402
from vllm_metax_amd import layout as L  # noqa: E402
from vllm_metax_amd.v1.attention.backends import int8_attn as gqa  # noqa: E402
from vllm_metax_amd.v1.attention.backends.mla import int8_mla as mla  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
R, ROPE, NOPE, VDIM = 512, 64, 128, 128   # the MLA layer's widths
MAX_NUM_SEQS = 256                        # what the metadata builders reserve for


def _gqa(name, **kw):
    """A GQA layer.  ``decodes`` sequences of ``ctx_lo..ctx_hi`` tokens with one new token each come first, then
    ``runs`` sequences with ``new_lo..new_hi`` new tokens on ``cached_lo..cached_hi`` cached ones."""
    case = dict(name=name, kind="gqa", hq=32, hkv=8, d=128, block=16, kv="int8", dtype="bf16", window=0, softcap=0.0,
                one_launch=False, decodes=0, ctx_lo=0, ctx_hi=0, runs=0, new_lo=0, new_hi=0, cached_lo=0, cached_hi=0,
                lengths=1)
    case.update(kw)
    return case


def _mla(name, **kw):
    """An MLA layer: ``decodes`` sequences, or ``runs`` prefills, as above."""
    case = dict(name=name, kind="mla", heads=128, block=64, dtype="bf16", decodes=0, ctx_lo=0, ctx_hi=0, runs=0,
                new_lo=0, new_hi=0, cached_lo=0, cached_hi=0, lengths=1)
    case.update(kw)
    return case


def listed():
    return [
        # one user, a short chat: the smallest call, nothing but latency
        _gqa("decode b1 ctx337", decodes=1, ctx_lo=337, ctx_hi=337),
        # a loaded server's decode step, the headline workload
        _gqa("decode b64 1k-8k", decodes=64, ctx_lo=1024, ctx_hi=8192),
        # long documents, the cache update inside the attention launch
        _gqa("decode b8 32k-128k", decodes=8, ctx_lo=32768, ctx_hi=131072, one_launch=True),
        # wide heads, sliding window and soft cap, fp8 codes, fp16 activations, an odd batch
        _gqa("decode b37 d256 fp8 window", hq=16, hkv=8, d=256, kv="fp8", dtype="fp16", window=4096, softcap=50.0,
             decodes=37, ctx_lo=200, ctx_hi=6500),
        # many short conversations on an int4 cache, few kv heads
        _gqa("decode b200 int4 hkv4", hq=28, hkv=4, kv="int4", decodes=200, ctx_lo=60, ctx_hi=2000),
        # a mixed step: four 2048-token prefill chunks on 0-6k cached tokens beside 60 decode rows
        _gqa("mixed 60 decodes 4x2048", hq=28, hkv=4, decodes=60, ctx_lo=512, ctx_hi=4096, runs=4, new_lo=2048,
             new_hi=2048, cached_lo=0, cached_hi=6144),
        # one request's 512-token chunk of a long prompt
        _gqa("chunk 512 on 32k", runs=1, new_lo=512, new_hi=512, cached_lo=32768, cached_hi=32768),
        # a speculative-decoding step: a few draft tokens per sequence to verify
        _gqa("verify b24 q2-6 1k-8k", runs=24, new_lo=2, new_hi=6, cached_lo=1024, cached_hi=8192),
        # an MLA decode step with all heads on one GPU
        _mla("mla decode b32 h128 ctx4096", decodes=32, ctx_lo=4096, ctx_hi=4096),
        # the same layer on one of eight tensor-parallel shards, a small ragged batch
        _mla("mla decode b7 h16 ragged", heads=16, decodes=7, ctx_lo=100, ctx_hi=3000),
        # MLA prefill: new tokens of several requests, most of them with cached context
        _mla("mla prefill 4 runs h128", runs=4, new_lo=300, new_hi=1500, cached_lo=0, cached_hi=4000),
        # a preempted request's blocks go to pinned host memory and another's come back
        dict(name="swap 192 blocks", kind="swap", blocks=192, hkv=8, d=128, block=16, kv="int8"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _span(rng, lo, hi):
    a, b = sorted((_log(rng, lo, hi), _log(rng, lo, hi)))
    return a, b


def _draw(rng):
    heads = rng.choice([(32, 8, 128), (28, 4, 128), (32, 8, 64), (16, 8, 256), (16, 2, 128), (32, 16, 128), (16, 1, 128)])
    g = dict(zip(("hq", "hkv", "d"), heads), kv=rng.choice(["int8", "int8", "fp8", "int4"]),
             dtype=rng.choice(["bf16", "bf16", "fp16"]), block=rng.choice([16, 16, 32, 64]),
             lengths=rng.randrange(1 << 20))
    if rng.random() < 0.25:
        g.update(window=_log(rng, 500, 5000), softcap=rng.choice([0.0, 50.0]))
    m = dict(heads=rng.choice([16, 16, 32, 64, 128, 128]), block=rng.choice([16, 64]), dtype=rng.choice(["bf16", "bf16", "fp16"]),
             lengths=rng.randrange(1 << 20))
    what = rng.choice(["decode", "decode", "decode", "mixed", "chunk", "verify", "mla decode", "mla decode",
                       "mla prefill", "swap"])
    if what == "decode":
        lo, hi = _span(rng, 40, 120000)
        return _gqa("", decodes=_log(rng, 1, 250), ctx_lo=lo, ctx_hi=hi, one_launch=rng.random() < 0.4, **g)
    if what == "mixed":
        lo, hi = _span(rng, 100, 8000)
        nlo, nhi = _span(rng, 60, 3000)
        return _gqa("", decodes=_log(rng, 1, 150), ctx_lo=lo, ctx_hi=hi, runs=_log(rng, 1, 8), new_lo=nlo, new_hi=nhi,
                    cached_lo=0, cached_hi=_log(rng, 16, 8000), **g)
    if what == "chunk":
        n, c = _log(rng, 64, 2048), _log(rng, 4000, 60000)
        return _gqa("", runs=1, new_lo=n, new_hi=n, cached_lo=c, cached_hi=c, **g)
    if what == "verify":
        lo, hi = _span(rng, 100, 16000)
        return _gqa("", runs=_log(rng, 1, 100), new_lo=2, new_hi=rng.randint(2, 8), cached_lo=lo, cached_hi=hi, **g)
    if what == "mla decode":
        lo, hi = _span(rng, 60, 30000)
        return _mla("", decodes=_log(rng, 1, 200), ctx_lo=lo, ctx_hi=hi, **m)
    if what == "mla prefill":
        nlo, nhi = _span(rng, 50, 3000)
        return _mla("", runs=_log(rng, 1, 8), new_lo=nlo, new_hi=nhi, cached_lo=0, cached_hi=_log(rng, 16, 8000), **m)
    return dict(kind="swap", blocks=_log(rng, 4, 600), hkv=g["hkv"], d=g["d"], block=g["block"], kv=g["kv"])


def draw(rng):
    """One more case of the listed kinds, within the cost of the largest listed one."""
    while True:
        case = _draw(rng)
        case.pop("name", None)
        w = work(case)
        if w["bytes"] <= 1.2e9 and w["flops"] <= 2.5e11:
            return case


# --- shapes -------------------------------------------------------------------------------------------------------

def _sequences(case):
    """(cached tokens, new tokens) of every sequence, decode rows first."""
    r = random.Random(case["lengths"])
    seqs = [(r.randint(case["ctx_lo"], case["ctx_hi"]) - 1, 1) for _ in range(case["decodes"])]
    for _ in range(case["runs"]):
        new = r.randint(case["new_lo"], case["new_hi"])
        seqs.append((r.randint(case["cached_lo"], case["cached_hi"]), new))
    return seqs


def _record_bytes(case):
    return 2 * ((case["d"] // 2 if case["kv"] == "int4" else case["d"]) + 4)


def _visible(cached, new, window):
    """(keys that any query of the run sees, (query, key) pairs)."""
    if not window:
        return cached + new, new * cached + new * (new + 1) // 2
    return min(cached + new, window + new - 1), sum(min(window, cached + i + 1) for i in range(new))


def work(case):
    if case["kind"] == "swap":   # read once and written once, in either direction
        return {"bytes": 4 * case["blocks"] * case["block"] * case["hkv"] * _record_bytes(case), "flops": 0}
    seqs = _sequences(case)
    new = sum(n for _, n in seqs)
    tables = sum(4 * -(-(c + n) // case["block"]) + 8 for c, n in seqs) + 8 * new
    if case["kind"] == "gqa":
        hq, hkv, d, rec = case["hq"], case["hkv"], case["d"], _record_bytes(case)
        seen = [_visible(c, n, case["window"]) for c, n in seqs]
        return {"bytes": sum(k for k, _ in seen) * hkv * rec + new * (2 * hq * d * 2 + 2 * hkv * d * 2 + hkv * rec) + tables,
                "flops": 4 * d * hq * sum(p for _, p in seen)}
    h = case["heads"]
    tokens = sum(c + n for c, n in seqs)
    pairs = sum(_visible(c, n, 0)[1] for c, n in seqs)
    row = R + ROPE + 4
    if case["decodes"]:
        return {"bytes": tokens * row + new * (h * (NOPE + ROPE + VDIM) * 2 + h * 4 + (R + ROPE) * 2 + row)
                + h * R * (NOPE + VDIM) * 2 + tables,
                "flops": 2 * new * h * R * (NOPE + VDIM) + 2 * pairs * h * (R + ROPE + R)}
    return {"bytes": (tokens - new) * row + new * (h * (NOPE + ROPE + VDIM) * 2 + (R + ROPE) * 2 + row)
            + h * R * (NOPE + VDIM) * 2 + tables,
            "flops": 2 * tokens * h * R * (NOPE + VDIM) + 2 * pairs * h * (NOPE + ROPE + VDIM)}


def tolerance(case):
    """Cache bytes are the same; attention outputs are bf16 or fp16 rows of fp32 sums whose operands have 8 to 11 bits."""
    return "exact" if case["kind"] == "swap" else {"rel": 1e-2}


# --- state --------------------------------------------------------------------------------------------------------

def _batch(case, block, dev):
    """The batch's metadata as an engine hands it to the builders, and the slots of cached and new tokens."""
    seqs = _sequences(case)
    r = random.Random(case["lengths"] + 1)
    need = [-(-(c + n) // block) for c, n in seqs]
    num_blocks = sum(need) + sum(need) // 16 + 9   # block 0 stays the null block, a few are free
    ids = list(range(1, num_blocks))
    r.shuffle(ids)
    ids = torch.tensor(ids, dtype=torch.int32)
    table = torch.zeros((len(seqs), max(need)), dtype=torch.int32)
    at = 0
    for i, n in enumerate(need):
        table[i, :n] = ids[at:at + n]
        at += n
    table_d = table.to(dev)
    old, fresh = [], []
    for i, (c, n) in enumerate(seqs):
        pos = torch.arange(c + n, device=dev)
        slots = table_d[i, pos // block].to(torch.int64) * block + pos % block
        old.append(slots[:c])
        fresh.append(slots[c:])
    starts = torch.tensor([0] + [n for _, n in seqs], dtype=torch.int32).cumsum(0).to(torch.int32)
    lens = torch.tensor([c + n for c, n in seqs], dtype=torch.int32)
    common = types.SimpleNamespace(
        num_reqs=len(seqs), num_actual_tokens=int(starts[-1]), max_query_len=max(n for _, n in seqs),
        max_seq_len=int(lens.max()), query_start_loc=starts.to(dev), query_start_loc_cpu=starts, seq_lens=lens.to(dev),
        seq_lens_cpu=lens, block_table_tensor=table_d, slot_mapping=torch.cat(fresh).contiguous(), causal=True)
    return common, torch.cat(old).contiguous(), num_blocks


def _config(num_q_heads, **spec):
    spec = types.SimpleNamespace(num_q_heads=num_q_heads, **spec)
    return spec, types.SimpleNamespace(scheduler_config=types.SimpleNamespace(max_num_seqs=MAX_NUM_SEQS))


def _prepare_gqa(case, rand, dev):
    hq, hkv, d, block, dtype = case["hq"], case["hkv"], case["d"], case["block"], DTYPES[case["dtype"]]
    kv_dtype = case["kv"] + "_per_token_head"
    backend = gqa.Int8FusedUpdateAttentionBackend if case["one_launch"] else gqa.Int8AttentionBackend
    impl = backend.get_impl_cls()(hq, d, d ** -0.5, hkv, sliding_window=case["window"] or None, kv_cache_dtype=kv_dtype,
                                  logits_soft_cap=case["softcap"] or None)
    common, old, num_blocks = _batch(case, block, dev)
    loud = 1 + 19 * (torch.rand((hkv, d), generator=rand, device=dev) < 0.01).to(dtype)

    def rows(n, heads, scale=None):
        x = torch.randn((n, heads, d), generator=rand, device=dev, dtype=dtype)
        return x if scale is None else x * scale

    cache = L.allocate_kv_cache(num_blocks, block, hkv, d, device=dev, cache_dtype_str=kv_dtype)
    layer = types.SimpleNamespace()
    for part in old.split(65536):
        impl.do_kv_cache_update(layer, rows(part.numel(), hkv, loud), rows(part.numel(), hkv), cache, part)
    spec, config = _config(hq, block_size=block, num_kv_heads=hkv, head_size=d)
    n = common.num_actual_tokens
    q = rows(n, hq).view(n, hq * d)
    return dict(kind="gqa", impl=impl, layer=layer, cache=cache, q=q, k=rows(n, hkv, loud), v=rows(n, hkv),
                out=torch.empty_like(q), update=not backend.forward_includes_kv_cache_update,
                md=backend.get_builder_cls()(spec, ["layer.0"], config, dev).build(0, common))


def _prepare_mla(case, rand, dev):
    h, block, dtype = case["heads"], case["block"], DTYPES[case["dtype"]]

    def rows(*shape, scale=1.0):
        return torch.randn(shape, generator=rand, device=dev, dtype=dtype) * scale

    weight = rows(h * (NOPE + VDIM), R, scale=R ** -0.5)   # kv_b_proj
    impl = mla.Int8MLAImpl(h, R + ROPE, (NOPE + ROPE) ** -0.5, kv_lora_rank=R, qk_rope_head_dim=ROPE,
                           qk_nope_head_dim=NOPE, v_head_dim=VDIM,
                           kv_b_proj=lambda x: torch.nn.functional.linear(x, weight))
    common, old, num_blocks = _batch(case, block, dev)
    cache = L.allocate_mla_cache(num_blocks, block, R + ROPE, device=dev)
    for part in old.split(65536):
        impl.do_kv_cache_update(rows(part.numel(), R), rows(part.numel(), ROPE), cache, part)
    spec, config = _config(h, block_size=block, kv_lora_rank=R)
    config.model_config = types.SimpleNamespace(dtype=dtype, max_model_len=8192)
    md = mla.Int8MLABackend.get_builder_cls()(spec, ["layer.0"], config, dev).build(0, common)
    n = common.num_actual_tokens
    state = dict(impl=impl, cache=cache, md=md, kv_c=rows(n, R), k_pe=rows(n, 1, ROPE),
                 out=torch.empty((n, h * VDIM), dtype=dtype, device=dev))
    if not case["decodes"]:
        return dict(state, kind="mla prefill", q=rows(n, h, NOPE + ROPE))
    per_head = weight.view(h, NOPE + VDIM, R)
    caller = mla.Int8MLADecodeCaller(impl, per_head[:, :NOPE].contiguous(), per_head[:, NOPE:].transpose(1, 2).contiguous())
    return dict(state, kind="mla decode", caller=caller, q_nope=rows(n, h, NOPE), q_pe=rows(n, h, ROPE))


def _prepare_swap(case, rand, dev):
    n = case["blocks"]
    cache = L.allocate_kv_cache(4 * n + 1, case["block"], case["hkv"], case["d"], device=dev, fill=None,
                                cache_dtype_str=case["kv"] + "_per_token_head")
    cache.view(torch.uint8).random_(0, 256, generator=rand)
    host = torch.empty((3 * n,) + tuple(cache.shape[1:]), dtype=torch.int8, pin_memory=True)
    host.copy_(cache[:3 * n])
    r = random.Random(n)
    ids = r.sample(range(1, 4 * n + 1), 2 * n)
    at = r.sample(range(3 * n), 2 * n)
    return dict(kind="swap", cache=cache, host=host, nbytes=cache[0].numel(),
                out=torch.tensor(list(zip(ids[:n], at[:n])), dtype=torch.int64),
                back=torch.tensor(list(zip(at[n:], ids[n:])), dtype=torch.int64))


def prepare(case, seed):
    dev = torch.device("cuda", torch.cuda.current_device())
    rand = torch.Generator(device=dev)
    rand.manual_seed(seed)
    return {"gqa": _prepare_gqa, "mla": _prepare_mla, "swap": _prepare_swap}[case["kind"]](case, rand, dev)


def run(s):
    if s["kind"] == "gqa":
        if s["update"]:
            s["impl"].do_kv_cache_update(s["layer"], s["k"], s["v"], s["cache"], s["md"].slot_mapping)
        s["impl"].forward(s["layer"], s["q"], s["k"], s["v"], s["cache"], s["md"], s["out"])
        return s["out"], s["cache"]
    if s["kind"] == "swap":
        ops.swap_blocks(s["cache"], s["host"], s["nbytes"], s["out"])
        ops.swap_blocks(s["host"], s["cache"], s["nbytes"], s["back"])
        return s["cache"], s["host"]
    s["impl"].do_kv_cache_update(s["kv_c"], s["k_pe"], s["cache"], s["md"].slot_mapping)
    if s["kind"] == "mla prefill":
        s["impl"].forward_mha(s["q"], s["kv_c"], s["k_pe"], s["cache"], s["md"], output=s["out"])
        return s["out"], s["cache"]
    lse = s["caller"].forward_decode(s["q_nope"], s["q_pe"], s["cache"], s["md"], s["out"])
    return s["out"], lse, s["cache"]
