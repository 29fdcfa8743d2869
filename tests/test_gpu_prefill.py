"""GPU parity of chunked prefill and mixed decode + prefill batches over the int8 cache, through
the C ABI's varlen entry point, against the oracle (causal attention of a query run of q_len
tokens that ends at the sequence end; the run's own K/V are already in the cache, as in the
unified attention op the reference calls, vllm_metax/v1/attention/backends/triton_attn.py:688-725,
and in its test oracle, tests/kernels/attention/test_triton_unified_attention.py:26-78)."""
import math

import pytest
import torch

import kvq_testlib as T
import oracle
from vllm_metax_amd import _custom_ops as ops
from vllm_metax_amd import layout as L

pytestmark = pytest.mark.gpu


def build(ctx_lens, q_lens, hq, hkv, d, bs, layout="NHD", seed=0, q_dtype=torch.bfloat16, outlier=False):
    g = torch.Generator().manual_seed(seed)
    nb = sum((c + bs - 1) // bs for c in ctx_lens) + 5
    kv, views, lay = T.cpu_cache(nb, bs, hkv, d, layout)
    T.storage_bytes(kv).fill_(0xFF)                    # NaN scales wherever nothing is written
    bt = T.make_block_tables(ctx_lens, bs, nb, g)
    mk = (lambda c: T.outlier_sources((c, hkv, d), g, torch.bfloat16)) if outlier else \
         (lambda c: torch.randn((c, hkv, d), generator=g).to(torch.bfloat16))
    T.fill_cache_from_sources(kv, lay, bt, ctx_lens, bs, [mk(c) for c in ctx_lens], [mk(c) for c in ctx_lens])
    q = torch.randn((sum(q_lens), hq, d), generator=g).to(q_dtype)
    sl = torch.tensor(ctx_lens, dtype=torch.int32)
    cu = torch.tensor([0] + torch.tensor(q_lens).cumsum(0).tolist(), dtype=torch.int32)
    return kv, lay, bt, q, sl, cu


def run(dev, kv_cpu, layout, bt, q, sl, cu, max_q, scale, out_dtype=None, want_lse=False, causal=True):
    kv = T.to_device_cache(kv_cpu, dev, layout)
    k, v = L.key_value_views(kv)
    ks, vs = L.scale_views(kv)
    out = torch.full(q.shape, float("nan"), dtype=out_dtype or q.dtype, device=dev)
    lse = torch.full(q.shape[:2], float("nan"), dtype=torch.float32, device=dev) if want_lse else None
    ops.unified_attention(q.to(dev), k, v, out, cu.to(dev), max_q, sl.to(dev), int(sl.max()), scale, causal,
                          block_table=bt.to(dev), k_scale_cache=ks, v_scale_cache=vs, lse=lse)
    torch.cuda.synchronize()
    return (out, lse) if want_lse else out


@pytest.mark.parametrize("hq,hkv,d,bs", [
    (28, 4, 128, 16),     # Qwen2-7B: 7 q heads per kv head (columns do not fill the MFMA tile evenly)
    (32, 8, 128, 16),     # Llama-3-8B
    (8, 8, 64, 32),       # no grouping
    (16, 1, 128, 16),     # 16 q heads on one kv head
    (4, 2, 256, 16),
])
def test_mixed_batch_matches_oracle(gpu_device, hq, hkv, d, bs):
    ctx = [700, 33, 129, 64, 257, 5]
    qls = [1, 33, 100, 1, 17, 5]      # decode rows, a pure prefill, chunks with context, a short full run
    kv, lay, bt, q, sl, cu = build(ctx, qls, hq, hkv, d, bs, seed=hq + d)
    scale = 1 / math.sqrt(d)
    want, want_lse = oracle.paged_attn(q, T.storage_bytes(kv), lay, bt, sl, cu, scale, return_lse=True)
    got, lse = run(gpu_device, kv, "NHD", bt, q, sl, cu, max(qls), scale, want_lse=True)
    T.assert_close_attn(got, want, what=f"mixed batch {hq}/{hkv} d{d}")
    torch.testing.assert_close(lse.cpu(), want_lse, atol=5e-3, rtol=1e-3)


@pytest.mark.parametrize("layout", ["NHD", "HND"])
@pytest.mark.parametrize("q_dtype,out_dtype", [(torch.float32, torch.float32), (torch.float16, torch.float16),
                                               (torch.bfloat16, torch.float32)])
def test_prefill_dtypes_and_layouts(gpu_device, layout, q_dtype, out_dtype):
    ctx, qls = [300, 48], [64, 48]
    kv, lay, bt, q, sl, cu = build(ctx, qls, 8, 2, 128, 16, layout=layout, seed=4, q_dtype=q_dtype)
    want = oracle.paged_attn(q, T.storage_bytes(kv), lay, bt, sl, cu, 0.09)
    got = run(gpu_device, kv, layout, bt, q, sl, cu, 64, 0.09, out_dtype=out_dtype)
    tol = dict(atol=4e-3, rtol=4e-3) if out_dtype == torch.float32 else {}
    T.assert_close_attn(got, want, what="prefill dtypes", **tol)


def test_long_chunk_with_outliers(gpu_device):
    """A 2048-token chunk on top of 1000 context tokens, 1 % outlier channels (x20)."""
    ctx, qls = [3048], [2048]
    kv, lay, bt, q, sl, cu = build(ctx, qls, 8, 2, 128, 16, seed=9, outlier=True)
    want = oracle.paged_attn(q, T.storage_bytes(kv), lay, bt, sl, cu, 0.0884)
    got = run(gpu_device, kv, "NHD", bt, q, sl, cu, 2048, 0.0884, out_dtype=torch.float32)
    T.assert_close_attn(got, want, atol=2e-2, rtol=1e-2, what="long chunk")


def test_causality_first_token_sees_only_itself_and_context(gpu_device):
    """Changing the K/V records of later tokens of a run must not change earlier rows."""
    ctx, qls = [96], [40]
    kv, lay, bt, q, sl, cu = build(ctx, qls, 8, 2, 128, 16, seed=12)
    dev = gpu_device
    a = run(dev, kv, "NHD", bt, q, sl, cu, 40, 0.1, out_dtype=torch.float32)
    # scramble the records of the last 10 tokens of the sequence
    slots = T.slots_for(bt, ctx, 16)[0][-10:]
    g = torch.Generator().manual_seed(1)
    oracle.cache_write(torch.randn((10, 2, 128), generator=g).to(torch.bfloat16) * 3,
                       torch.randn((10, 2, 128), generator=g).to(torch.bfloat16) * 3, T.storage_bytes(kv), lay, slots)
    b = run(dev, kv, "NHD", bt, q, sl, cu, 40, 0.1, out_dtype=torch.float32)
    assert torch.equal(a[:30].cpu(), b[:30].cpu()), "rows before the changed tokens moved"
    assert not torch.equal(a[30:].cpu(), b[30:].cpu())


def test_prefill_golden_mixed_batch(gpu_device):
    import os
    G = torch.load(os.path.join(os.path.dirname(__file__), "golden", "kvq_golden_small.pt"), weights_only=True)
    dev = gpu_device
    hq, hkv, d, bs, nb = (int(G[k]) for k in ("hq", "hkv", "d", "bs", "nb"))
    kv = L.allocate_kv_cache(nb, bs, hkv, d, device=dev, layout="NHD")
    T.storage_bytes(kv).copy_(G["cache_bytes"].to(dev))
    k, v = L.key_value_views(kv)
    ks, vs = L.scale_views(kv)
    out = torch.empty(G["q"].shape, dtype=torch.float32, device=dev)
    lse = torch.empty(G["q"].shape[:2], dtype=torch.float32, device=dev)
    ops.unified_attention(G["q"].to(dev), k, v, out, G["cu"].to(dev), 5, G["ctx"].to(dev), int(G["ctx"].max()),
                          float(G["scale"]), True, block_table=G["block_table"].to(dev), k_scale_cache=ks,
                          v_scale_cache=vs, lse=lse)
    torch.cuda.synchronize()
    T.assert_close_attn(out, G["out"], atol=2e-3, rtol=2e-3, what="golden mixed batch")
    torch.testing.assert_close(lse.cpu(), G["lse"], atol=5e-3, rtol=1e-3)


def test_backend_forward_mixed_batch(gpu_device, monkeypatch):
    """Through the backend mirror: builder metadata -> do_kv_cache_update of the runs' own tokens ->
    forward, on a batch holding a decode row, a pure prefill and a chunk with context."""
    import types

    from vllm_metax_amd.v1.attention.backends.int8_attn import Int8AttentionBackend

    monkeypatch.setenv("VLLM_KV_CACHE_LAYOUT", "NHD")
    dev = gpu_device
    hq, hkv, d, bs, nb = 8, 2, 128, 16, 24
    ctx, qls = [50, 20, 90], [1, 20, 7]
    B = len(ctx)
    g = torch.Generator().manual_seed(31)
    shape = Int8AttentionBackend.get_kv_cache_shape(nb, bs, hkv, d, "int8_per_token_head")
    order = Int8AttentionBackend.get_kv_cache_stride_order()
    phys = torch.zeros(tuple(shape[i] for i in order), dtype=torch.int8, device=dev)
    kv_cache = phys.permute(*[order.index(i) for i in range(4)])
    kv_cpu, views, lay = T.cpu_cache(nb, bs, hkv, d, "NHD")
    views[2].fill_(1.0)
    views[3].fill_(1.0)
    bt = T.make_block_tables(ctx, bs, nb, g)
    impl = Int8AttentionBackend.get_impl_cls()(hq, d, 0.0884, hkv, kv_cache_dtype="int8_per_token_head")
    spec = types.SimpleNamespace(block_size=bs, num_kv_heads=hkv, head_size=d, num_q_heads=hq)
    cfg = types.SimpleNamespace(scheduler_config=types.SimpleNamespace(max_num_seqs=16))
    builder = Int8AttentionBackend.get_builder_cls()(spec, ["layer.0"], cfg, dev)
    layer = types.SimpleNamespace(_k_scale=torch.ones(1, device=dev), _v_scale=torch.ones(1, device=dev))
    slots = T.slots_for(bt, ctx, bs)
    ksrc = [torch.randn((c, hkv, d), generator=g).to(torch.bfloat16) for c in ctx]
    vsrc = [torch.randn((c, hkv, d), generator=g).to(torch.bfloat16) for c in ctx]
    for i, c in enumerate(ctx):                      # earlier steps: everything before the run
        n = c - qls[i]
        if n > 0:
            impl.do_kv_cache_update(layer, ksrc[i][:n].to(dev), vsrc[i][:n].to(dev), kv_cache, slots[i][:n].to(dev))
        oracle.cache_write(ksrc[i], vsrc[i], T.storage_bytes(kv_cpu), lay, slots[i])
    new_k = torch.cat([ksrc[i][ctx[i] - qls[i]:] for i in range(B)])
    new_v = torch.cat([vsrc[i][ctx[i] - qls[i]:] for i in range(B)])
    new_slots = torch.cat([slots[i][ctx[i] - qls[i]:] for i in range(B)])
    n_tok = sum(qls)
    q = torch.randn((n_tok, hq * d), generator=g).to(torch.bfloat16)
    cu = torch.tensor([0] + torch.tensor(qls).cumsum(0).tolist(), dtype=torch.int32)
    common = types.SimpleNamespace(
        num_reqs=B, num_actual_tokens=n_tok, max_query_len=max(qls), max_seq_len=max(ctx),
        query_start_loc=cu.to(dev), seq_lens=torch.tensor(ctx, dtype=torch.int32, device=dev),
        block_table_tensor=bt.to(dev), slot_mapping=new_slots.to(dev), causal=True)
    md = builder.build(0, common)
    impl.do_kv_cache_update(layer, new_k.to(dev), new_v.to(dev), kv_cache, md.slot_mapping)
    out = torch.zeros((n_tok, hq * d), dtype=torch.bfloat16, device=dev)
    impl.forward(layer, q.to(dev), new_k.to(dev), new_v.to(dev), kv_cache, md, out)
    torch.cuda.synchronize()
    assert torch.equal(T.storage_bytes(kv_cache).cpu(), T.storage_bytes(kv_cpu)), "cache bytes differ"
    want = oracle.paged_attn(q.view(n_tok, hq, d), T.storage_bytes(kv_cpu), lay, bt,
                             torch.tensor(ctx, dtype=torch.int32), cu, 0.0884)
    T.assert_close_attn(out.view(n_tok, hq, d), want, what="backend forward, mixed batch")


@pytest.mark.parametrize("step", [0.2, 2.0])
def test_prefill_logits_that_keep_rising(gpu_device, step):
    """Keys whose logits grow along the sequence by ``step`` (log2 units) per 32-token tile: the
    prefill tile's reference maximum may lag the true one by up to 2^8 before it moves.  A 300-token
    chunk on 1500 cached tokens (workgroup-shared tile) plus short runs."""
    hq, hkv, d, bs = 8, 2, 128, 16
    ctx, qls = [1800, 400, 90], [300, 40, 1]
    kv, lay, bt, q, sl, cu = build(ctx, qls, hq, hkv, d, bs, seed=12)
    g = torch.Generator().manual_seed(13)
    u = torch.randn(d, generator=g)
    u = u / u.norm()
    ks = [0.3 * torch.randn((c, hkv, d), generator=g) + (torch.arange(c) / 32.0 * step * 0.6931)[:, None, None] * u for c in ctx]
    vs = [torch.randn((c, hkv, d), generator=g) for c in ctx]
    T.fill_cache_from_sources(kv, lay, bt, ctx, bs, [k.to(torch.bfloat16) for k in ks], [v.to(torch.bfloat16) for v in vs])
    q = (0.3 * q.float() + u).to(torch.bfloat16)          # unit projection on the ramp direction
    want, want_lse = oracle.paged_attn(q, T.storage_bytes(kv), lay, bt, sl, cu, 1.0, return_lse=True)
    got, lse = run(gpu_device, kv, "NHD", bt, q, sl, cu, max(qls), 1.0, want_lse=True)
    T.assert_close_attn(got, want, what=f"prefill, rising logits {step}")
    torch.testing.assert_close(lse.cpu(), want_lse, atol=2e-2, rtol=1e-3)


def test_prefill_huge_value_scales(gpu_device):
    """V rows in the thousands in every other tile: scales above 1, for which the tile moves its
    reference maximum eagerly (p * scale must stay inside fp16)."""
    hq, hkv, d, bs = 8, 2, 128, 16
    ctx, qls = [1200, 64], [500, 64]
    kv, lay, bt, q, sl, cu = build(ctx, qls, hq, hkv, d, bs, seed=14)
    g = torch.Generator().manual_seed(15)
    ks = [torch.randn((c, hkv, d), generator=g) for c in ctx]
    vs = [torch.randn((c, hkv, d), generator=g) * (((torch.arange(c) // 32) % 2 == 1).float() * 1999.0 + 1.0)[:, None, None]
          for c in ctx]
    T.fill_cache_from_sources(kv, lay, bt, ctx, bs, [k.to(torch.bfloat16) for k in ks], [v.to(torch.bfloat16) for v in vs])
    scale = 1 / math.sqrt(d)
    want = oracle.paged_attn(q, T.storage_bytes(kv), lay, bt, sl, cu, scale)
    got = run(gpu_device, kv, "NHD", bt, q, sl, cu, max(qls), scale, out_dtype=torch.float32)
    assert torch.isfinite(got).all()
    T.assert_close_attn(got, want, atol=2e-2 * 2000, rtol=1e-2, what="prefill, huge value scales")


def test_pure_prefill_batch_with_the_no_decode_rows_promise(gpu_device):
    """has_decode_rows=False (KVQ_ATTN_NO_DECODE_ROWS): the decode kernels are skipped; a batch without one-row
    sequences gives the same bits either way, for both prefill tiles."""
    dev = gpu_device
    for hq, hkv, qls in ((32, 8, [300, 64, 2048]), (8, 8, [5, 33, 2])):
        ctx = [q + extra for q, extra in zip(qls, [700, 0, 133])]
        kv_cpu, lay, bt, q, sl, cu = build(ctx, qls, hq, hkv, 128, 16, seed=21)
        kv = T.to_device_cache(kv_cpu, dev, "NHD")
        k, v = L.key_value_views(kv)
        ks, vs = L.scale_views(kv)
        outs = []
        for promise in (True, False):
            out = torch.full(q.shape, float("nan"), dtype=torch.bfloat16, device=dev)
            lse = torch.full(q.shape[:2], float("nan"), dtype=torch.float32, device=dev)
            ops.unified_attention(q.to(dev), k, v, out, cu.to(dev), max(qls), sl.to(dev), int(sl.max()), 0.0884, True,
                                  block_table=bt.to(dev), k_scale_cache=ks, v_scale_cache=vs, lse=lse,
                                  has_decode_rows=promise)
            torch.cuda.synchronize()
            outs.append((out.cpu(), lse.cpu()))
        assert torch.equal(outs[0][0].view(torch.int16), outs[1][0].view(torch.int16)) and torch.equal(outs[0][1], outs[1][1])
        want = oracle.paged_attn(q, T.storage_bytes(kv_cpu), lay, bt, sl, cu, 0.0884)
        T.assert_close_attn(outs[1][0], want, what="pure prefill batch")


@pytest.mark.parametrize("hq,hkv,d,layout", [(32, 8, 128, "HND"), (28, 4, 128, "NHD"), (8, 2, 64, "HND"), (4, 2, 256, "NHD")])
def test_non_causal_rows_see_every_key(gpu_device, hq, hkv, d, layout):
    """causal=False, the cross-attention form of the reference's call (`causal=attn_metadata.causal`,
    vllm_metax/v1/attention/backends/triton_attn.py:698; AttentionType.ENCODER_DECODER goes through the cached
    path, :394-402): every query row of a run attends all `seq_len` keys, whatever its place in the run -- decode
    rows, short runs (the per-wave tile), long runs (the workgroup-shared tile), output and lse against the oracle,
    and every row of a run of copies of one query gets the same bits."""
    ctx = [700, 33, 1500, 64, 257, 5, 900]
    qls = [1, 33, 300, 1, 17, 5, 70]
    kv, lay, bt, q, sl, cu = build(ctx, qls, hq, hkv, d, 16, layout=layout, seed=hq + d + 1)
    # the last run: copies of one query row
    q[int(cu[-2]):] = q[int(cu[-2])].clone()
    scale = 1 / math.sqrt(d)
    want, want_lse = oracle.paged_attn(q, T.storage_bytes(kv), lay, bt, sl, cu, scale, causal=False, return_lse=True)
    causal = oracle.paged_attn(q, T.storage_bytes(kv), lay, bt, sl, cu, scale, causal=True)
    assert not torch.allclose(want, causal, atol=5e-2)
    got, lse = run(gpu_device, kv, layout, bt, q, sl, cu, max(qls), scale, want_lse=True, causal=False)
    T.assert_close_attn(got, want, what=f"non-causal {hq}/{hkv} d{d}")
    torch.testing.assert_close(lse.cpu(), want_lse, atol=5e-3, rtol=1e-3)
    tail = got[int(cu[-2]):].cpu()
    assert torch.equal(tail.view(torch.int16), tail[:1].expand_as(tail).contiguous().view(torch.int16))


@pytest.mark.parametrize("hq,hkv,d,layout,qmax", [(32, 8, 128, "HND", 4), (32, 8, 128, "NHD", 8), (28, 4, 128, "HND", 2),
                                                  (8, 8, 64, "HND", 16), (16, 2, 256, "NHD", 2), (16, 1, 128, "HND", 1)])
def test_short_runs_on_long_contexts_spread_over_a_workgroup(gpu_device, hq, hkv, d, layout, qmax):
    """A speculative-decoding step: every sequence brings a few query tokens (1 + k) on a long context.  With few
    items per launch the short-run kernel spreads an item's tiles over the waves of a workgroup and folds their
    states; contexts shorter than the waves' stride (waves without a tile), one-token sequences next to them (the
    decode kernel's) and a sliding window are in the batch.  Output and lse against the oracle."""
    ctx = [9000, 37, 2500, 300, 64, 5000, 1, 700]
    qls = [min(c, q) for c, q in zip(ctx, [qmax, 2, qmax, 1, 3, qmax, 1, 2])]
    kv, lay, bt, q, sl, cu = build(ctx, qls, hq, hkv, d, 16, layout=layout, seed=hq + qmax)
    scale = 1 / math.sqrt(d)
    for window in (0, 1000):
        want, want_lse = oracle.paged_attn(q, T.storage_bytes(kv), lay, bt, sl, cu, scale, return_lse=True,
                                           sliding_window=window)
        dev = gpu_device
        kvd = T.to_device_cache(kv, dev, layout)
        k, v = L.key_value_views(kvd)
        ks, vs = L.scale_views(kvd)
        out = torch.full(q.shape, float("nan"), dtype=q.dtype, device=dev)
        lse = torch.full(q.shape[:2], float("nan"), dtype=torch.float32, device=dev)
        ops.unified_attention(q.to(dev), k, v, out, cu.to(dev), max(qls), sl.to(dev), int(sl.max()), scale, True,
                              window_size=(window - 1, 0) if window else (-1, -1), block_table=bt.to(dev),
                              k_scale_cache=ks, v_scale_cache=vs, lse=lse)
        torch.cuda.synchronize()
        T.assert_close_attn(out, want, what=f"short runs {hq}/{hkv} d{d} q<={qmax} window {window}")
        torch.testing.assert_close(lse.cpu(), want_lse, atol=5e-3, rtol=1e-3)


def test_many_short_runs_take_one_wave_per_item(gpu_device):
    """Beyond a few thousand items per launch an item stays with one wave (300 sequences x 8 kv heads here): the
    same rows as the oracle's, also when the batch is cut in three launches that spread their items over
    workgroups."""
    hq, hkv, d = 32, 8, 128
    g = torch.Generator().manual_seed(17)
    n = 300
    ctx = torch.randint(20, 400, (n,), generator=g).tolist()
    qls = [min(c, int(x)) for c, x in zip(ctx, torch.randint(1, 5, (n,), generator=g).tolist())]
    kv, lay, bt, q, sl, cu = build(ctx, qls, hq, hkv, d, 16, layout="HND", seed=3)
    scale = 1 / math.sqrt(d)
    want = oracle.paged_attn(q, T.storage_bytes(kv), lay, bt, sl, cu, scale)
    got = run(gpu_device, kv, "HND", bt, q, sl, cu, max(qls), scale)
    T.assert_close_attn(got, want, what="300 short runs, one wave per item")
    parts = []
    for lo_, hi_ in ((0, 100), (100, 200), (200, 300)):
        qq = q[int(cu[lo_]):int(cu[hi_])]
        cc = (cu[lo_:hi_ + 1] - cu[lo_]).contiguous()
        parts.append(run(gpu_device, kv, "HND", bt[lo_:hi_].contiguous(), qq, sl[lo_:hi_].contiguous(), cc, max(qls), scale))
    T.assert_close_attn(torch.cat(parts), want, what="the same runs in three launches")


@pytest.mark.parametrize("hq,hkv,d,layout,code", [(32, 8, 128, "HND", "int8"), (28, 4, 128, "NHD", "int8"),
                                                  (8, 2, 64, "HND", "fp8"), (16, 8, 128, "HND", "int4")])
@pytest.mark.parametrize("window,cap,extras", [(0, 0.0, False), (1500, 30.0, True)])
def test_context_splits_of_long_runs(gpu_device, hq, hkv, d, layout, code, window, cap, extras):
    """kvq_paged_attn_int8_split_prefill: the context of the long query runs in 2..8 ranges, merged afterwards.  A
    small chunk on a long context, a run that starts its sequence, a decode row and a short run (both served as in
    the plain call) in one batch; ranges without a visible tile (window, causal limit); sinks and ALiBi on top.
    Output and lse against the oracle for every split count, and within 1e-2 of the plain call."""
    from vllm_metax_amd.kv_cache_interface import KVQuantMode
    ct = {"int8": oracle.CODE_INT8, "fp8": oracle.CODE_FP8, "int4": oracle.CODE_INT4}[code]
    mode = {"int8": KVQuantMode.INT8_PER_TOKEN_HEAD, "fp8": KVQuantMode.FP8_PER_TOKEN_HEAD,
            "int4": KVQuantMode.INT4_PER_TOKEN_HEAD}[code]
    dev = gpu_device
    bs = 16
    ctx = [6000, 700, 200, 64, 3000]
    qls = [200, 1, 200, 3, 77]
    g = torch.Generator().manual_seed(hq + d + window)
    nb = sum((c + bs - 1) // bs for c in ctx) + 5
    kv_cpu, _, lay = T.cpu_cache(nb, bs, hkv, d, layout, code_type=ct)
    bt = T.make_block_tables(ctx, bs, nb, g)
    ks = [torch.randn((c, hkv, d), generator=g).to(torch.bfloat16) for c in ctx]
    vs_ = [torch.randn((c, hkv, d), generator=g).to(torch.bfloat16) for c in ctx]
    T.fill_cache_from_sources(kv_cpu, lay, bt, ctx, bs, ks, vs_, code_type=ct)
    q = torch.randn((sum(qls), hq, d), generator=g).to(torch.bfloat16)
    sl = torch.tensor(ctx, dtype=torch.int32)
    cu = torch.tensor([0] + torch.tensor(qls).cumsum(0).tolist(), dtype=torch.int32)
    scale = 1 / math.sqrt(d)
    sinks = (torch.randn(hq, generator=g) * 2).float() if extras else None
    slopes = torch.tensor([2.0 ** (-8.0 * (i + 1) / hq) for i in range(hq)], dtype=torch.float32) if extras else None
    want, want_lse = oracle.paged_attn(q, T.storage_bytes(kv_cpu), lay, bt, sl, cu, scale, return_lse=True,
                                       sliding_window=window, soft_cap=cap, code_type=ct, sinks=sinks, alibi_slopes=slopes)
    kv = T.to_device_cache(kv_cpu, dev, layout, code_type=ct)
    k, v = L.key_value_views(kv)
    ksc, vsc = L.scale_views(kv)
    plain = None
    for splits in (1, 2, 3, 5, 8):
        out = torch.full(q.shape, float("nan"), dtype=torch.bfloat16, device=dev)
        lse = torch.full(q.shape[:2], float("nan"), dtype=torch.float32, device=dev)
        ops.unified_attention(q.to(dev), k, v, out, cu.to(dev), max(qls), sl.to(dev), max(ctx), scale, True,
                              window_size=(window - 1, 0) if window else (-1, -1), softcap=cap, block_table=bt.to(dev),
                              k_scale_cache=ksc, v_scale_cache=vsc, kv_quant_mode=mode, lse=lse,
                              sinks=None if sinks is None else sinks.to(dev),
                              alibi_slopes=None if slopes is None else slopes.to(dev), prefill_splits=splits)
        torch.cuda.synchronize()
        T.assert_close_attn(out, want, what=f"{splits} context splits, {code}")
        torch.testing.assert_close(lse.cpu(), want_lse, atol=5e-3, rtol=1e-3)
        if plain is None:
            plain = out.float().cpu()
        else:
            torch.testing.assert_close(out.float().cpu(), plain, atol=1e-2, rtol=1e-2)


def test_context_splits_need_their_workspace(gpu_device):
    dev = gpu_device
    kv = L.allocate_kv_cache(40, 16, 2, 128, device=dev)
    k, v = L.key_value_views(kv)
    ks, vs = L.scale_views(kv)
    q = torch.zeros((64, 8, 128), dtype=torch.bfloat16, device=dev)
    cu = torch.tensor([0, 64], dtype=torch.int32, device=dev)
    sl = torch.tensor([500], dtype=torch.int32, device=dev)
    bt = torch.arange(32, dtype=torch.int32, device=dev).view(1, 32)
    small = torch.empty(ops.paged_attn_workspace_bytes(1, 8, 128), dtype=torch.uint8, device=dev)
    need = ops.split_prefill_workspace_bytes(1, 8, 128, 64, 4)
    assert need >= small.numel() + 64 * 8 * 4 * 130 * 4
    with pytest.raises(RuntimeError, match="workspace"):
        ops.unified_attention(q, k, v, torch.empty_like(q), cu, 64, sl, 500, 0.1, True, block_table=bt,
                              k_scale_cache=ks, v_scale_cache=vs, workspace=small, prefill_splits=4)
    with pytest.raises(RuntimeError):
        ops.unified_attention(q, k, v, torch.empty_like(q), cu, 64, sl, 500, 0.1, True, block_table=bt,
                              k_scale_cache=ks, v_scale_cache=vs, prefill_splits=9)


@pytest.mark.parametrize("hq,hkv,d,qmax,code,q_dtype", [
    (32, 8, 128, 8, "int8", torch.bfloat16),    # two column tiles, full
    (16, 1, 128, 3, "int8", torch.float16),     # one head: eight waves on it, two items per sequence
    (28, 4, 128, 9, "int4", torch.bfloat16),    # 63 columns, columns that do not fill the tiles
    (16, 2, 64, 2, "fp8", torch.bfloat16),      # one column tile, full
    (32, 16, 128, 5, "fp8", torch.float32),     # two workgroups' worth of heads
    (8, 8, 64, 17, "int4", torch.float16)])
@pytest.mark.parametrize("extras", [False, True])
def test_short_run_line(gpu_device, hq, hkv, d, qmax, code, q_dtype, extras):
    """Short runs on a head-major cache, cut along one line of tiles: lengths at the edges of tiles, runs that cover
    their sequence, one-token sequences, an empty one, one long enough to be cut dozens of times; with and without
    window, soft cap, sinks and ALiBi.  Output and lse against the oracle; a workspace without room for the
    states goes through the other kernels, with the same result."""
    from vllm_metax_amd.kv_cache_interface import KVQuantMode
    ct = {"int8": oracle.CODE_INT8, "fp8": oracle.CODE_FP8, "int4": oracle.CODE_INT4}[code]
    mode = {"int8": KVQuantMode.INT8_PER_TOKEN_HEAD, "fp8": KVQuantMode.FP8_PER_TOKEN_HEAD,
            "int4": KVQuantMode.INT4_PER_TOKEN_HEAD}[code]
    dev, bs = gpu_device, 16
    ctx = [31, 32, 33, 5000, 64, 2, 0, 700, 1, qmax, 129]
    qls = [min(c, q) for c, q in zip(ctx, [qmax, qmax, 2, qmax, 1, qmax, 0, 3, 1, qmax, 2])]
    g = torch.Generator().manual_seed(hq + d + qmax)
    nb = sum((c + bs - 1) // bs for c in ctx) + 5
    kv_cpu, _, lay = T.cpu_cache(nb, bs, hkv, d, "HND", code_type=ct)
    T.storage_bytes(kv_cpu).fill_(0xFF)                # NaN scales and codes wherever nothing is written
    bt = T.make_block_tables(ctx, bs, nb, g)
    keys = [torch.randn((c, hkv, d), generator=g).to(torch.bfloat16) for c in ctx]
    vals = [torch.randn((c, hkv, d), generator=g).to(torch.bfloat16) for c in ctx]
    T.fill_cache_from_sources(kv_cpu, lay, bt, ctx, bs, keys, vals, code_type=ct)
    q = torch.randn((sum(qls), hq, d), generator=g).to(q_dtype)
    sl = torch.tensor(ctx, dtype=torch.int32)
    cu = torch.tensor([0] + torch.tensor(qls).cumsum(0).tolist(), dtype=torch.int32)
    scale, window, cap = 1 / math.sqrt(d), (900 if extras else 0), (30.0 if extras else 0.0)
    sinks = (torch.randn(hq, generator=g) * 2).float() if extras else None
    slopes = torch.tensor([2.0 ** (-8.0 * (i + 1) / hq) for i in range(hq)], dtype=torch.float32) if extras else None
    want, want_lse = oracle.paged_attn(q, T.storage_bytes(kv_cpu), lay, bt, sl, cu, scale, return_lse=True,
                                       sliding_window=window, soft_cap=cap, code_type=ct, sinks=sinks, alibi_slopes=slopes)
    kv = T.to_device_cache(kv_cpu, dev, "HND", code_type=ct)
    k, v = L.key_value_views(kv)
    ksc, vsc = L.scale_views(kv)
    tight = torch.empty(ops.paged_attn_workspace_bytes(len(ctx), hq, d), dtype=torch.uint8, device=dev)
    for workspace in (None, tight):
        out = torch.full(q.shape, float("nan"), dtype=q_dtype, device=dev)
        lse = torch.full(q.shape[:2], float("nan"), dtype=torch.float32, device=dev)
        ops.unified_attention(q.to(dev), k, v, out, cu.to(dev), max(qls), sl.to(dev), max(ctx), scale, True,
                              window_size=(window - 1, 0) if window else (-1, -1), softcap=cap, block_table=bt.to(dev),
                              k_scale_cache=ksc, v_scale_cache=vsc, kv_quant_mode=mode, lse=lse, workspace=workspace,
                              sinks=None if sinks is None else sinks.to(dev),
                              alibi_slopes=None if slopes is None else slopes.to(dev))
        torch.cuda.synchronize()
        T.assert_close_attn(out, want, what=f"short runs, {code}, workspace {'tight' if workspace is not None else 'default'}")
        torch.testing.assert_close(lse.cpu(), want_lse, atol=5e-3, rtol=1e-3)


@pytest.mark.parametrize("hq,hkv,d,qmax", [(32, 8, 128, 4), (16, 16, 64, 30), (28, 4, 128, 9)])
def test_short_runs_are_asked_for_and_do_not_depend_on_the_workspace(gpu_device, hq, hkv, d, qmax):
    """The launch for batches of short runs is taken when the caller asks for it, never because its states happen to fit:
    the bits of a call are the same in a workspace of exactly the stated size and in a larger one, asked for or not, and
    a workspace one byte short is refused.  The workspaces hold NaN patterns, which no state that was not written may
    bring into a row."""
    ctx = [700, 33, 2100, 64, 257, 5, 31] * 6
    qls = [min(c, 1 + i % qmax) for i, c in enumerate(ctx)]
    qls[0] = qmax
    kv, lay, bt, q, sl, cu = build(ctx, qls, hq, hkv, d, 16, layout="HND", seed=hq + qmax)
    dev, scale = gpu_device, 1 / math.sqrt(d)
    want = oracle.paged_attn(q, T.storage_bytes(kv), lay, bt, sl, cu, scale)
    kvd = T.to_device_cache(kv, dev, "HND")
    k, v = L.key_value_views(kvd)
    ks, vs = L.scale_views(kvd)
    qd, cu_d, sl_d, bt_d = q.to(dev), cu.to(dev), sl.to(dev), bt.to(dev)

    def call(nbytes, **kw):
        out = torch.full(q.shape, float("nan"), dtype=q.dtype, device=dev)
        ops.unified_attention(qd, k, v, out, cu_d, qmax, sl_d, max(ctx), scale, True, block_table=bt_d, k_scale_cache=ks,
                              v_scale_cache=vs, workspace=torch.full((nbytes,), 0xFF, dtype=torch.uint8, device=dev), **kw)
        torch.cuda.synchronize()
        return out

    for kw in ({}, dict(short_runs=True)):
        exact = ops.paged_attn_workspace_bytes(len(ctx), hq, d)
        if kw:
            exact, smaller = ops.short_runs_workspace_bytes(len(ctx), hq, hkv, d, qmax), exact
            assert smaller <= exact <= ops.short_runs_workspace_bytes(len(ctx) + 100, hq, hkv, d)
        out = call(exact, **kw)
        T.assert_close_attn(out, want, what=f"short runs {hq}/{hkv} d{d} q<={qmax} {kw}")
        same = torch.equal(out, call(256 << 20, **kw))
        assert same, f"the bits depend on the workspace's size {kw}"
        with pytest.raises(RuntimeError, match="workspace"):
            call(exact - 1, **kw)


@pytest.mark.parametrize("hq,hkv,d,bs,layout,code,shift", [
    (32, 8, 128, 16, "HND", "int8", 0),
    (28, 4, 128, 48, "NHD", "int8", 4),      # a block that is no whole number of tiles; records 4 bytes off
    (32, 8, 128, 48, "HND", "fp8", 4),
    (16, 2, 128, 32, "HND", "int4", 0),
    (8, 8, 64, 16, "NHD", "fp8", 0),
    (8, 2, 64, 64, "HND", "int4", 4),        # 72-byte records: one load covers a half tile
    (16, 1, 64, 16, "HND", "int8", 0),
])
def test_shared_tile_at_its_edges(gpu_device, hq, hkv, d, bs, layout, code, shift):
    """The workgroup-shared tile where lengths end at, before and behind a tile, a half tile and a column block, on caches
    whose base is only 4-byte aligned, with NaN scales and codes in every slot that holds no token."""
    from vllm_metax_amd.kv_cache_interface import KVQuantMode
    dev = gpu_device
    ct = {"int8": oracle.CODE_INT8, "fp8": oracle.CODE_FP8, "int4": oracle.CODE_INT4}[code]
    ctx = [64, 65, 96, 31, 700, 129, 16, 450]
    qls = [64, 33, 95, 31, 128, 2, 16, 450]
    g = torch.Generator().manual_seed(hq + d + bs)
    nb = sum((c + bs - 1) // bs for c in ctx) + 5
    kv_cpu, _, lay = T.cpu_cache(nb, bs, hkv, d, layout, code_type=ct)
    T.storage_bytes(kv_cpu).fill_(0xFF)
    bt = T.make_block_tables(ctx, bs, nb, g)
    src = [[torch.randn((c, hkv, d), generator=g).to(torch.bfloat16) for c in ctx] for _ in range(2)]
    T.fill_cache_from_sources(kv_cpu, lay, bt, ctx, bs, *src, code_type=ct)
    q = torch.randn((sum(qls), hq, d), generator=g).to(torch.bfloat16)
    sl = torch.tensor(ctx, dtype=torch.int32)
    cu = torch.tensor([0] + torch.tensor(qls).cumsum(0).tolist(), dtype=torch.int32)
    scale = 1 / math.sqrt(d)
    want, want_lse = oracle.paged_attn(q, T.storage_bytes(kv_cpu), lay, bt, sl, cu, scale, return_lse=True, code_type=ct)
    kv = T.to_device_cache(kv_cpu, dev, layout, code_type=ct)
    flat = torch.full((T.storage_bytes(kv).numel() + 16,), 0xFF, dtype=torch.uint8, device=dev)
    flat[shift:shift + T.storage_bytes(kv).numel()] = T.storage_bytes(kv)
    kv = flat.view(kv.dtype).as_strided(kv.shape, kv.stride(), shift // kv.element_size())
    k, v = L.key_value_views(kv)
    ks, vs = L.scale_views(kv)
    for splits in (1, 3):
        out = torch.full(q.shape, float("nan"), dtype=torch.bfloat16, device=dev)
        lse = torch.full(q.shape[:2], float("nan"), dtype=torch.float32, device=dev)
        ops.unified_attention(q.to(dev), k, v, out, cu.to(dev), max(qls), sl.to(dev), max(ctx), scale, True,
                              block_table=bt.to(dev), k_scale_cache=ks, v_scale_cache=vs, lse=lse, prefill_splits=splits,
                              kv_quant_mode=getattr(KVQuantMode, code.upper() + "_PER_TOKEN_HEAD"))
        torch.cuda.synchronize()
        T.assert_close_attn(out, want, what=f"shared tile {code} d{d}, {splits} ranges")
        torch.testing.assert_close(lse.cpu(), want_lse, atol=5e-3, rtol=1e-3)


@pytest.mark.parametrize("hq,hkv,n", [(32, 8, 5), (32, 8, 6), (32, 8, 2), (28, 4, 10), (28, 4, 11), (24, 12, 3), (9, 3, 1), (32, 16, 1),
                                      (8, 2, 64), (8, 2, 65), (32, 32, 1), (40, 40, 7), (32, 16, 30)])
def test_short_run_shares_by_kv_heads(gpu_device, hq, hkv, n):
    """The batch sizes around which a workgroup of the short-run launch serves fewer kv heads (24 cuts per item, on
    256 compute units), kv head counts that do not divide into them, and a single item; 64 items, the most that the prologue holds, and
    one more: against the oracle."""
    ctx = [(4000 if n < 64 else 400) - (331 if n < 64 else 33) * (i % 7) + i for i in range(n)]
    qls = [2 + i % 3 for i in range(n - 1)] + [4]
    kv, lay, bt, q, sl, cu = build(ctx, qls, hq, hkv, 128, 16, layout="HND", seed=hkv + n)
    scale = 1 / math.sqrt(128)
    want, want_lse = oracle.paged_attn(q, T.storage_bytes(kv), lay, bt, sl, cu, scale, return_lse=True)
    got, lse = run(gpu_device, kv, "HND", bt, q, sl, cu, 4, scale, want_lse=True)
    T.assert_close_attn(got, want, what=f"{n} short runs, {hq}/{hkv}")
    torch.testing.assert_close(lse.cpu(), want_lse, atol=5e-3, rtol=1e-3)


@pytest.mark.parametrize("hq,hkv,d", [(32, 8, 128), (24, 12, 128), (32, 32, 128), (40, 40, 64)])
def test_short_runs_are_one_round_of_workgroups(gpu_device, hq, hkv, d):
    """One run of three tokens on 125 tiles: a workgroup per (share, group of kv heads), one kv head each here, and no more
    of them than compute units.  A share leaves its states in slots 2 w and 2 w + 1 ([slot][kv head][row][dim])."""
    kv, lay, bt, q, sl, cu = build([4000], [3], hq, hkv, d, 16, layout="HND", seed=hkv)
    dev = gpu_device
    kvd = T.to_device_cache(kv, dev, "HND")
    k, v = L.key_value_views(kvd)
    ks, vs = L.scale_views(kvd)
    ws = torch.full((ops.short_runs_workspace_bytes(1, hq, hkv, d, 3, dev),), 0xFF, dtype=torch.uint8, device=dev)
    out = torch.empty_like(q, device=dev)
    ops.unified_attention(q.to(dev), k, v, out, cu.to(dev), 3, sl.to(dev), 4000, 0.1, True, block_table=bt.to(dev),
                          k_scale_cache=ks, v_scale_cache=vs, workspace=ws, short_runs=True)
    torch.cuda.synchronize()
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    states = ws[:2 * cus * hq * 3 * d * 4].view(cus, -1)
    shares = int((states != 0xFF).any(1).sum())
    assert 1 < shares and shares * hkv <= max(cus, hkv), f"{shares} shares x {hkv} kv heads on {cus} compute units"


@pytest.mark.parametrize("hq,hkv,splits", [(32, 8, 6), (32, 8, 3), (16, 4, 2), (16, 4, 3), (12, 3, 8), (16, 2, 4), (9, 1, 8)])
def test_context_ranges_on_their_xcd(gpu_device, hq, hkv, splits):
    """(kv head, range) pairs that can and that cannot be dealt out to eight XCDs evenly, two runs of different
    numbers of query blocks: every row comes from every range once."""
    ctx, qls = [5000, 4300], [150, 40]
    kv, lay, bt, q, sl, cu = build(ctx, qls, hq, hkv, 128, 16, layout="HND", seed=hkv + splits)
    scale = 1 / math.sqrt(128)
    want = oracle.paged_attn(q, T.storage_bytes(kv), lay, bt, sl, cu, scale)
    dev = gpu_device
    kvd = T.to_device_cache(kv, dev, "HND")
    k, v = L.key_value_views(kvd)
    ks, vs = L.scale_views(kvd)
    out = torch.full(q.shape, float("nan"), dtype=q.dtype, device=dev)
    ops.unified_attention(q.to(dev), k, v, out, cu.to(dev), max(qls), sl.to(dev), max(ctx), scale, True, block_table=bt.to(dev),
                          k_scale_cache=ks, v_scale_cache=vs, prefill_splits=splits)
    torch.cuda.synchronize()
    T.assert_close_attn(out, want, what=f"{splits} ranges, {hq}/{hkv}")


@pytest.mark.parametrize("d,window,cap", [(128, 0, 0.0), (64, 0, 0.0), (128, 200, 30.0), (64, 200, 30.0), (256, 0, 0.0)])
@pytest.mark.parametrize("code", ["int8", "fp8", "int4"])
def test_negative_softmax_scale(gpu_device, code, d, window, cap):
    """A softmax scale below zero turns the weights round, in every kernel that one call can take: decode rows, short
    runs, long runs whole and in context ranges."""
    from vllm_metax_amd.kv_cache_interface import KVQuantMode
    hq, hkv, bs, dev = 16, 4, 16, gpu_device
    ct = {"int8": oracle.CODE_INT8, "fp8": oracle.CODE_FP8, "int4": oracle.CODE_INT4}[code]
    ctx, qls = [900, 300, 450, 65], [1, 5, 300, 65]
    g = torch.Generator().manual_seed(d)
    nb = sum((c + bs - 1) // bs for c in ctx) + 5
    kv_cpu, _, lay = T.cpu_cache(nb, bs, hkv, d, "HND", code_type=ct)
    T.storage_bytes(kv_cpu).fill_(0xFF)
    bt = T.make_block_tables(ctx, bs, nb, g)
    src = [[torch.randn((c, hkv, d), generator=g).to(torch.bfloat16) for c in ctx] for _ in range(2)]
    T.fill_cache_from_sources(kv_cpu, lay, bt, ctx, bs, *src, code_type=ct)
    q = torch.randn((sum(qls), hq, d), generator=g).to(torch.bfloat16)
    sl = torch.tensor(ctx, dtype=torch.int32)
    cu = torch.tensor([0] + torch.tensor(qls).cumsum(0).tolist(), dtype=torch.int32)
    scale = -1 / math.sqrt(d)
    want, want_lse = oracle.paged_attn(q, T.storage_bytes(kv_cpu), lay, bt, sl, cu, scale, return_lse=True, code_type=ct,
                                       sliding_window=window, soft_cap=cap)
    kv = T.to_device_cache(kv_cpu, dev, "HND", code_type=ct)
    k, v = L.key_value_views(kv)
    ks, vs = L.scale_views(kv)
    for splits in (1, 3):
        out = torch.full(q.shape, float("nan"), dtype=torch.bfloat16, device=dev)
        lse = torch.full(q.shape[:2], float("nan"), dtype=torch.float32, device=dev)
        ops.unified_attention(q.to(dev), k, v, out, cu.to(dev), max(qls), sl.to(dev), max(ctx), scale, True,
                              window_size=(window - 1, 0) if window else (-1, -1), softcap=cap, block_table=bt.to(dev),
                              k_scale_cache=ks, v_scale_cache=vs, lse=lse, prefill_splits=splits,
                              kv_quant_mode=getattr(KVQuantMode, code.upper() + "_PER_TOKEN_HEAD"))
        torch.cuda.synchronize()
        T.assert_close_attn(out, want, what=f"negative scale {code} d{d}, {splits} ranges")
        torch.testing.assert_close(lse.cpu(), want_lse, atol=5e-3, rtol=1e-3)


@pytest.mark.parametrize("d,window", [(128, 0), (64, 0), (128, 100), (64, 100)])
@pytest.mark.parametrize("code", ["int8", "fp8", "int4"])
def test_output_types_of_the_shared_tile(gpu_device, code, d, window):
    """Long runs write bf16, fp16 or fp32 rows: the 16-bit ones are the fp32 row rounded to nearest even."""
    from vllm_metax_amd.kv_cache_interface import KVQuantMode
    hq, hkv, bs, dev = 14, 2, 16, gpu_device
    ct = {"int8": oracle.CODE_INT8, "fp8": oracle.CODE_FP8, "int4": oracle.CODE_INT4}[code]
    ctx, qls = [70, 333, 96], [70, 100, 33]
    g = torch.Generator().manual_seed(d)
    nb = sum((c + bs - 1) // bs for c in ctx) + 5
    kv_cpu, _, lay = T.cpu_cache(nb, bs, hkv, d, "HND", code_type=ct)
    bt = T.make_block_tables(ctx, bs, nb, g)
    src = [[torch.randn((c, hkv, d), generator=g).to(torch.bfloat16) for c in ctx] for _ in range(2)]
    T.fill_cache_from_sources(kv_cpu, lay, bt, ctx, bs, *src, code_type=ct)
    q = torch.randn((sum(qls), hq, d), generator=g).to(torch.bfloat16)
    kv = T.to_device_cache(kv_cpu, dev, "HND", code_type=ct)
    k, v = L.key_value_views(kv)
    ks, vs = L.scale_views(kv)
    cu = torch.tensor([0] + torch.tensor(qls).cumsum(0).tolist(), dtype=torch.int32, device=dev)
    outs = {}
    for dtype in (torch.float32, torch.bfloat16, torch.float16):
        outs[dtype] = torch.zeros(q.shape, dtype=dtype, device=dev)
        ops.unified_attention(q.to(dev), k, v, outs[dtype], cu, max(qls), torch.tensor(ctx, dtype=torch.int32, device=dev),
                              max(ctx), d ** -0.5, True, window_size=(window - 1, 0) if window else (-1, -1),
                              block_table=bt.to(dev), k_scale_cache=ks, v_scale_cache=vs,
                              kv_quant_mode=getattr(KVQuantMode, code.upper() + "_PER_TOKEN_HEAD"))
    torch.cuda.synchronize()
    for dtype, out in outs.items():
        assert torch.equal(out, outs[torch.float32].to(dtype)), dtype


@pytest.mark.parametrize("hq,hkv,d", [(28, 4, 128), (8, 8, 64), (32, 8, 128)])
@pytest.mark.parametrize("window", [0, 1, 20, 40, 100])
def test_odd_ends_of_the_shared_tile(gpu_device, hq, hkv, d, window):
    """Runs that end in an odd tile, whole and in ranges, with windows that put some waves of a workgroup into the steps at
    its lower edge to the very end and others not: the same steps for all of them."""
    ctx, qls = [33, 95, 161, 224, 290], [33, 95, 150, 130, 65]
    kv, lay, bt, q, sl, cu = build(ctx, qls, hq, hkv, d, 16, layout="HND", seed=hq + window)
    scale = 1 / math.sqrt(d)
    want = oracle.paged_attn(q, T.storage_bytes(kv), lay, bt, sl, cu, scale, sliding_window=window)
    dev = gpu_device
    kvd = T.to_device_cache(kv, dev, "HND")
    k, v = L.key_value_views(kvd)
    ks, vs = L.scale_views(kvd)
    for splits in (1, 2):
        out = torch.full(q.shape, float("nan"), dtype=q.dtype, device=dev)
        ops.unified_attention(q.to(dev), k, v, out, cu.to(dev), max(qls), sl.to(dev), max(ctx), scale, True,
                              window_size=(window - 1, 0) if window else (-1, -1), block_table=bt.to(dev), k_scale_cache=ks,
                              v_scale_cache=vs, prefill_splits=splits)
        torch.cuda.synchronize()
        T.assert_close_attn(out, want, what=f"odd ends, window {window}, {splits} ranges")


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 64, 65, 100, 257, 300])
@pytest.mark.parametrize("hq,hkv,d,splits", [(32, 8, 128, 1), (32, 8, 128, 3), (8, 2, 256, 1), (8, 8, 64, 2)])
def test_runs_of_a_batch_by_its_number_of_sequences(gpu_device, n, hq, hkv, d, splits):
    """Up to 16 sequences every workgroup finds its query run itself, beyond the decode launch lists them: runs between decode
    rows and sequences without tokens, several of one length.  The oracle decides, within the bounds of the other tests; an empty
    sequence's one row is zeros with lse -inf, its several rows are left alone."""
    lens = [(90, 90, 40, 200)[i % 4] + (i % 3) * 16 for i in range(n)]
    qls = [(70, 1, 33, 90)[i % 4] if n > 2 else 70 for i in range(n)]
    empty = [n - 3] if n > 2 else []
    if n > 256:
        qls[256] = 1
        empty.append(256)
    kv, lay, bt, q, sl, cu = build(lens, qls, hq, hkv, d, 16, seed=n + d)
    sl[empty] = 0
    scale = 1 / math.sqrt(d)
    want, want_lse = oracle.paged_attn(q, T.storage_bytes(kv), lay, bt, sl, cu, scale, return_lse=True)
    kvd = T.to_device_cache(kv, gpu_device, "NHD")
    k, v = L.key_value_views(kvd)
    ks, vs = L.scale_views(kvd)
    out = torch.full(q.shape, float("nan"), dtype=q.dtype, device=gpu_device)
    lse = torch.full(q.shape[:2], float("nan"), dtype=torch.float32, device=gpu_device)
    ops.unified_attention(q.to(gpu_device), k, v, out, cu.to(gpu_device), max(qls), sl.to(gpu_device), int(sl.max()), scale,
                          True, block_table=bt.to(gpu_device), k_scale_cache=ks, v_scale_cache=vs, prefill_splits=splits, lse=lse)
    torch.cuda.synchronize()
    out, lse = out.cpu(), lse.cpu()
    written = torch.ones(q.shape[0], dtype=torch.bool)
    for i in empty:
        at = slice(int(cu[i]), int(cu[i + 1]))
        if qls[i] == 1:
            assert (out[at] == 0).all() and (lse[at] == -math.inf).all(), f"sequence {i} of {n}: empty, one row"
        else:
            assert out[at].isnan().all() and lse[at].isnan().all(), f"sequence {i} of {n}: empty, {qls[i]} rows"
        written[at] = False
    T.assert_close_attn(out[written], want[written], what=f"{n} sequences d{d} splits {splits}")
    torch.testing.assert_close(lse[written], want_lse[written], atol=5e-3, rtol=1e-3)


@pytest.mark.parametrize("hq,hkv,d", [(8, 2, 64), (32, 8, 128), (4, 4, 256)])
@pytest.mark.parametrize("run", [9, 70])
def test_empty_decode_rows_of_a_mixed_batch_of_any_size(gpu_device, hq, hkv, d, run):
    """One-row sequences of length 0 anywhere in a batch of more sequences than the chip has compute units, next to query runs:
    zeros, lse -inf.  What the rows held before is NaN, so a row that no workgroup takes shows."""
    n = 2 * torch.cuda.get_device_properties(gpu_device).multi_processor_count + 20
    qls = [run if i % 50 == 7 else 1 for i in range(n)]
    lens = [max(qls[i], 1 + 3 * (i % 11)) for i in range(n)]
    kv, lay, bt, q, sl, cu = build(lens, qls, hq, hkv, d, 16, seed=run + d)
    for i in range(n):
        if qls[i] == 1 and (i % 3 == 0 or i > n // 2 - 12):
            sl[i] = 0
    scale = 1 / math.sqrt(d)
    want, want_lse = oracle.paged_attn(q, T.storage_bytes(kv), lay, bt, sl, cu, scale, return_lse=True)
    kvd = T.to_device_cache(kv, gpu_device, "NHD")
    k, v = L.key_value_views(kvd)
    ks, vs = L.scale_views(kvd)
    out = torch.full(q.shape, float("nan"), dtype=torch.float32, device=gpu_device)
    lse = torch.full(q.shape[:2], float("nan"), dtype=torch.float32, device=gpu_device)
    ops.unified_attention(q.to(gpu_device), k, v, out, cu.to(gpu_device), max(qls), sl.to(gpu_device), int(sl.max()), scale,
                          True, block_table=bt.to(gpu_device), k_scale_cache=ks, v_scale_cache=vs, lse=lse)
    torch.cuda.synchronize()
    left = [i for i in range(n) if out[int(cu[i])].isnan().any() or lse[int(cu[i])].isnan().any()]
    assert not left, f"rows that nobody wrote: sequences {left} of {n}"
    T.assert_close_attn(out, want, what=f"empty decode rows d{d}")
    torch.testing.assert_close(lse.cpu(), want_lse, atol=5e-3, rtol=1e-3)
