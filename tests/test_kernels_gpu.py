"""Numerics tests for the hand-written CDNA4 HIP kernels.

Every kernel is compared against the plain-PyTorch fp32 reference in
vllm_amd/ops/_torch_ref.py (the pattern of the reference repo's
tests/kernels/). Runs only on an MI355X (-m gpu).
"""

import pytest
import torch

from vllm_amd.ops import _torch_ref as ref

pytestmark = pytest.mark.gpu


def _hip():
    from vllm_amd.ops import hip_ops

    return hip_ops


def assert_close(hip_out, ref_out, atol=2e-2, rtol=2e-2, msg=""):
    hip_f = hip_out.float()
    ref_f = ref_out.float()
    torch.testing.assert_close(hip_f, ref_f, atol=atol, rtol=rtol, msg=msg)


@pytest.fixture(autouse=True)
def _seed():
    torch.manual_seed(0)


@pytest.mark.parametrize("shape", [(1, 128), (17, 4096), (256, 8192)])
def test_rms_norm(shape):
    hip = _hip()
    x = torch.randn(shape, dtype=torch.bfloat16, device="cuda")
    w = torch.randn(shape[-1], dtype=torch.bfloat16, device="cuda")
    out = hip.rms_norm(x, w, 1e-5)
    expect = ref.rms_norm(x.float(), w.float(), 1e-5)
    assert_close(out, expect)


@pytest.mark.parametrize("shape", [(3, 512), (129, 4096)])
def test_fused_add_rms_norm(shape):
    hip = _hip()
    x = torch.randn(shape, dtype=torch.bfloat16, device="cuda")
    res = torch.randn(shape, dtype=torch.bfloat16, device="cuda")
    w = torch.randn(shape[-1], dtype=torch.bfloat16, device="cuda")
    ex_out, ex_res = ref.fused_add_rms_norm(
        x.clone().float(), res.clone().float(), w.float(), 1e-5
    )
    out, new_res = hip.fused_add_rms_norm(x, res, w, 1e-5)
    assert_close(new_res, ex_res)
    assert_close(out, ex_out)


@pytest.mark.parametrize("act", ["silu", "gelu"])
@pytest.mark.parametrize("shape", [(5, 256), (300, 28672)])
def test_act_and_mul(act, shape):
    hip = _hip()
    x = torch.randn(shape, dtype=torch.bfloat16, device="cuda")
    fn = hip.silu_and_mul if act == "silu" else hip.gelu_and_mul
    rfn = ref.silu_and_mul if act == "silu" else ref.gelu_and_mul
    assert_close(fn(x), rfn(x.float()))


@pytest.mark.parametrize("rotary_dim", [128, 64])
def test_rope_neox(rotary_dim):
    hip = _hip()
    T, Hq, Hkv, D = 33, 8, 2, 128
    max_pos = 2048
    inv = 1.0 / (10000.0 ** (
        torch.arange(0, rotary_dim, 2).float() / rotary_dim))
    t = torch.arange(max_pos).float()
    freqs = torch.outer(t, inv)
    cache = torch.cat([freqs.cos(), freqs.sin()], dim=-1).cuda()
    pos = torch.randint(0, max_pos, (T,), device="cuda")
    q = torch.randn(T, Hq, D, dtype=torch.bfloat16, device="cuda")
    k = torch.randn(T, Hkv, D, dtype=torch.bfloat16, device="cuda")
    eq, ek = ref.apply_rope(pos, q.clone().float(), k.clone().float(),
                            cache, rotary_dim)
    hq, hk = hip.apply_rope(pos, q, k, cache, rotary_dim)
    assert_close(hq, eq)
    assert_close(hk, ek)


def test_reshape_and_cache():
    hip = _hip()
    T, Hkv, D, BS, NB = 200, 8, 128, 64, 32
    k = torch.randn(T, Hkv, D, dtype=torch.bfloat16, device="cuda")
    v = torch.randn(T, Hkv, D, dtype=torch.bfloat16, device="cuda")
    cache = torch.zeros(2, NB, Hkv, BS, D, dtype=torch.bfloat16,
                        device="cuda")
    ref_cache = cache.clone()
    slots = torch.randperm(NB * BS, device="cuda")[:T]
    hip.reshape_and_cache(k, v, cache, slots)
    ref.reshape_and_cache(k, v, ref_cache, slots)
    torch.testing.assert_close(cache, ref_cache)


def _make_paged(num_reqs, q_lens, ctx_lens, Hq, Hkv, D=128, BS=64):
    """Build q + populated paged cache + metadata for attention tests."""
    total_q = sum(q_lens)
    max_blocks = max((c + BS - 1) // BS for c in ctx_lens)
    num_blocks = num_reqs * max_blocks + 1
    q = torch.randn(total_q, Hq, D, dtype=torch.bfloat16, device="cuda")
    cache = torch.randn(2, num_blocks, Hkv, BS, D, dtype=torch.bfloat16,
                        device="cuda")
    block_table = torch.zeros(num_reqs, max_blocks, dtype=torch.int32,
                              device="cuda")
    nxt = 1
    for i, c in enumerate(ctx_lens):
        nb = (c + BS - 1) // BS
        block_table[i, :nb] = torch.arange(nxt, nxt + nb)
        nxt += nb
    qsl = torch.zeros(num_reqs + 1, dtype=torch.int32, device="cuda")
    qsl[1:] = torch.cumsum(
        torch.tensor(q_lens, device="cuda", dtype=torch.int32), 0)
    seq_lens = torch.tensor(ctx_lens, dtype=torch.int32, device="cuda")
    return q, cache, block_table, qsl, seq_lens


@pytest.mark.parametrize("group", [1, 4, 8])
@pytest.mark.parametrize("ctx", [1, 63, 64, 200, 511, 513, 2000])
def test_decode_attention(group, ctx):
    hip = _hip()
    Hkv = 2
    Hq = Hkv * group
    n = 4
    q, cache, bt, qsl, sl = _make_paged(n, [1] * n, [ctx] * n, Hq, Hkv)
    scale = 1.0 / 128**0.5
    out = hip.attention_unified(q, cache, bt, qsl, sl, scale,
                                num_decodes=n, max_seq_len=ctx,
                                max_query_len=1)
    expect = ref.attention_unified(q, cache, bt, qsl, sl, scale,
                                   num_decodes=n)
    assert_close(out, expect, msg=f"group={group} ctx={ctx}")


@pytest.mark.parametrize("hd,group,dtype,cache_dtype,window", [
    (128, 7, torch.bfloat16, torch.bfloat16, 0),
    (128, 4, torch.bfloat16, torch.bfloat16, 150),
    (64, 3, torch.bfloat16, torch.float8_e4m3fn, 0),
    (256, 5, torch.bfloat16, torch.float8_e4m3fn, 33),
    (128, 8, torch.float16, torch.float16, 0),
    (64, 1, torch.float16, torch.float8_e4m3fn, 1),
])
@pytest.mark.parametrize("n", [6, 300])  # split and unsplit keys
def test_decode_attention_edges(hd, group, dtype, cache_dtype, window, n):
    """Ragged rows at the edges of a wave's 32 keys, a workgroup's 128
    and a cache block; rows of the last block that no token has written
    hold NaN. Tolerance: the output's own rounding, 2^-8 (bf16) or
    2^-11 (fp16) of values up to 4, once more for the order of sums."""
    hip = _hip()
    Hkv = 2
    lens = [1, 31, 33, 64, 129, 640]
    ctx = [lens[i % 6] for i in range(n)]
    q, cache, bt, qsl, sl = _make_paged(n, [1] * n, ctx, Hkv * group, Hkv,
                                        D=hd)
    q = q.to(dtype)
    cache = cache.to(cache_dtype)
    raw = cache if cache_dtype != torch.float8_e4m3fn \
        else cache.view(torch.uint8)
    nan = float("nan") if raw is cache else 0x7F
    for i in range(6):
        if ctx[i] % 64:
            raw[:, bt[i, ctx[i] // 64], :, ctx[i] % 64:] = nan
    out = hip.attention_unified(q, cache, bt, qsl, sl, hd**-0.5,
                                num_decodes=n, max_seq_len=max(ctx),
                                max_query_len=1, sliding_window=window)
    rows = list(range(6))
    expect = ref.attention_unified(
        q[rows].float(), cache.float(), bt[rows], qsl[:7], sl[rows],
        hd**-0.5, num_decodes=6, sliding_window=window)
    atol = 2 * 4 * (2**-8 if dtype == torch.bfloat16 else 2**-11)
    assert_close(out[rows], expect, atol=atol, rtol=atol / 4)


def _check_decode_rows(n, lens, Hkv, group, hd, dtype, cache_dtype, window,
                       bound=0):
    """Rows of the given lengths in turn against fp32, unwritten rows of
    their last block NaN. Tolerance: the output's own rounding, 2^-8
    (bf16) or 2^-11 (fp16) of values up to 4, once more for the order of
    sums."""
    hip = _hip()
    ctx = [lens[i % len(lens)] for i in range(n)]
    q, cache, bt, qsl, sl = _make_paged(n, [1] * n, ctx, Hkv * group, Hkv,
                                        D=hd)
    q, cache = q.to(dtype), cache.to(cache_dtype)
    raw = cache if cache_dtype != torch.float8_e4m3fn \
        else cache.view(torch.uint8)
    rows = sorted({*range(len(lens)), n - 1})
    for i in rows:
        if ctx[i] % 64:
            raw[:, bt[i, ctx[i] // 64], :, ctx[i] % 64:] = \
                float("nan") if raw is cache else 0x7F
    out = hip.attention_unified(q, cache, bt, qsl, sl, hd**-0.5,
                                num_decodes=n,
                                max_seq_len=bound or max(ctx),
                                max_query_len=1, sliding_window=window)
    expect = ref.attention_unified(
        q[rows].float(), cache.float(), bt[rows], qsl[:len(rows) + 1],
        sl[rows], hd**-0.5, num_decodes=len(rows), sliding_window=window)
    atol = 2 * 4 * (2**-8 if dtype == torch.bfloat16 else 2**-11)
    assert_close(out[rows], expect, atol=atol, rtol=atol / 4)


@pytest.mark.parametrize("dtype,group,window", [
    (torch.bfloat16, 3, 0), (torch.float16, 8, 0), (torch.bfloat16, 1, 33)])
@pytest.mark.parametrize("n", [7, 300])  # split and unsplit keys
def test_decode_attention_16_key_steps(dtype, group, window, n):
    """Heads of 256 take 16 keys a step: rows around 16 keys, a
    workgroup's 64 and a cache block."""
    _check_decode_rows(n, [1, 15, 17, 63, 65, 128, 641], 2, group, 256,
                       dtype, dtype, window)


@pytest.mark.parametrize("hd,group,dtype,cache_dtype,window,bound", [
    (128, 4, torch.bfloat16, torch.bfloat16, 0, 0),
    (128, 7, torch.float16, torch.float8_e4m3fn, 40, 0),
    (64, 8, torch.bfloat16, torch.bfloat16, 0, 512),
    (64, 1, torch.float16, torch.float16, 33, 0),
    (256, 2, torch.bfloat16, torch.bfloat16, 0, 0),
    (256, 3, torch.bfloat16, torch.float8_e4m3fn, 17, 0),
    (128, 2, torch.bfloat16, torch.bfloat16, 0, 512),
])
def test_decode_attention_wave_rows(hd, group, dtype, cache_dtype, window,
                                    bound):
    """Many short rows, a wave each: rows around the steps of 16 and 32
    keys, a number of rows that is no multiple of a workgroup's four, a
    bound far above the rows as a captured step has."""
    lens = [1, 15, 16, 17, 31, 33, 64, 127, 128, 97]
    if bound:
        lens += [129, 480, 512]
    _check_decode_rows(2063 if bound else 803, lens, 2, group, hd, dtype,
                       cache_dtype, window, bound)


@pytest.mark.parametrize("hd", [64, 128, 256])
def test_decode_wave_rows_without_keys(hd):
    hip = _hip()
    n = 801
    q, cache, bt, qsl, sl = _make_paged(n, [1] * n, [40] * n, 8, 2, D=hd)
    sl[1::2] = 0
    junk = torch.full_like(q, float("nan"))
    del junk
    out = hip.attention_unified(q, cache, bt, qsl, sl, 0.1, num_decodes=n,
                                max_seq_len=40, max_query_len=1)
    assert (out[1::2] == 0).all() and out[::2].isfinite().all()


@pytest.mark.parametrize("n,longest", [(300, 700), (3, 700), (300, 90)])
def test_decode_rows_without_keys(n, longest):
    """A row of length 0 (a captured step's padding) gives exact zeros,
    whether its keys would be split or not, and leaves the others alone.
    The memory that results are taken from holds NaN."""
    hip = _hip()
    q, cache, bt, qsl, sl = _make_paged(n, [1] * n, [longest] * n, 8, 2)
    sl[1::2] = 0
    junk = torch.full_like(q, float("nan"))
    del junk
    out = hip.attention_unified(q, cache, bt, qsl, sl, 0.1, num_decodes=n,
                                max_seq_len=longest, max_query_len=1)
    assert (out[1::2] == 0).all() and out[::2].isfinite().all()
    lat = torch.randn(n * 2, 64, 576, device="cuda", dtype=torch.bfloat16)
    bt = torch.arange(n * 2, device="cuda", dtype=torch.int32).view(n, 2)
    sl.clamp_(max=128)
    for heads in (20, 130):
        qn = torch.randn(n, heads, 512, device="cuda", dtype=torch.bfloat16)
        junk = torch.full_like(qn, float("nan"))
        del junk
        out = hip.mla_decode(qn, qn[..., :64].contiguous(), lat, bt, sl,
                             0.07, 128)
        assert (out[1::2] == 0).all() and out[::2].isfinite().all()


@pytest.mark.parametrize("group", [4])
@pytest.mark.parametrize(
    "q_lens,ctx_lens",
    [
        ([16, 33], [16, 33]),            # pure prefill from scratch
        ([64, 128], [64, 128]),
        ([17, 70], [100, 300]),           # chunked-prefill continuation
        ([1, 1, 5, 200], [40, 513, 60, 200]),  # mixed decode+prefill
    ],
)
def test_prefill_attention(group, q_lens, ctx_lens):
    hip = _hip()
    Hkv = 2
    Hq = Hkv * group
    n = len(q_lens)
    num_decodes = sum(1 for x in q_lens if x == 1)
    # decodes-first ordering as the model runner produces
    order = sorted(range(n), key=lambda i: q_lens[i] != 1)
    q_lens = [q_lens[i] for i in order]
    ctx_lens = [ctx_lens[i] for i in order]
    q, cache, bt, qsl, sl = _make_paged(n, q_lens, ctx_lens, Hq, Hkv)
    scale = 1.0 / 128**0.5
    out = hip.attention_unified(
        q, cache, bt, qsl, sl, scale, num_decodes=num_decodes,
        max_seq_len=max(ctx_lens), max_query_len=max(q_lens))
    expect = ref.attention_unified(q, cache, bt, qsl, sl, scale,
                                   num_decodes=num_decodes)
    assert_close(out, expect)


@pytest.mark.parametrize("hd,group,dtype,cache_dtype,window,scale", [
    (128, 7, torch.bfloat16, torch.bfloat16, 0, 0.09),
    (128, 4, torch.bfloat16, torch.bfloat16, 5, 0.5),
    (128, 4, torch.float16, torch.float16, 0, 0.5),
    (64, 3, torch.bfloat16, torch.float8_e4m3fn, 0, -0.125),
    (64, 1, torch.float16, torch.float8_e4m3fn, 70, 0.125),
    (256, 5, torch.bfloat16, torch.bfloat16, 200, 0.06),
    (256, 2, torch.bfloat16, torch.float8_e4m3fn, 0, 0.06),
])
def test_prefill_attention_edges(hd, group, dtype, cache_dtype, window,
                                 scale):
    """Portions that end on, before and after the edges of a row tile
    (128 rows = tokens x heads) and of a key tile, after contexts of the
    same kind; an empty portion; unwritten rows of the last block hold
    NaN; scores large enough for the running maximum to move. Tolerance:
    weights and outputs rounded to 16 bits (2^-8 bf16, 2^-11 fp16), of
    values up to 4."""
    hip = _hip()
    Hkv = 2
    q_lens = [2, 33, 64, 0, 65, 129]
    ctx = [2, 64, 64 + 63, 9, 65 + 300, 129]
    n = len(ctx)
    q, cache, bt, qsl, sl = _make_paged(n, q_lens, ctx, Hkv * group, Hkv,
                                        D=hd)
    q = q.to(dtype)
    cache = cache.to(cache_dtype)
    raw = cache if cache_dtype != torch.float8_e4m3fn \
        else cache.view(torch.uint8)
    nan = float("nan") if raw is cache else 0x7F
    for i in range(n):
        if ctx[i] % 64:
            raw[:, bt[i, ctx[i] // 64], :, ctx[i] % 64:] = nan
    out = hip.attention_unified(q, cache, bt, qsl, sl, scale,
                                num_decodes=0, max_seq_len=max(ctx),
                                max_query_len=max(q_lens),
                                sliding_window=window)
    expect = ref.attention_unified(q.float(), cache.float(), bt, qsl, sl,
                                   scale, sliding_window=window)
    atol = 3 * 4 * (2**-8 if dtype == torch.bfloat16 else 2**-11)
    assert_close(out, expect, atol=atol, rtol=atol / 4)


@pytest.mark.parametrize("hd,cache_dtype", [
    (64, torch.bfloat16), (128, torch.bfloat16), (256, torch.bfloat16),
    (64, torch.float8_e4m3fn), (128, torch.float8_e4m3fn)])
@pytest.mark.parametrize("window", [0, 70])
def test_prefill_attention_tile_counts(hd, cache_dtype, window):
    """One to seven key tiles a workgroup, odd and even, from an odd and an
    even tile on. Tolerance as above."""
    hip = _hip()
    ctx = [64 * i - 3 for i in range(1, 8)] + [64 * i + 2 for i in range(1, 8)]
    q_lens = [1 + i % 3 for i in range(len(ctx))]
    n = len(ctx)
    q, cache, bt, qsl, sl = _make_paged(n, q_lens, ctx, 8, 2, D=hd)
    cache = cache.to(cache_dtype)
    out = hip.attention_unified(q, cache, bt, qsl, sl, hd**-0.5,
                                num_decodes=0, max_seq_len=max(ctx),
                                max_query_len=max(q_lens),
                                sliding_window=window)
    expect = ref.attention_unified(q.float(), cache.float(), bt, qsl, sl,
                                   hd**-0.5, sliding_window=window)
    atol = 3 * 4 * 2**-8
    assert_close(out, expect, atol=atol, rtol=atol / 4)


def test_model_forward_matches_cpu_reference():
    """Tiny Llama forward on GPU (bf16, HIP kernels) vs CPU fp32 torch
    reference: logits must be directionally identical (cosine > 0.99)."""
    from vllm_amd.config import ModelConfig
    from vllm_amd.models.registry import load_model
    from vllm_amd.worker.forward_context import (
        AttentionMetadata, ForwardContext, set_forward_context)

    def run(device, dtype):
        torch.manual_seed(0)
        cfg = ModelConfig(model="tiny-llama-128", dtype=dtype,
                          load_format="dummy")
        model = load_model(cfg, torch.device(device))
        T = 9
        ids = torch.arange(1, T + 1, device=device)
        pos = torch.arange(T, device=device)
        spec = cfg.spec
        caches = [
            torch.zeros(2, 4, spec.num_kv_heads, 64, spec.head_dim,
                        dtype=cfg.torch_dtype, device=device)
            for _ in range(spec.num_layers)
        ]
        meta = AttentionMetadata(
            query_start_loc=torch.tensor([0, T], dtype=torch.int32,
                                         device=device),
            seq_lens=torch.tensor([T], dtype=torch.int32, device=device),
            block_table=torch.tensor([[1]], dtype=torch.int32,
                                     device=device),
            slot_mapping=torch.arange(64, 64 + T, dtype=torch.int64,
                                      device=device),
            num_reqs=1,
            num_actual_tokens=T,
            max_query_len=T,
            max_seq_len=T,
            num_decodes=0,
        )
        ctx = ForwardContext(attn_metadata=meta, kv_caches=caches)
        with set_forward_context(ctx), torch.inference_mode():
            h = model(ids, pos)
            logits = model.compute_logits(h)
        return logits.float().cpu()

    gpu = run("cuda", "bf16")
    cpu = run("cpu", "fp32")
    cos = torch.nn.functional.cosine_similarity(gpu, cpu, dim=-1)
    # bf16 2-layer stack vs fp32: tighter than an earlier gate (0.99 /
    # 0.8 argmax, loose enough to hide drift) while leaving bf16
    # headroom; op-level tests carry the per-kernel tolerances.
    assert cos.min() > 0.995, cos
    assert (gpu.argmax(-1) == cpu.argmax(-1)).float().mean() > 0.85
    # Absolute scale agreement too (functioning init => O(1) logits).
    rel = (gpu - cpu).abs().max() / cpu.abs().max().clamp_min(1e-6)
    assert rel < 0.3, rel


@pytest.mark.parametrize("m,k,n,bias", [
    (7, 512, 1024, False),
    (256, 4096, 6144, False),
    (256, 14336, 4096, False),
    (1024, 4096, 4096, True),
])
def test_lt_linear(m, k, n, bias):
    hip = _hip()
    a = torch.randn(m, k, dtype=torch.bfloat16, device="cuda") * 0.1
    w = torch.randn(n, k, dtype=torch.bfloat16, device="cuda") * 0.1
    b = (torch.randn(n, dtype=torch.bfloat16, device="cuda")
         if bias else None)
    out = hip.linear(a, w, b)
    expect = torch.nn.functional.linear(
        a.float(), w.float(), b.float() if bias else None)
    assert_close(out, expect, atol=5e-2, rtol=5e-2)


@pytest.mark.parametrize("first", ["fp32", "fp8"])
def test_algorithms_are_chosen_by_types(first):
    """Products of the same sizes in fp32 and in fp8, one after the other:
    each runs by an algorithm of its own types."""
    hip = _hip()
    m, n, k = (272, 640, 512) if first == "fp32" else (272, 512, 640)
    a = torch.randint(-4, 5, (m, k), device="cuda").float() / 4
    w = torch.randint(-4, 5, (n, k), device="cuda").float() / 4
    expect = a @ w.t()   # fp8 holds these, fp32 their sums

    def fp32():
        assert torch.equal(hip._C.lt_linear(a, w, None), expect)

    def fp8():
        out = hip._C.lt_linear_fp8(a.to(torch.float8_e4m3fn),
                                   w.to(torch.float8_e4m3fn))
        assert torch.equal(out, expect.bfloat16())

    for run in (fp32, fp8) if first == "fp32" else (fp8, fp32):
        run()


def test_fused_moe_matches_reference():
    T, H, I, E, K = 37, 256, 512, 4, 2
    hidden = torch.randn(T, H, dtype=torch.bfloat16, device="cuda") * 0.1
    w13 = torch.randn(E, 2 * I, H, dtype=torch.bfloat16, device="cuda") * 0.1
    w2 = torch.randn(E, H, I, dtype=torch.bfloat16, device="cuda") * 0.1
    logits = torch.randn(T, E, dtype=torch.float32, device="cuda")
    hip = _hip()
    tw, ti = hip.topk_softmax(logits, K)
    out = hip.fused_moe(hidden, w13, w2, tw, ti)
    expect = ref.fused_moe(hidden.float(), w13.float(), w2.float(), tw, ti)
    assert_close(out, expect, atol=5e-2, rtol=5e-2)


def test_fp8_kv_cache_attention():
    """fp8 e4m3fn KV cache: write-path conversion + decode/prefill reads
    must match the fp32 reference within fp8 quantization error."""
    hip = _hip()
    n, Hq, Hkv, D, BS = 4, 8, 2, 128, 64
    ctx = 300
    nb = (ctx + BS - 1) // BS
    kfull = torch.randn(n * ctx, Hkv, D, dtype=torch.bfloat16,
                        device="cuda")
    vfull = torch.randn(n * ctx, Hkv, D, dtype=torch.bfloat16,
                        device="cuda")
    cache = torch.zeros(2, n * nb + 1, Hkv, BS, D,
                        dtype=torch.float8_e4m3fn, device="cuda")
    bt = torch.zeros(n, nb, dtype=torch.int32, device="cuda")
    slots = []
    for i in range(n):
        bt[i] = torch.arange(1 + i * nb, 1 + (i + 1) * nb)
        base = (1 + i * nb) * BS
        slots.extend(range(base, base + ctx))
    slots = torch.tensor(slots, dtype=torch.int64, device="cuda")
    hip.reshape_and_cache(kfull, vfull, cache, slots)
    # Reference cache written by torch conversions.
    ref_cache = torch.zeros_like(cache)
    ref.reshape_and_cache(kfull, vfull, ref_cache, slots)
    assert (cache.view(torch.uint8) == ref_cache.view(torch.uint8)) \
        .float().mean() > 0.999

    q = torch.randn(n, Hq, D, dtype=torch.bfloat16, device="cuda")
    qsl = torch.arange(n + 1, dtype=torch.int32, device="cuda")
    sl = torch.full((n,), ctx, dtype=torch.int32, device="cuda")
    scale = D**-0.5
    out = hip.attention_unified(q, cache, bt, qsl, sl, scale,
                                num_decodes=n, max_seq_len=ctx,
                                max_query_len=1)
    expect = ref.attention_unified(q, ref_cache, bt, qsl, sl, scale,
                                   num_decodes=n)
    assert_close(out, expect, atol=6e-2, rtol=6e-2)

    # Prefill read path over the fp8 cache.
    ql = 32
    q2 = torch.randn(n * ql, Hq, D, dtype=torch.bfloat16, device="cuda")
    qsl2 = torch.arange(0, n * ql + 1, ql, dtype=torch.int32, device="cuda")
    out2 = hip.attention_unified(q2, cache, bt, qsl2, sl, scale,
                                 num_decodes=0, max_seq_len=ctx,
                                 max_query_len=ql)
    expect2 = ref.attention_unified(q2, ref_cache, bt, qsl2, sl, scale,
                                    num_decodes=0)
    assert_close(out2, expect2, atol=6e-2, rtol=6e-2)


@pytest.mark.parametrize("window", [8, 64, 200])
def test_decode_attention_sliding_window(window):
    hip = _hip()
    Hkv, group = 2, 4
    Hq = Hkv * group
    n, ctx = 4, 150
    q, cache, bt, qsl, sl = _make_paged(n, [1] * n, [ctx] * n, Hq, Hkv)
    scale = 1.0 / 128**0.5
    out = hip.attention_unified(q, cache, bt, qsl, sl, scale,
                                num_decodes=n, max_seq_len=ctx,
                                max_query_len=1, sliding_window=window)
    expect = ref.attention_unified(q, cache, bt, qsl, sl, scale,
                                   num_decodes=n, sliding_window=window)
    assert_close(out, expect, msg=f"window={window}")


@pytest.mark.parametrize("window", [16, 128])
def test_prefill_attention_sliding_window(window):
    hip = _hip()
    Hkv, group = 2, 4
    Hq = Hkv * group
    q_lens, ctx_lens = [17, 70], [100, 300]
    n = len(q_lens)
    q, cache, bt, qsl, sl = _make_paged(n, q_lens, ctx_lens, Hq, Hkv)
    scale = 1.0 / 128**0.5
    out = hip.attention_unified(
        q, cache, bt, qsl, sl, scale, num_decodes=0,
        max_seq_len=max(ctx_lens), max_query_len=max(q_lens),
        sliding_window=window)
    expect = ref.attention_unified(q, cache, bt, qsl, sl, scale,
                                   num_decodes=0, sliding_window=window)
    assert_close(out, expect, msg=f"window={window}")


@pytest.mark.parametrize("hd", [64, 256])
@pytest.mark.parametrize("group", [1, 2, 8])
@pytest.mark.parametrize("ctx", [30, 144, 1500])
def test_decode_attention_head_dims(hd, group, ctx):
    """head_dim 64 (OPT-class) and 256 (Gemma3-class) decode paths of the
    HD-templated kernel vs the torch reference."""
    hip = _hip()
    Hkv = 2
    Hq = Hkv * group
    n = 3
    q, cache, bt, qsl, sl = _make_paged(n, [1] * n, [ctx] * n, Hq, Hkv,
                                        D=hd)
    scale = 1.0 / hd**0.5
    out = hip.attention_unified(q, cache, bt, qsl, sl, scale,
                                num_decodes=n, max_seq_len=ctx,
                                max_query_len=1)
    expect = ref.attention_unified(q, cache, bt, qsl, sl, scale,
                                   num_decodes=n)
    assert_close(out, expect, msg=f"hd={hd} group={group} ctx={ctx}")


@pytest.mark.parametrize("hd", [64, 256])
def test_decode_attention_head_dims_window(hd):
    hip = _hip()
    Hkv, group = 2, 2
    Hq = Hkv * group
    n, ctx = 3, 300
    q, cache, bt, qsl, sl = _make_paged(n, [1] * n, [ctx] * n, Hq, Hkv,
                                        D=hd)
    scale = 1.0 / hd**0.5
    out = hip.attention_unified(q, cache, bt, qsl, sl, scale,
                                num_decodes=n, max_seq_len=ctx,
                                max_query_len=1, sliding_window=128)
    expect = ref.attention_unified(q, cache, bt, qsl, sl, scale,
                                   num_decodes=n, sliding_window=128)
    assert_close(out, expect, msg=f"hd={hd}")


@pytest.mark.parametrize("hd", [64, 256])
def test_prefill_other_head_dims(hd):
    """Mixed decode+prefill at head_dim 64/256: both row kinds now run
    the templated MFMA/HIP kernels (Gemma3 256, OPT 64)."""
    hip = _hip()
    Hkv, group = 2, 2
    Hq = Hkv * group
    q_lens = [1, 1, 40]
    ctx_lens = [90, 33, 40]
    q, cache, bt, qsl, sl = _make_paged(3, q_lens, ctx_lens, Hq, Hkv, D=hd)
    scale = 1.0 / hd**0.5
    out = hip.attention_unified(q, cache, bt, qsl, sl, scale,
                                num_decodes=2, max_seq_len=90,
                                max_query_len=40)
    expect = ref.attention_unified(q, cache, bt, qsl, sl, scale,
                                   num_decodes=2)
    assert_close(out, expect, msg=f"hd={hd}")


@pytest.mark.parametrize("T,H,I,E,K", [
    (1, 128, 64, 4, 2),        # single decode token
    (64, 256, 512, 8, 2),      # mixtral-shaped decode batch
    (37, 256, 128, 16, 4),     # skewed routing, many experts
    (512, 128, 192, 64, 8),    # deepseek-ish expert count, K=8
])
def test_moe_grouped_gemm_kernel(T, H, I, E, K):
    """fused_moe_hip (csrc/moe.hip grouped MFMA GEMM + align + combine)
    vs the fp32 torch reference, across batch/expert/topk sweeps incl.
    empty experts (E > T*K cases route nothing to most experts)."""
    hip = _hip()
    assert hip._moe_hip_ok(
        torch.zeros(1, H, dtype=torch.bfloat16), torch.zeros(E, 2 * I, H),
        None, "silu")
    hidden = torch.randn(T, H, dtype=torch.bfloat16, device="cuda") * 0.3
    w13 = torch.randn(E, 2 * I, H, dtype=torch.bfloat16, device="cuda") * 0.2
    w2 = torch.randn(E, H, I, dtype=torch.bfloat16, device="cuda") * 0.2
    logits = torch.randn(T, E, dtype=torch.float32, device="cuda")
    tw, ti = hip.topk_softmax(logits, K)
    out = hip.fused_moe_hip(hidden, w13, w2, tw, ti)
    expect = ref.fused_moe(hidden.float(), w13.float(), w2.float(), tw, ti)
    assert_close(out, expect, atol=8e-2, rtol=8e-2)


# An expert of more row tiles than a wave finds at a time, between one of a row
# and one of a group and a tile: 77 row tiles of 256, in the second product all
# of them on every XCD (24 column blocks in 8 parts); and of 128, beside 400.
@pytest.mark.parametrize("form,rows", [
    (2, [1, 66 * 256 + 5, 2300, 0]),
    (1, [1, 66 * 128 + 5, 1100, 0] + [3] * 396)])
def test_moe_expert_of_many_tiles(form, rows):
    hip = _hip()
    H, I, E = 6144, 64, len(rows)
    T = sum(rows)
    assert hip._moe_form(T, T, E, H) == form
    tile = 128 * form
    experts = [e for e, n in enumerate(rows) for _ in range(-(-n // tile))]
    assert experts.count(1) == 67
    flat = hip._C.moe_tile_order(experts, H // 256, 8, tile)
    assert {(m, n) for m, n in zip(flat[1::3], flat[2::3])} == {
        (m, n) for m in range(len(experts)) for n in range(H // 256)}
    assert flat[::3].count(0) == len(experts) * 3   # an eighth of the blocks
    hidden = torch.randn(T, H, dtype=torch.bfloat16, device="cuda") * 0.04
    w13 = torch.randn(E, 2 * I, H, dtype=torch.bfloat16, device="cuda") * 0.2
    w2 = torch.randn(E, H, I, dtype=torch.bfloat16, device="cuda") * 0.2
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(rows))
    ids = ids[torch.randperm(T)].view(T, 1).cuda()
    w = torch.rand(T, 1, device="cuda")
    out = hip.fused_moe_hip(hidden, w13, w2, w, ids)
    # An expert at a time: the reference's products are of all tokens.
    expect = torch.empty_like(hidden, dtype=torch.float32)
    for e in range(E):
        mine = ids[:, 0] == e
        gate, up = (hidden[mine].float() @ w13[e].float().t()).chunk(2, -1)
        act = torch.nn.functional.silu(gate) * up
        expect[mine] = act @ w2[e].float().t() * w[mine]
    assert_close(out, expect, atol=8e-2, rtol=8e-2)


# Captured under inference mode like the engine's own captures: the
# default CUDA generator's capture state may have been created by an
# earlier inference-mode step, and capture_begin updates it in place.
@torch.inference_mode()
def test_moe_hip_graph_capturable():
    """The grouped-GEMM path must capture and replay in a hipGraph with
    correct results (static shapes, no host syncs)."""
    hip = _hip()
    T, H, I, E, K = 32, 256, 256, 8, 2
    hidden = torch.randn(T, H, dtype=torch.bfloat16, device="cuda") * 0.3
    w13 = torch.randn(E, 2 * I, H, dtype=torch.bfloat16, device="cuda") * 0.2
    w2 = torch.randn(E, H, I, dtype=torch.bfloat16, device="cuda") * 0.2
    logits = torch.randn(T, E, dtype=torch.float32, device="cuda")
    tw, ti = hip.topk_softmax(logits, K)
    static_h = hidden.clone()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        hip.fused_moe_hip(static_h, w13, w2, tw, ti)
    torch.cuda.current_stream().wait_stream(s)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = hip.fused_moe_hip(static_h, w13, w2, tw, ti)
    for scale in (1.0, 2.0):
        static_h.copy_(hidden * scale)
        g.replay()
        torch.cuda.synchronize()
        expect = ref.fused_moe((hidden * scale).float(), w13.float(),
                               w2.float(), tw, ti)
        assert_close(out, expect, atol=8e-2, rtol=8e-2)


@pytest.mark.parametrize("T,Hq,ctx", [
    (1, 128, 33),       # single seq, TP=1 head count, partial subtile
    (4, 128, 300),      # multi-seq single-partition
    (3, 16, 2500),      # TP=8 head count, multi-partition (>1024)
    (2, 32, 1024),      # exact partition boundary
])
def test_mla_decode_kernel(T, Hq, ctx):
    """MFMA MLA decode (csrc/mla.hip) vs the fp32 torch composition over
    the compressed latent cache (DeepSeek geometry: lora 512 + rope 64)."""
    hip = _hip()
    lora, rope, bs = 512, 64, 16
    nb_per = (ctx + bs - 1) // bs
    total_blocks = T * nb_per + 1
    kv_cache = (torch.randn(total_blocks, bs, lora + rope,
                            dtype=torch.bfloat16, device="cuda") * 0.5)
    block_table = torch.zeros(T, nb_per, dtype=torch.int32, device="cuda")
    perm = torch.randperm(T * nb_per, device="cuda").int() + 1
    block_table[:] = perm.view(T, nb_per)
    seq_lens = torch.full((T,), ctx, dtype=torch.int32, device="cuda")
    seq_lens[0] = max(1, ctx - 7)  # ragged lengths
    q_nope = torch.randn(T, Hq, lora, dtype=torch.bfloat16,
                         device="cuda") * 0.3
    q_pe = torch.randn(T, Hq, rope, dtype=torch.bfloat16, device="cuda") * 0.3
    scale = (128 + 64) ** -0.5
    out = hip.mla_decode(q_nope, q_pe, kv_cache, block_table, seq_lens,
                         scale, ctx)
    qsl = torch.arange(T + 1, dtype=torch.int32, device="cuda")
    expect = ref.mla_attention(q_nope.float(), q_pe.float(),
                               kv_cache.float(), block_table, qsl,
                               seq_lens, scale)
    assert_close(out, expect, atol=4e-2, rtol=4e-2)


# Workgroups of 32, 64 and 128 heads; heads that end within one, and within a
# wave's 16; keys of one tile, whole and in parts.
@pytest.mark.parametrize("T,Hq,wide,bound", [
    (3, 128, 32, 200), (2, 72, 32, 64), (17, 128, 32, 900),
    (64, 100, 32, 130), (24, 128, 64, 2176), (100, 90, 64, 500),
    (100, 128, 128, 1500), (5, 33, 128, 1500)])
def test_mla_decode_head_groups(T, Hq, wide, bound):
    hip = _hip()
    parts = hip._mla_split(T, Hq, bound)
    assert hip._C.mla_group_heads(T * parts, Hq) == wide
    ctx = [1 + (bound - 1) * i // max(T - 1, 1) for i in range(T - 1)] + [bound]
    nb = -(-bound // 64)
    kv = torch.randn(T * nb, 64, 576, dtype=torch.bfloat16, device="cuda")
    bt = torch.randperm(T * nb, device="cuda").int().view(T, nb)
    sl = torch.tensor(ctx, dtype=torch.int32, device="cuda")
    qn = torch.randn(T, Hq, 512, dtype=torch.bfloat16, device="cuda") * 0.3
    qp = torch.randn(T, Hq, 64, dtype=torch.bfloat16, device="cuda") * 0.3
    out = hip.mla_decode(qn, qp, kv, bt, sl, 0.07, bound)
    expect = ref.mla_attention(
        qn.float(), qp.float(), kv.float(), bt,
        torch.arange(T + 1, dtype=torch.int32, device="cuda"), sl, 0.07)
    # As below: weights and results rounded to 16 bits, values up to 4.
    assert_close(out, expect, atol=8 * 2**-8, rtol=2 * 2**-8)


@pytest.mark.parametrize("heads,bs,dtype", [
    (128, 64, torch.bfloat16),   # whole tiles from one cache block
    (130, 16, torch.bfloat16),   # second head group nearly empty
    (20, 128, torch.float16),    # idle waves
])
def test_mla_attention_edges(heads, bs, dtype):
    """Decode rows and prompt portions around the 64-key tile, an empty
    portion, padded partitions; unwritten rows of the last block hold
    NaN. Tolerance: weights of decode rows and all outputs are rounded to
    16 bits, values up to 4."""
    hip = _hip()
    q_lens = [1, 1, 1, 2, 0, 65, 40]
    ctx = [1, 65, 700, 64, 5, 130, 40]
    n, T = len(ctx), sum(q_lens)
    nb = -(-max(ctx) // bs)
    cache = torch.randn(n * nb, bs, 576, device="cuda", dtype=dtype)
    bt = torch.randperm(n * nb, device="cuda").int().view(n, nb)
    for i, c in enumerate(ctx):
        if c % bs:
            cache[bt[i, c // bs], c % bs:] = float("nan")
    qn = torch.randn(T, heads, 512, device="cuda", dtype=dtype)
    qp = torch.randn(T, heads, 64, device="cuda", dtype=dtype)
    qsl = torch.tensor([0] + [sum(q_lens[:i + 1]) for i in range(n)],
                       device="cuda", dtype=torch.int32)
    sl = torch.tensor(ctx, device="cuda", dtype=torch.int32)
    out = hip.mla_attention(qn, qp, cache, bt, qsl, sl, 0.07,
                            num_decodes=3, max_seq_len=max(ctx))
    expect = ref.mla_attention(qn.float(), qp.float(), cache.float(), bt,
                               qsl, sl, 0.07)
    atol = 2 * 4 * (2**-8 if dtype == torch.bfloat16 else 2**-11)
    assert_close(out, expect, atol=atol, rtol=atol / 4)


@pytest.mark.parametrize("T,H,K,N", [(1, 3, 128, 512), (65, 2, 512, 128),
                                     (130, 1, 256, 256)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_head_matmul(T, H, K, N, dtype):
    """Strided head slices, ragged token tiles, several K steps. fp32
    sums: off by the result's own rounding (2^-8, 2^-11) at most."""
    hip = _hip()
    x = torch.randn(T, H, K + 64, device="cuda", dtype=dtype)[..., :K]
    w = torch.randn(H, K, N, device="cuda", dtype=dtype) * K**-0.5
    assert_close(hip.head_matmul(x, w), ref.head_matmul(x, w),
                 atol=2**-9, rtol=2**-8 if dtype == torch.bfloat16
                 else 2**-10)


# Four steps of K at once up to 256 workgroups (both sides), and five steps.
# Off from sums that are not rounded by the result's own rounding: 2^-8 of it
# (from rounded ones by twice that, where a sum lies between two results).
@pytest.mark.parametrize("T,H,K,N", [(128, 128, 512, 128), (129, 86, 512, 128),
                                     (3, 2, 640, 128)])
def test_head_matmul_steps(T, H, K, N):
    hip = _hip()
    x = torch.randn(T, H, K, device="cuda", dtype=torch.bfloat16)
    w = torch.randn(H, K, N, device="cuda", dtype=torch.bfloat16) * K**-0.5
    assert_close(hip.head_matmul(x, w), ref.head_matmul(x.float(), w.float()),
                 atol=2**-9, rtol=2**-8)


@pytest.mark.parametrize("T,H,I,E,K,act", [
    (33, 128, 128, 6, 2, "relu2"),    # streamed, part of a 64-row tile
    (1100, 128, 64, 128, 2, "silu"),  # streamed, counted by blocks of rows
    (70, 256, 192, 5, 2, "silu"),     # 128-row tiles, ragged last columns
    (260, 128, 128, 3, 1, "relu2"),
    (1100, 128, 192, 4, 2, "silu"),   # 256-row tiles
    (400, 384, 128, 2, 1, "relu2"),
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_moe_forms(T, H, I, E, K, act, dtype):
    """Each form of the expert products, half of the rows on one expert
    and none on the last. Against 64 bits; three roundings to the type
    (activation, expert's output, sum) and fp32 sums bound the error."""
    hip = _hip()
    hidden = torch.randn(T, H, device="cuda", dtype=dtype)
    g = 2 if act == "silu" else 1
    w13 = torch.randn(E, g * I, H, device="cuda", dtype=dtype) * H**-0.5
    w2 = torch.randn(E, H, I, device="cuda", dtype=dtype) * I**-0.5
    ti = torch.randint(0, E - 1, (T, K), device="cuda", dtype=torch.int32)
    ti[: T // 2, 0] = 0
    tw = torch.rand(T, K, device="cuda")
    out = hip.fused_moe(hidden, w13, w2, tw, ti, act).double()
    expect, bound = torch.zeros_like(out), torch.zeros_like(out)
    for e in range(E):
        t, k = (ti == e).nonzero(as_tuple=True)
        y = hidden[t].double() @ w13[e].double().T
        a = (torch.nn.functional.silu(y[:, :I]) * y[:, I:] if g == 2
             else y.relu() ** 2)
        w = tw[t, k].double()[:, None]
        y, mag = a @ w2[e].double().T, a.abs() @ w2[e].double().abs().T
        expect.index_add_(0, t, w * y)
        bound.index_add_(0, t, w * (mag + y.abs()))
    # Rounding to p significant bits is off by 2^-p of the value: p = 8, 11.
    eps = 2**-8 if dtype == torch.bfloat16 else 2**-11
    assert ((out - expect).abs()
            <= 1.1 * eps * (bound + expect.abs()) + 2**-20).all()


@pytest.mark.parametrize("nd,qls,ctxs,H,bs,at_once", [
    (0, [130], [130], 3, 64, 3),               # no context before it
    (2, [1, 1, 200, 57, 131], [70, 300, 200, 311, 131], 10, 16, 4),
    (0, [1, 300, 128], [1, 300, 128], 16, 64, 16),
    (1, [1, 129, 255], [5, 640, 257], 2, 80, 1),
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_mla_heads(nd, qls, ctxs, H, bs, at_once, dtype, monkeypatch):
    """Prompt portions with keys and values carried out of the latent
    space: ragged tiles, contexts before the portion, several passes over
    the heads. Scores of unit variance are off by at most 4 * 2^-8 (2^-11)
    through rounded queries and keys, values up to 4 by as much, the
    result once more; the reference's own roundings double that."""
    hip = _hip()
    n, S, T = len(qls), max(ctxs), sum(qls)
    nb = (S + bs - 1) // bs
    cache = torch.randn(n * nb, bs, 576, device="cuda", dtype=dtype)
    bt = torch.randperm(n * nb, device="cuda").to(torch.int32).view(n, nb)
    q = torch.randn(T, H, 192, device="cuda", dtype=dtype)
    qn, qp = q[..., :128], q[..., 128:].contiguous()
    wk = torch.randn(H, 128, 512, device="cuda", dtype=dtype) * 512**-0.5
    wv = torch.randn(H, 512, 128, device="cuda", dtype=dtype) * 512**-0.5
    qsl = torch.tensor([sum(qls[:i]) for i in range(n + 1)], device="cuda",
                       dtype=torch.int32)
    sl = torch.tensor(ctxs, device="cuda", dtype=torch.int32)
    monkeypatch.setattr(hip, "_MLA_PROMPT_SCRATCH",
                        at_once * (n - nd) * S * 512)
    assert hip._mla_prompt_heads(qn, wk, wv, cache, n, 1.0, nd, max(qls),
                                 S) == at_once
    out = hip.mla_heads(qn, qp, wk, wv, cache, bt, qsl, sl, 192**-0.5,
                        num_decodes=nd, max_query_len=max(qls),
                        max_seq_len=S)
    expect = ref.mla_heads(qn.float(), qp.float(), wk.float(), wv.float(),
                           cache.float(), bt, qsl, sl, 192**-0.5)
    atol = 2 * 4 * (2**-8 if dtype == torch.bfloat16 else 2**-11)
    assert_close(out, expect, atol=atol, rtol=atol / 4)


@pytest.mark.parametrize("T,H", [(1, 3), (5, 128), (70, 65)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_mla_prepare(T, H, dtype):
    """Strided inputs, a padding slot, untouched rows stay. fp32 math of
    the same 16-bit values: one rounding, or its neighbour."""
    hip = _hip()
    q = torch.randn(T, H, 192, device="cuda", dtype=dtype)[..., 128:]
    kv_a = torch.randn(T, 584, device="cuda", dtype=dtype)[:, :576]
    w = torch.randn(512, device="cuda", dtype=dtype)
    cs = torch.randn(100, 64, device="cuda")
    pos = torch.randint(0, 100, (T,), device="cuda")
    cache = torch.randn(12, 16, 576, device="cuda", dtype=dtype)
    want = cache.float()
    slots = torch.randperm(12 * 16, device="cuda")[:T]
    pad = torch.cat([slots[:-1], slots.new_tensor([-1])])
    out = hip.mla_prepare(pos, q, kv_a, w, 1e-5, cs, cache, pad)
    keep = slice(0, T - 1)
    ref.mla_prepare(pos[keep], q[keep].float(), kv_a[keep].float(),
                    w.float(), 1e-5, cs, want, slots[keep])
    qf = q.float().contiguous()
    ref.apply_rope(pos, qf, torch.zeros_like(qf), cs, 64)
    tol = dict(atol=2**-12, rtol=2**-7 if dtype == torch.bfloat16
               else 2**-10)
    assert_close(out, qf, **tol)
    assert_close(cache, want, **tol)


@pytest.mark.parametrize("T,Hq,Hkv,D,rot,bs", [
    (1, 4, 1, 64, 64, 16), (9, 32, 8, 128, 128, 64), (3, 5, 5, 80, 16, 16),
    (70, 40, 8, 256, 128, 64)])
@pytest.mark.parametrize("dtype,fp8", [
    (torch.bfloat16, False), (torch.float16, False), (torch.bfloat16, True)])
def test_rope_and_cache(T, Hq, Hkv, D, rot, bs, dtype, fp8):
    """Slices of one projection, partial rotation, a padding slot. The
    same fp32 math on 16-bit values as rotation and cache write apart:
    the cached bytes are the same."""
    hip = _hip()
    qkv = torch.randn(T, (Hq + 2 * Hkv) * D, device="cuda", dtype=dtype)
    both = qkv.clone()
    cs = torch.randn(100, rot, device="cuda")
    pos = torch.randint(0, 100, (T,), device="cuda")
    cache = torch.zeros(2, 12, Hkv, bs, D, device="cuda", dtype=dtype)
    if fp8:
        cache = cache.to(torch.float8_e4m3fn)
    want = cache.clone()
    slots = torch.randperm(12 * bs, device="cuda")[:T]
    if T > 1:
        slots[T // 2] = -1

    def split(x):
        return [y.view(T, -1, D) for y in
                x.split([Hq * D, Hkv * D, Hkv * D], dim=1)]

    q, k, v = split(qkv)
    hip.rope_and_cache(pos, q, k, v, cs, rot, True, cache, slots)
    q2, k2, v2 = split(both)
    hip.apply_rope(pos, q2, k2, cs, rot)
    hip.reshape_and_cache(k2, v2, want, slots)
    assert torch.equal(q, q2)
    assert torch.equal(cache.view(torch.uint8), want.view(torch.uint8))


@pytest.mark.parametrize("T", [1, 70])
def test_mla_a_projections_as_one(T):
    """One product over both weights, through a move of the module, and
    the norm of rows of a wider matrix: the same as apart but for the order
    of fp32 sums, one rounding of values up to about 4 (2^-8 of them)."""
    from vllm_amd.config import get_model_spec
    from vllm_amd.models.deepseek import DeepseekMLAAttention

    block = DeepseekMLAAttention(get_model_spec("deepseek-v3-lite"), 0,
                                 torch.bfloat16, 64)
    for p in block.parameters():
        p.data.normal_(std=0.01)
    block = block.cuda()
    q, kv = block.q_a_proj.weight, block.kv_a_proj_with_mqa.weight
    assert kv.data_ptr() == q.data_ptr() + 2 * q.numel()
    x = torch.randn(T, q.shape[1], device="cuda", dtype=torch.bfloat16)
    q_a, kv_a = block._a_projs(x)
    assert not T > 1 or not q_a.is_contiguous()
    assert_close(q_a, x.float() @ q.float().T, atol=2**-8, rtol=2**-7)
    assert_close(kv_a, x.float() @ kv.float().T, atol=2**-8, rtol=2**-7)
    assert torch.equal(block.q_a_layernorm(q_a),
                       block.q_a_layernorm(q_a.contiguous()))
    kv.data = kv.data.clone()     # no longer behind the other: apart
    assert_close(block._a_projs(x)[1], kv_a, atol=2**-8, rtol=2**-7)


def test_mla_unified_dispatch_mixed_batch():
    """hip_ops.mla_attention runs decode rows (mla_decode) and prompt rows
    (mla_prefill) of one batch on the kernel; both must agree with the
    all-torch result."""
    hip = _hip()
    lora, rope, bs, Hq = 512, 64, 16, 32
    T_dec, ql_pre, ctx_pre = 3, 5, 40
    ctx_dec = 77
    nb = 16
    kv_cache = torch.randn(64, bs, lora + rope, dtype=torch.bfloat16,
                           device="cuda") * 0.5
    bt = torch.arange(4 * nb, dtype=torch.int32, device="cuda").view(4, nb)
    seq_lens = torch.tensor([ctx_dec, ctx_dec, ctx_dec, ctx_pre],
                            dtype=torch.int32, device="cuda")
    qsl = torch.tensor([0, 1, 2, 3, 3 + ql_pre], dtype=torch.int32,
                       device="cuda")
    Ttot = 3 + ql_pre
    q_nope = torch.randn(Ttot, Hq, lora, dtype=torch.bfloat16,
                         device="cuda") * 0.3
    q_pe = torch.randn(Ttot, Hq, rope, dtype=torch.bfloat16,
                       device="cuda") * 0.3
    scale = 0.08
    out = hip.mla_attention(q_nope, q_pe, kv_cache, bt, qsl, seq_lens,
                            scale, num_decodes=T_dec, max_seq_len=ctx_dec)
    expect = ref.mla_attention(q_nope.float(), q_pe.float(),
                               kv_cache.float(), bt, qsl, seq_lens, scale)
    assert_close(out, expect, atol=4e-2, rtol=4e-2)


@pytest.mark.parametrize("hd", [64, 128, 256])
@pytest.mark.parametrize("q_lens,ctx_lens", [
    ([16, 33], [16, 33]),                 # pure prefill from scratch
    ([17, 70], [100, 300]),               # chunked-prefill continuation
    ([1, 1, 5, 200], [40, 513, 60, 200]),  # mixed decode+prefill
])
def test_prefill_attention_head_dim_sweep(hd, q_lens, ctx_lens):
    """head_dim-templated MFMA prefill (64/128/256) vs fp32 reference."""
    hip = _hip()
    Hkv = 2
    Hq = Hkv * 4
    n = len(q_lens)
    num_decodes = sum(1 for x in q_lens if x == 1)
    order = sorted(range(n), key=lambda i: q_lens[i] != 1)
    q_lens = [q_lens[i] for i in order]
    ctx_lens = [ctx_lens[i] for i in order]
    q, cache, bt, qsl, sl = _make_paged(n, q_lens, ctx_lens, Hq, Hkv, D=hd)
    scale = 1.0 / hd**0.5
    out = hip.attention_unified(
        q, cache, bt, qsl, sl, scale, num_decodes=num_decodes,
        max_seq_len=max(ctx_lens), max_query_len=max(q_lens))
    expect = ref.attention_unified(q, cache, bt, qsl, sl, scale,
                                   num_decodes=num_decodes)
    assert_close(out, expect, msg=f"hd={hd}")


@pytest.mark.parametrize("T,H,I,E,K", [
    (64, 256, 512, 8, 2),
    (37, 256, 128, 16, 4),
])
def test_moe_shuffled_weight_gemm(T, H, I, E, K):
    """Fragment-major pre-shuffled weight stream (moe_gemm_shuf) must
    match the stream of plain weights and the fp32 reference."""
    hip = _hip()
    hidden = torch.randn(T, H, dtype=torch.bfloat16, device="cuda") * 0.3
    w13 = torch.randn(E, 2 * I, H, dtype=torch.bfloat16, device="cuda") * 0.2
    w2 = torch.randn(E, H, I, dtype=torch.bfloat16, device="cuda") * 0.2
    logits = torch.randn(T, E, dtype=torch.float32, device="cuda")
    tw, ti = hip.topk_softmax(logits, K)
    w13s = hip.moe_shuffle_weights(w13)
    w2s = hip.moe_shuffle_weights(w2)
    out = hip.fused_moe_hip(hidden, w13, w2, tw, ti,
                            w13_shuf=w13s, w2_shuf=w2s)
    base = hip.fused_moe_hip(hidden, w13, w2, tw, ti)
    expect = ref.fused_moe(hidden.float(), w13.float(), w2.float(), tw, ti)
    assert_close(out, base, atol=1e-3, rtol=1e-3)  # same math, same order
    assert_close(out, expect, atol=8e-2, rtol=8e-2)


@pytest.mark.parametrize("heads,bs,dtype", [
    (128, 64, torch.bfloat16),
    (130, 16, torch.bfloat16),
    (20, 64, torch.float16),
])
@pytest.mark.parametrize("bound", [1300, 500, 0])
def test_mla_prompt_keys_split(heads, bs, dtype, bound):
    """Few prompt tokens after long contexts: their keys go over
    partitions, of which some rows fill one, some all, by a bound that is
    exact, too short (the last partition takes what is left) or missing.
    Tolerance: queries and keys are exact here, so only the results'
    rounding and the order of sums are left, of values up to 4."""
    hip = _hip()
    q_lens, ctx = [1, 2, 0, 5, 1], [70, 1300, 9, 640, 33]
    n, T, nb = 5, sum(q_lens), -(-1300 // bs)
    cache = torch.randn(n * nb, bs, 576, device="cuda", dtype=dtype)
    bt = torch.randperm(n * nb, device="cuda").int().view(n, nb)
    qn = torch.randn(T, heads, 512, device="cuda", dtype=dtype)
    qp = torch.randn(T, heads, 64, device="cuda", dtype=dtype)
    qsl = torch.tensor([0, 1, 3, 3, 8, 9], device="cuda", dtype=torch.int32)
    sl = torch.tensor(ctx, device="cuda", dtype=torch.int32)
    out = hip.mla_attention(qn, qp, cache, bt, qsl, sl, 0.07, num_decodes=1,
                            max_prompt_len=bound)
    expect = ref.mla_attention(qn.float(), qp.float(), cache.float(), bt,
                               qsl, sl, 0.07)
    atol = 2 * 4 * (2**-8 if dtype == torch.bfloat16 else 2**-11)
    assert_close(out, expect, atol=atol, rtol=atol / 4)


@pytest.mark.parametrize("T", [40, 1100])  # one block of rows, two
@torch.inference_mode()   # as the runner captures
def test_moe_more_experts_than_lds_counters(T):
    """More experts than LDS counters take the same path, captured too:
    no synchronisation, each replay gives the eager bytes. Every row's
    result against its two experts in 64 bits, within three roundings to
    bf16 (2^-8 each) of sums of magnitudes."""
    hip = _hip()
    E, H, I, K = 1500, 128, 64, 2
    bf = torch.bfloat16
    x = torch.randn(T, H, device="cuda", dtype=bf)
    w13 = torch.randn(E, 2 * I, H, device="cuda", dtype=bf) * H**-0.5
    w2 = torch.randn(E, H, I, device="cuda", dtype=bf) * I**-0.5
    assert hip._moe_hip_ok(x, w13, w2, "silu")
    ids = torch.stack([torch.randperm(E, device="cuda")[:K]
                       for _ in range(T)]).int()
    ids[: T // 2, 0], ids[: T // 2, 1] = E - 1, 3
    w = torch.rand(T, K, device="cuda")
    out = hip.fused_moe(x, w13, w2, w, ids)
    y = torch.matmul(w13[ids.long()].double(), x.double()[:, None, :, None])
    a = torch.nn.functional.silu(y[:, :, :I]) * y[:, :, I:]
    w2d, wd = w2[ids.long()].double(), w.double()[..., None, None]
    terms = torch.matmul(w2d, a) * wd
    bound = (torch.matmul(w2d.abs(), a.abs()) * wd).sum(1) + terms.abs().sum(1)
    expect = terms.sum(1)
    err = (out.double()[..., None] - expect).abs()
    assert (err <= 1.1 * 2**-8 * (bound + expect.abs()) + 2**-20).all()

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        hip.fused_moe(x, w13, w2, w, ids)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        again = hip.fused_moe(x, w13, w2, w, ids)
    for _ in range(3):
        again.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(again, out)
        assert torch.equal(hip.fused_moe(x, w13, w2, w, ids), out)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_mla_prompt_key_ranges(dtype):
    """Keys outside fp16's range, far below one, or of very different size
    in the two halves of a head or in neighbouring blocks of tokens, with
    queries that make up for it: the powers of two cancel, so tolerances
    are those of ordinary heads (test_mla_heads)."""
    hip = _hip()
    n, H = 300, 8
    cache = torch.randn(5, 64, 576, device="cuda", dtype=dtype)
    bt = torch.randperm(5, device="cuda").int()[None]
    q = torch.randn(n, H, 192, device="cuda", dtype=dtype)
    wk = torch.randn(H, 128, 512, device="cuda", dtype=dtype) * 512**-0.5
    wv = torch.randn(H, 512, 128, device="cuda", dtype=dtype) * 512**-0.5
    big = 20 if dtype == torch.bfloat16 else 8
    for h, lo, hi, e in [(0, 0, 128, big), (1, 0, 128, -big),
                         (2, 0, 64, big // 2), (3, 64, 128, -big // 2),
                         (4, 0, 128, big * 3 if big == 20 else 9)]:
        wk[h, lo:hi] *= 2.0**e
        q[:, h, lo:hi] *= 2.0**-e
    q[5, 6] = 0
    # Tokens 64..127 carry larger latents, weighed down by their rotary part.
    cache[bt[0, 1], :, :512] *= 32
    qsl = torch.tensor([0, n], device="cuda", dtype=torch.int32)
    out = hip.mla_heads(q[..., :128], q[..., 128:], wk, wv, cache, bt, qsl,
                        qsl[1:].clone(), 192**-0.5, max_query_len=n,
                        max_seq_len=n)
    expect = ref.mla_heads(q[..., :128].double(), q[..., 128:].double(),
                           wk.double(), wv.double(), cache.double(), bt, qsl,
                           qsl[1:].clone(), 192**-0.5)
    assert out.isfinite().all()
    err = (out - expect).double().norm(dim=(0, 2))
    rel = err / expect.norm(dim=(0, 2))
    assert (rel < 4 * (2**-8 if dtype == torch.bfloat16 else 2**-11)).all(), \
        rel


def test_mla_prompt_precision(monkeypatch):
    """In sharp softmaxes (scores of deviation 4) the per-head form is no
    further from 64 bits than the latent one: there a query's 512 values
    are rounded to bf16 and decide the error, here a key's are fp16, an
    eighth of that; what both share, values and results in bf16, is about
    0.6 of the latent form's error."""
    hip = _hip()
    n, H, bf = 250, 16, torch.bfloat16
    cache = torch.randn(4, 64, 576, device="cuda", dtype=bf)
    bt = torch.randperm(4, device="cuda").int()[None]
    q = torch.randn(n, H, 192, device="cuda", dtype=bf) * 8
    wk = torch.randn(H, 128, 512, device="cuda", dtype=bf) * 900**-0.5
    wv = torch.randn(H, 512, 128, device="cuda", dtype=bf) * 900**-0.5
    qsl = torch.tensor([0, n], device="cuda", dtype=torch.int32)
    args = (cache, bt, qsl, qsl[1:].clone(), 192**-0.5)
    rule, err = hip._mla_prompt_heads, {}
    expect = None
    for name, form in (("heads", rule), ("latent", lambda *a: 0)):
        monkeypatch.setattr(hip, "_mla_prompt_heads", form)
        out = hip.mla_heads(q[..., :128], q[..., 128:], wk, wv, *args,
                            max_query_len=n, max_seq_len=n).double()
        if expect is None:
            expect = torch.empty_like(out)
            rows = cache[bt[0].long()].flatten(0, 1)[:n].double()
            hide = torch.ones(n, n, device="cuda").triu(1).bool()
            for h in range(H):
                k = rows[:, :512] @ wk[h].double().T
                s = (q[:, h, :128].double() @ k.T
                     + q[:, h, 128:].double() @ rows[:, 512:].T)
                p = (s * 192**-0.5).masked_fill(hide, -torch.inf).softmax(-1)
                expect[:, h] = p @ (rows[:, :512] @ wv[h].double())
        err[name] = ((out - expect).norm() / expect.norm()).item()
    assert err["heads"] < 0.8 * err["latent"], err
