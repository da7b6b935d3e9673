"""Which kernel, split and scratch a call gets: rules of ops/hip_ops.py on
host numbers alone, checked on CPU tensors with the compiled ops
replaced by recorders."""

import types

import pytest
import torch


class Recorder:
    """Stands for the compiled ops; keeps every call's arguments."""

    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        def call(*args):
            self.calls.append((name, args))
            return torch.empty(0)
        return call

    def args(self, name):
        return [a for n, a in self.calls if n == name]


@pytest.fixture
def hip(monkeypatch):
    try:
        from vllm_amd.ops import hip_ops
    except (ImportError, OSError) as e:
        pytest.skip(f"extension not built: {e}")
    monkeypatch.setattr(hip_ops, "_C", Recorder())
    return hip_ops


def _lens(*n):
    return torch.tensor(n, dtype=torch.int32)


@pytest.mark.parametrize("rows", [1, 8, 64])
def test_decode_split_ignores_prompts(hip, rows):
    """Decode rows are cut by their own longest context, not by that of a
    prompt in the same step."""
    def split(prompt):
        n = rows + bool(prompt)
        q = torch.empty(rows + prompt, 32, 128, dtype=torch.bfloat16)
        kv = torch.empty(2, 1, 8, 64, 128, dtype=torch.bfloat16)
        hip._C.calls.clear()
        hip.attention_unified(
            q, kv, torch.zeros(n, 1, dtype=torch.int32), _lens(*range(n + 1)),
            _lens(*[1000] * n), 0.1, num_decodes=rows,
            max_seq_len=max(1000, prompt), max_query_len=max(1, prompt),
            max_decode_len=1000)
        (a,) = hip._C.args("paged_decode_attention")
        return a[6], a[8].shape   # the bound on contexts, the partials

    assert split(32768) == split(0)


@pytest.mark.parametrize("rows", [1, 32])
def test_mla_decode_split_ignores_prompts(hip, rows, monkeypatch):
    def split(prompt):
        n, t = rows + bool(prompt), rows + prompt
        q = torch.empty(t, 16, 192, dtype=torch.bfloat16)
        monkeypatch.setattr(hip, "head_matmul", lambda x, w: torch.empty(
            x.shape[0], x.shape[1], w.shape[2], dtype=x.dtype))
        hip._C.calls.clear()
        hip.mla_heads(
            q[..., :128], q[..., 128:],
            torch.empty(16, 128, 512, dtype=torch.bfloat16),
            torch.empty(16, 512, 128, dtype=torch.bfloat16),
            torch.empty(1, 64, 576, dtype=torch.bfloat16),
            torch.zeros(n, 1, dtype=torch.int32), _lens(*range(n + 1)),
            _lens(*[1000] * n), 0.07, num_decodes=rows,
            max_query_len=max(1, prompt), max_seq_len=max(1000, prompt),
            max_decode_len=1000)
        (a,) = hip._C.args("mla_decode")
        return a[7], a[8].shape

    assert split(8192) == split(0)


@pytest.mark.parametrize("rows,heads,keys,parts", [
    (1, 128, 60, 1), (1, 128, 1000, 8), (1, 128, 16000, 64),
    (16, 128, 2000, 8), (64, 128, 130, 1), (128, 128, 1000, 1),
    (128, 128, 2176, 2), (32, 128, 8192, 8), (200, 128, 2176, 1),
    (300, 128, 500, 1), (1, 16, 4000, 32), (64, 16, 1000, 4)])
def test_mla_split(hip, rows, heads, keys, parts):
    assert hip._mla_split(rows, heads, keys) == parts


@pytest.mark.parametrize("rows,heads,told,parts", [
    (4, 64, 8192, 64), (6, 64, 6000, 42), (3, 128, 8192, 42),
    (8, 64, 4096, 32), (4, 128, 16384, 64),    # shorter rows would lose
    (1, 128, 4096, 32), (128, 128, 1000, 1),   # as many, or they gain too
    (3, 128, 0, 1)])
def test_mla_split_of_rows_shorter_than_told(hip, rows, heads, told, parts):
    """Partitions get longer than two tiles only where rows much shorter than
    the bound do not pay for it: captured steps are told the longest that
    rows may become."""
    assert hip._mla_split(rows, heads, told) == parts


def test_mla_heads_of_a_workgroup_as_the_kernel_plans_them():
    """_mla_split counts on the rule of csrc/mla.hip."""
    try:
        from vllm_amd.ops import hip_ops
    except (ImportError, OSError) as e:
        pytest.skip(f"extension not built: {e}")
    seen = set()
    for heads in (1, 16, 32, 33, 64, 65, 72, 100, 128, 129, 160, 256):
        for pairs in (0, 1, 15, 16, 32, 63, 64, 65, 85, 86, 127, 128, 129, 255,
                      256, 257, 4096, 1 << 20):
            n = hip_ops._mla_group_heads(pairs, heads)
            assert n == torch.ops.vllm_amd.mla_group_heads(pairs, heads)
            seen.add(n)
    assert seen == {32, 64, 128}


@pytest.mark.parametrize("rows,kv,span,window,parts", [
    (1, 8, 1000, 0, 8),       # none shorter than 128 keys
    (1, 8, 8192, 0, 32),      # one workgroup a CU ...
    (2, 8, 8192, 0, 16),
    (3, 8, 8192, 0, 22),      # ... two
    (1, 8, 200000, 0, 64),    # the lanes of a wave
    (2, 256, 8192, 0, 4),     # none longer than 2048 keys
    (1, 8, 8192, 97, 1),      # a window's keys
])
def test_decode_parts(hip, rows, kv, span, window, parts):
    assert hip._decode_parts(rows, kv, span, window) == parts


@pytest.mark.parametrize("rows,kv,span,hd,size,parts", [
    (1, 8, 384, 128, 2, 1), (1, 8, 385, 128, 2, 4),    # not worth a merge
    (16, 8, 384, 64, 1, 1), (1, 2, 256, 256, 2, 1), (1, 2, 257, 256, 2, 3),
    (4, 8, 8192, 128, 2, 8), (4, 8, 8192, 128, 1, 16),  # one a CU, two
    (3, 8, 8192, 128, 2, 10), (5, 8, 8192, 128, 2, 6),
    (7, 8, 8192, 128, 2, 4), (9, 8, 8192, 128, 2, 8),   # 224 CUs, 216
    (16, 8, 2000, 128, 2, 2), (17, 8, 2000, 128, 2, 4),
    (16, 8, 8192, 128, 2, 4),     # none longer than 2048 keys
    (1, 28, 8192, 128, 2, 9)])
def test_decode_parts_of_short_and_few_rows(hip, rows, kv, span, hd, size,
                                            parts):
    assert hip._decode_parts(rows, kv, span, 0, hd, size) == parts


@pytest.mark.parametrize("tokens,topk,E,H,form", [
    (64, 8, 64, 7168, 0),      # one streamed tile holds any expert's rows
    (65, 8, 64, 7168, 1),      # no longer
    (767, 8, 256, 7168, 1),
    (95, 2, 8, 4096, 0),       # 8 x 16 tiles leave half the chip idle
    (96, 2, 8, 4096, 1),
    (500, 1, 128, 2048, 0),    # below 4 rows an expert
    (512, 1, 128, 2048, 1),
    (1536, 8, 64, 7168, 2),
    (383, 2, 16, 1024, 0),     # 16 x 4 tiles leave three quarters idle
    (384, 2, 16, 1024, 1),
    (192, 2, 16, 2048, 1),     # 16 x 8 tiles half of it
])
def test_expert_form(hip, tokens, topk, E, H, form):
    """Where rows may meet in few experts the weights are not streamed
    once per 64 of them."""
    I = 64
    w13 = torch.empty(E, 2 * I, 1).expand(E, 2 * I, H)
    w2 = torch.empty(E, H, 1).expand(E, H, I)
    rows = (64, 128, 256)[form]
    hip._C.moe_tile_rows = lambda f: (64, 128, 256)[f]
    hip.fused_moe_hip(torch.empty(tokens, H, dtype=torch.bfloat16), w13, w2,
                      torch.empty(tokens, topk),
                      torch.zeros(tokens, topk, dtype=torch.int32))
    gemms = hip._C.args("moe_gemm")
    assert [a[8] for a in gemms] == [form, form]
    assert hip._C.args("moe_align")[0][2] == rows


def test_runner_tells_lengths(monkeypatch):
    """The runner's mixed steps say how long their decode rows are, and
    how long their prompts' contexts."""
    from vllm_amd.entrypoints.llm import LLM
    from vllm_amd.layers import attention
    from vllm_amd.sampling_params import SamplingParams

    real, seen = attention.ops, []

    def spy(q, kv, bt, qsl, sl, scale, **kw):
        meta = attention.get_forward_context().attn_metadata
        nd = meta.num_decodes
        if 0 < nd < len(sl):
            assert kw["max_decode_len"] == int(sl[:nd].max())
            assert meta.max_prompt_len == int(sl[nd:].max())
            seen.append(kw["max_decode_len"] < kw["max_seq_len"])
        return real.attention_unified(q, kv, bt, qsl, sl, scale, **kw)

    monkeypatch.setattr(attention, "ops", types.SimpleNamespace(
        rope_and_cache=real.rope_and_cache,
        reshape_and_cache=real.reshape_and_cache, attention_unified=spy))
    llm = LLM(model="tiny-llama", dtype="fp32", device="cpu", block_size=16,
              num_gpu_blocks=64, max_model_len=256,
              max_num_batched_tokens=32, max_num_seqs=4)
    llm.generate([[5, 6, 7], list(range(3, 103))],
                 SamplingParams(temperature=0.0, max_tokens=8,
                                ignore_eos=True))
    llm.shutdown()
    assert any(seen)


def _mla_prompts(hip, monkeypatch, decodes, prompts, H=128, **kw):
    """The arguments of the per-head prompt kernel for 400-token prompts
    beside decode rows of 8192 keys."""
    n, t = decodes + prompts, decodes + prompts * 400
    q = torch.empty(t, H, 192, dtype=torch.bfloat16)
    monkeypatch.setattr(hip, "mla_attention",
                        lambda q, *a, **k: torch.empty_like(q))
    monkeypatch.setattr(hip, "head_matmul", lambda x, w: torch.empty(
        x.shape[0], x.shape[1], w.shape[2], dtype=x.dtype))
    hip._C.calls.clear()
    hip.mla_heads(
        q[..., :128], q[..., 128:],
        torch.empty(H, 128, 512, dtype=torch.bfloat16),
        torch.empty(H, 512, 128, dtype=torch.bfloat16),
        torch.empty(1, 64, 576, dtype=torch.bfloat16),
        torch.zeros(n, 1, dtype=torch.int32), _lens(*range(n + 1)),
        _lens(*[400] * n), 0.07, num_decodes=decodes, max_query_len=400,
        max_seq_len=8192 if decodes else 400, **kw)
    (a,) = hip._C.args("mla_prompt_attention")
    return a[12], a[13].numel()   # S, scratch


def test_mla_prompt_scratch_ignores_decodes(hip, monkeypatch):
    """Prompts' scratch is sized by the prompts' own contexts."""
    alone = _mla_prompts(hip, monkeypatch, 0, 20)
    beside = _mla_prompts(hip, monkeypatch, 1, 20, max_decode_len=8192,
                          max_prompt_len=400)
    assert alone == beside == (400, 20 * 400 * (64 + 128 * 256))


def test_mla_prompt_heads_at_a_time(hip, monkeypatch):
    """Heads that do not fit at once go in multiples of eight, one per
    XCD, while eight fit."""
    S, numel = _mla_prompts(hip, monkeypatch, 1, 60)
    per = 60 * S
    heads = (numel // per - 64) // 256
    assert numel == per * (64 + heads * 256) and 1 <= heads < 8
    monkeypatch.setattr(hip, "_MLA_PROMPT_SCRATCH", 13 * 60 * S * 512)
    _, numel = _mla_prompts(hip, monkeypatch, 1, 60)
    assert (numel // per - 64) // 256 == 8


def _odd(*shape):
    """A contiguous bf16 tensor that begins 2 B past a 16 B boundary."""
    n = 1
    for x in shape:
        n *= x
    flat = torch.empty(n + 8, dtype=torch.bfloat16)
    at = next(i for i in range(8)
              if flat[i:].data_ptr() % 16 == 2)
    return flat[at:at + n].view(shape)


def test_odd_places_take_plain_loads(hip, monkeypatch):
    """Operands that do not begin on 16 B never reach a kernel that fills
    LDS from them directly."""
    bf, H, I, E = torch.bfloat16, 128, 64, 2
    hip._C.moe_tile_rows = lambda f: (64, 128, 256)[f]
    weights = (torch.empty(E, 2 * I, H, dtype=bf),
               torch.empty(E, H, I, dtype=bf))
    for x, w13, w2, form in (
            (torch.empty(600, H, dtype=bf), *weights, 2),
            (_odd(600, H), *weights, 0),
            (torch.empty(600, H, dtype=bf), _odd(E, 2 * I, H), weights[1],
             0)):
        hip._C.calls.clear()
        hip.fused_moe_hip(x, w13, w2, torch.empty(600, 1),
                          torch.zeros(600, 1, dtype=torch.int32))
        assert [a[8] for a in hip._C.args("moe_gemm")] == [form, form]

    hip._C.calls.clear()
    hip.head_matmul(torch.randn(3, 2, 128).to(bf), _odd(2, 128, 128).zero_())
    assert not hip._C.calls

    q = torch.empty(400, 128, 192, dtype=bf)[..., :128]
    w_uk = torch.empty(128, 128, 512, dtype=bf)
    w_uv = torch.empty(128, 512, 128, dtype=bf)
    cache = torch.empty(1, 64, 576, dtype=bf)
    args = (1, 0.07, 0, 400, 400)
    assert hip._mla_prompt_heads(q, w_uk, w_uv, cache, *args) == 128
    for odd in ((_odd(128, 128, 512), w_uv, cache),
                (w_uk, _odd(128, 512, 128), cache),
                (w_uk, w_uv, _odd(1, 64, 576))):
        assert hip._mla_prompt_heads(q, *odd, *args) == 0
    one = torch.ones(1, dtype=torch.int32)
    hip.mla_attention(torch.zeros(1, 4, 512, dtype=bf),
                      torch.zeros(1, 4, 64, dtype=bf),
                      _odd(1, 64, 576).zero_(), one[None] * 0,
                      _lens(0, 1), one, 0.07, num_decodes=1, max_seq_len=1)
    assert not hip._C.calls


@pytest.mark.parametrize("rows,keys,new,heads,hd,mixed", [
    (96, 4000, 1000, 32, 128, True),
    (8, 1000, 2000, 32, 128, True),
    (1, 1000, 8191, 32, 128, False),     # nothing to run beside
    (256, 300, 500, 32, 128, True),
    (256, 128, 500, 32, 128, False),     # a wave a row
    (512, 300, 500, 32, 128, False),     # a wave a row
    (160, 128, 500, 32, 64, True),
    (8, 1000, 200, 72, 128, False),      # nine heads a KV head
    (8, 1000, 200, 32, 256, False),
    (8, 1000, 2000, 32, 64, True),
])
def test_rows_beside_portions(hip, rows, keys, new, heads, hd, mixed):
    q = torch.empty(rows + new, heads, hd, dtype=torch.bfloat16)
    kv = torch.empty(2, 1, 8, 64, hd, dtype=torch.bfloat16)
    hip.attention_unified(
        q, kv, torch.zeros(rows + 1, 1, dtype=torch.int32),
        _lens(*range(rows + 2)), _lens(*[keys] * rows, new), 0.1,
        num_decodes=rows, max_seq_len=max(keys, new), max_query_len=new,
        max_decode_len=keys)
    names = [n for n, _ in hip._C.calls]
    assert names == (["mixed_attention"] if mixed else
                     ["paged_decode_attention", "prefill_attention"])


@pytest.mark.parametrize("rows,keys,past,new,portions,window,fp8,mixed", [
    (64, 2000, 0, 1000, 4, 0, False, True),
    (64, 2000, 4000, 1000, 4, 0, False, False),   # tiles of one length
    (64, 2000, 4000, 1000, 1, 0, False, True),    # of one portion
    (64, 8000, 4000, 1000, 4, 0, False, True),    # their past is not known
    (512, 2000, 4000, 1000, 4, 0, False, True),   # as much to read
    (2, 2000, 0, 2000, 1, 0, False, True),
    (2, 2000, 0, 2000, 1, 0, True, False),        # half the bytes
    (3, 8000, 0, 4000, 1, 0, False, True),
    (3, 8000, 0, 4000, 1, 128, False, False),     # the keys of a window
])
def test_rows_beside_portions_by_what_they_read(hip, rows, keys, past, new,
                                                portions, window, fp8, mixed):
    q = torch.empty(rows + new * portions, 32, 128, dtype=torch.bfloat16)
    kv = torch.empty(2, 1, 8, 64, 128, dtype=torch.bfloat16)
    if fp8:
        kv = kv.to(torch.float8_e4m3fn)
    lens = [keys] * rows + [past + new] * portions
    starts = torch.tensor([0] + [1] * rows + [new] * portions).cumsum(0)
    hip.attention_unified(
        q, kv, torch.zeros(len(lens), 1, dtype=torch.int32),
        starts.to(torch.int32), _lens(*lens), 0.1, num_decodes=rows,
        max_seq_len=max(lens), max_query_len=new, max_decode_len=keys,
        sliding_window=window)
    names = [n for n, _ in hip._C.calls]
    assert names == (["mixed_attention"] if mixed else
                     ["paged_decode_attention", "prefill_attention"])


def test_wave_rows_as_the_kernel_plans_them():
    try:
        from vllm_amd.ops import hip_ops
    except (ImportError, OSError) as e:
        pytest.skip(f"extension not built: {e}")
    for units in (1, 1023, 1024, 1535, 1536, 4095, 4096):
        for hd in (64, 128, 256):
            for parts in (1, 2):
                for span in (1, 128, 129, 512, 513):
                    assert hip_ops._decode_waves(
                        units, hd, parts, span) == hip_ops._C.decode_waves(
                            units, hd, parts, span)
