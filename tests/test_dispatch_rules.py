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


def test_runner_tells_decode_lengths(monkeypatch):
    """The runner's steps say how long their decode rows are, with and
    without prompts beside them."""
    from vllm_amd.entrypoints.llm import LLM
    from vllm_amd.layers import attention
    from vllm_amd.sampling_params import SamplingParams

    real, seen = attention.ops, []

    def spy(q, kv, bt, qsl, sl, scale, **kw):
        nd = kw["num_decodes"]
        if 0 < nd < len(sl):
            seen.append((kw["max_decode_len"], int(sl[:nd].max()),
                         kw["max_seq_len"]))
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
    assert all(told == real_max for told, real_max, _ in seen)
    assert any(told < longest for told, _, longest in seen)
