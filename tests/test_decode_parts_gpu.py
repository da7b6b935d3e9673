"""Decode rows whose keys are split over workgroups: the last of them to
arrive merges (csrc/attention_decode.hip, arrivals.h)."""

import pytest
import torch

from vllm_amd.ops import _torch_ref as ref

pytestmark = pytest.mark.gpu


def _rows(ctx, hq, hkv, hd, dtype, cache_dtype):
    g = torch.Generator(device="cuda")
    g.manual_seed(sum(ctx) + hq + hd)
    need = [-(-c // 64) for c in ctx]
    width = max(max(need), 1)
    table = torch.zeros(len(ctx), width, dtype=torch.int32, device="cuda")
    at = 1
    for i, n in enumerate(need):
        table[i, :n] = torch.arange(at, at + n)
        at += n
    q = torch.randn(len(ctx), hq, hd, device="cuda", generator=g).to(dtype)
    cache = torch.randn(2, at, hkv, 64, hd, device="cuda",
                        generator=g).to(cache_dtype)
    qsl = torch.arange(len(ctx) + 1, dtype=torch.int32, device="cuda")
    lens = torch.tensor(ctx, dtype=torch.int32, device="cuda")
    return q, cache, table, qsl, lens


# Rows without keys, of one, of some and of all of their partitions; few
# rows (up to 64 partitions) and many; every head width; a window.
@pytest.mark.parametrize("ctx,hq,hkv,hd,window,dtype,cache", [
    ([1000], 32, 8, 128, 0, torch.bfloat16, None),
    ([0, 1, 127, 128, 129, 1023, 4097], 8, 2, 128, 0, torch.float16, None),
    ([8190, 3, 0, 700], 4, 1, 128, 0, torch.bfloat16, torch.float8_e4m3fn),
    ([2000, 31, 640], 3, 1, 64, 0, torch.bfloat16, None),
    ([900, 64, 1500], 16, 2, 256, 0, torch.bfloat16, None),
    ([3000, 100, 500], 8, 8, 128, 300, torch.bfloat16, None),
    ([2176 - 7 * i for i in range(256)], 8, 2, 128, 0, torch.bfloat16, None),
])
def test_merge(ctx, hq, hkv, hd, window, dtype, cache):
    from vllm_amd.ops import hip_ops
    q, kv, table, qsl, lens = _rows(ctx, hq, hkv, hd, dtype, cache or dtype)
    out = hip_ops.attention_unified(
        q, kv, table, qsl, lens, hd ** -0.5, num_decodes=len(ctx),
        max_seq_len=max(ctx), sliding_window=window)
    live = [i for i, c in enumerate(ctx) if c > 0]
    for i in set(range(len(ctx))) - set(live):
        assert (out[i] == 0).all()
    # Against fp32 on the same cached values: weights carried at 16 bits
    # more than the type, so the result's own rounding (2^-8 or 2^-11) and
    # the like of it in the reference, which rounds its weights.
    expect = ref.attention_unified(
        q[live].float(), kv.float() if cache is None else
        kv.to(torch.float32), table[live], torch.arange(
            len(live) + 1, dtype=torch.int32, device="cuda"), lens[live],
        hd ** -0.5, num_decodes=len(live), sliding_window=window)
    tol = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    torch.testing.assert_close(out[live].float(), expect, rtol=tol,
                               atol=2.0 ** -9)


def test_replays_and_streams():
    """Counters are left zero: by replays, by eager calls beside them and by
    calls on other streams."""
    from vllm_amd.ops import hip_ops
    ctx = [1500, 200, 0, 3000, 129]
    q, kv, table, qsl, lens = _rows(ctx, 32, 8, 128, torch.bfloat16,
                                    torch.bfloat16)

    def call():
        return hip_ops.attention_unified(
            q, kv, table, qsl, lens, 0.09, num_decodes=len(ctx),
            max_seq_len=4096)

    streams = [torch.cuda.Stream() for _ in range(3)]
    expect = call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=streams[0]):
        out = call()
    for _ in range(4):
        out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        beside = []
        for s in streams:
            with torch.cuda.stream(s):
                beside.append(call())
        torch.cuda.synchronize()
        assert torch.equal(out, expect)
        for o in beside:
            assert torch.equal(o, expect)
