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
    ([4100, 1030], 16, 2, 256, 0, torch.float16, None),   # merged in two runs
    ([2176 - 7 * i for i in range(256)], 8, 2, 128, 0, torch.bfloat16, None),
    # More counters than lines, and than a stream's set holds.
    ([2100 + i if i % 9 == 0 else i % 150 for i in range(300)], 8, 4, 64, 0,
     torch.bfloat16, None),
    ([2500 if i % 65 == 0 else 1 + i % 70 for i in range(520)], 32, 32, 64, 0,
     torch.float16, None),
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


# Rows at the ends of what one partition takes in one, two and three steps of
# its waves, and past it.
@pytest.mark.parametrize("hd,cache", [(64, None), (128, None), (256, None),
                                      (128, torch.float8_e4m3fn)])
@pytest.mark.parametrize("told", [129, 256, 257, 384, 385])
def test_short_rows(hd, cache, told):
    from vllm_amd.ops import hip_ops
    ctx = [told, 1, 128, 129, min(told, 256), 64, 0]
    q, kv, table, qsl, lens = _rows(ctx, 8, 2, hd, torch.bfloat16,
                                    cache or torch.bfloat16)
    out = hip_ops.attention_unified(
        q, kv, table, qsl, lens, hd ** -0.5, num_decodes=len(ctx),
        max_seq_len=told)
    assert (out[-1] == 0).all()
    n = len(ctx) - 1
    expect = ref.attention_unified(q[:n].float(), kv.float(), table[:n],
                                   qsl[:n + 1], lens[:n], hd ** -0.5,
                                   num_decodes=n)
    # The output's own rounding, as above.
    torch.testing.assert_close(out[:n].float(), expect, rtol=2.0 ** -8,
                               atol=2.0 ** -9)


# A key's halves lie on neighbouring lanes where its row has 128 B or more:
# every row size, with all of the columns that a group may have and with one.
@pytest.mark.parametrize("group", [1, 8])
@pytest.mark.parametrize("hd", [64, 128, 256])
@pytest.mark.parametrize("cache", [None, torch.float8_e4m3fn])
@pytest.mark.parametrize("n", [5, 600])   # rows in parts, and a wave each
def test_key_rows_by_halves(group, hd, cache, n):
    from vllm_amd.ops import hip_ops
    ctx = [(1, 2, 31, 33, 100)[i % 5] for i in range(n)]
    if n == 5:
        ctx[2:] = [700, 65, 1999]
    q, kv, table, qsl, lens = _rows(ctx, 2 * group, 2, hd, torch.bfloat16,
                                    cache or torch.bfloat16)
    out = hip_ops.attention_unified(
        q, kv, table, qsl, lens, hd ** -0.5, num_decodes=n,
        max_seq_len=max(ctx))
    expect = ref.attention_unified(q.float(), kv.float(), table, qsl, lens,
                                   hd ** -0.5, num_decodes=n)
    # The output's own rounding, as above.
    torch.testing.assert_close(out.float(), expect, rtol=2.0 ** -8,
                               atol=2.0 ** -9)


@torch.inference_mode()   # as the runner captures
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


def test_more_streams_than_sets():
    """More streams than have counters of their own, and one that is not
    torch's."""
    import ctypes
    from vllm_amd.ops import hip_ops
    ctx = [1500, 200, 0, 3000, 129]
    q, kv, table, qsl, lens = _rows(ctx, 32, 8, 128, torch.bfloat16,
                                    torch.bfloat16)

    def call():
        return hip_ops.attention_unified(
            q, kv, table, qsl, lens, 0.09, num_decodes=len(ctx),
            max_seq_len=4096)

    expect = call()
    hip = ctypes.CDLL("libamdhip64.so")
    handle = ctypes.c_void_p()
    assert hip.hipStreamCreate(ctypes.byref(handle)) == 0
    streams = [torch.cuda.Stream() for _ in range(34)]
    streams += [torch.cuda.ExternalStream(handle.value)]
    torch.cuda.synchronize()
    outs = []
    for _ in range(3):
        for s in streams:
            with torch.cuda.stream(s):
                outs.append(call())
    torch.cuda.synchronize()
    assert hip.hipStreamDestroy(handle) == 0
    for o in outs:
        assert torch.equal(o, expect)


def _nodes(graph):
    import ctypes
    hip = ctypes.CDLL("libamdhip64.so")
    n = ctypes.c_size_t(0)
    assert hip.hipGraphGetNodes(ctypes.c_void_p(graph.raw_cuda_graph()),
                                None, ctypes.byref(n)) == 0
    return n.value


@torch.inference_mode()
def test_captured_launches_share_counters():
    """A graph clears counters once for each of its streams, not once for
    each launch; graphs of one pool, captured one after the other without an
    eager call between them, do not disturb each other."""
    from vllm_amd.ops import hip_ops
    ctx = [1500, 200, 0, 3000, 129]
    q, kv, table, qsl, lens = _rows(ctx, 32, 8, 128, torch.bfloat16,
                                    torch.bfloat16)
    x = torch.randn(33, 7168, device="cuda").bfloat16()
    w = torch.randn(2112, 7168, device="cuda").bfloat16() * 0.01

    def call():
        return (hip_ops.attention_unified(
            q, kv, table, qsl, lens, 0.09, num_decodes=len(ctx),
            max_seq_len=4096), hip_ops.linear(x, w))

    expect = call()
    main, side = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    graphs, outs, pool = [], [], None
    for _ in range(3):
        graph = torch.cuda.CUDAGraph(keep_graph=True)
        with torch.cuda.graph(graph, stream=main, pool=pool):
            out = [call(), call()]
            side.wait_stream(main)
            with torch.cuda.stream(side):
                out.append(call())
            out.append(call())
            main.wait_stream(side)
        assert _nodes(graph) == 8 + 2   # kernels and a fill for each stream
        graph.instantiate()
        pool = graph.pool()
        graphs.append(graph)
        outs.append(out)
    for i in (0, 1, 2, 0, 2, 1):
        for o in outs[i]:
            for t in o:
                t.zero_()
        torch.cuda.synchronize()
        graphs[i].replay()
        eager = call()
        torch.cuda.synchronize()
        for o in outs[i] + [eager]:
            for t, e in zip(o, expect):
                assert torch.equal(t, e)


# More tiles than rows and fewer, one of each; a portion shorter than a
# tile, after cached tokens; heads in groups of 1, 7 and 8; rows in one and
# in several partitions; a window; an fp8 cache; a negative scale.
MIXED = [
    ([1000], [70], [0], 32, 8, 128, 0, torch.bfloat16, None, 0.09),
    ([0, 1, 129, 3000], [1, 300], [5, 64], 14, 2, 128, 0, torch.float16,
     None, 0.09),
    ([500] * 40, [2], [1], 8, 8, 64, 0, torch.bfloat16, None, -0.1),
    ([2000, 60], [513, 40, 129], [100, 0, 700], 16, 2, 128, 200,
     torch.bfloat16, None, 0.09),
    ([700, 1500, 64], [200], [31], 8, 2, 128, 0, torch.bfloat16,
     torch.float8_e4m3fn, 0.09),
    ([300] * 37, [1000, 3, 129], [0, 900, 7], 8, 2, 64, 0, torch.bfloat16,
     None, 0.1),
]
NAMES = "rows,new,past,hq,hkv,hd,window,dtype,cache,scale"


def _step(rows, new, past, hq, hkv, hd, dtype, cache):
    ctx = rows + [n + p for n, p in zip(new, past)]
    _, kv, table, _, lens = _rows(ctx, hq, hkv, hd, dtype, cache or dtype)
    g = torch.Generator(device="cuda")
    g.manual_seed(sum(ctx))
    q = torch.randn(len(rows) + sum(new), hq, hd, device="cuda",
                    generator=g).to(dtype)
    qsl = torch.tensor([0] + [1] * len(rows) + new, device="cuda").cumsum(
        0).to(torch.int32)
    return q, kv, table, qsl, lens


def _joint(q, kv, table, qsl, lens, rows, new, window, scale):
    """mixed_attention, whatever the rule says of the sizes."""
    from vllm_amd.ops import hip_ops
    n, hq, hd = len(rows), q.shape[1], q.shape[2]
    parts = hip_ops._decode_parts(n, kv.shape[2], max(rows), window)
    tmp = [q.new_empty(n, hq, parts, w, dtype=torch.float32)
           if parts > 1 else q.new_empty(0, dtype=torch.float32)
           for w in (hd, 2)]
    out = torch.empty_like(q)
    hip_ops._C.mixed_attention(out, q, kv, table, qsl, lens, scale, n,
                               max(rows), max(new), window, *tmp)
    return out


@pytest.mark.parametrize(NAMES, MIXED)
def test_mixed_exact(rows, new, past, hq, hkv, hd, window, dtype, cache,
                     scale):
    """The joint launch against fp32: weights of portions and the result are
    rounded to p bits (p = 8, 11), each off by 2^-p at most: 2^-p of the same
    sums over |v|, and of the result once for their own sum and once for
    itself."""
    q, kv, table, qsl, lens = _step(rows, new, past, hq, hkv, hd, dtype,
                                    cache)
    out = _joint(q, kv, table, qsl, lens, rows, new, window, scale).float()
    live = [i for i, c in enumerate(lens.tolist()) if c > 0]
    starts = qsl.tolist()
    take = torch.cat([torch.arange(starts[i], starts[i + 1]) for i in live])
    lq = torch.tensor([0] + [starts[i + 1] - starts[i] for i in live],
                      dtype=torch.int32, device="cuda").cumsum(0).int()

    def exact(values):
        return ref.attention_unified(
            q[take].float(), values, table[live], lq, lens[live], scale,
            num_decodes=len([i for i in live if i < len(rows)]),
            sliding_window=window)

    wide = kv.float()
    expect, mag = exact(wide), exact(torch.stack([wide[0], wide[1].abs()]))
    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    bound = eps * (mag + 2 * expect.abs()) + 2.0 ** -16
    assert ((out[take] - expect).abs() <= bound).all()
    dead = torch.ones(len(q), dtype=torch.bool)
    dead[take] = False
    assert (out[dead.cuda()] == 0).all()


@torch.inference_mode()   # as the runner captures
def test_mixed_replays():
    case = MIXED[1]
    q, kv, table, qsl, lens = _step(*case[:6], case[7], case[8])

    def call():
        return _joint(q, kv, table, qsl, lens, case[0], case[1], case[6],
                      case[9])

    expect = call()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    for _ in range(4):
        out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        beside = call()
        torch.cuda.synchronize()
        assert torch.equal(out, expect)
        assert torch.equal(beside, expect)


@pytest.mark.parametrize(NAMES, MIXED)
def test_mixed(rows, new, past, hq, hkv, hd, window, dtype, cache, scale):
    """Rows and portions in one launch against each in its own: the same
    work by the same code, so the same but for the order in which the
    compiler adds (a unit of fp32 sums, the result's rounding)."""
    from vllm_amd.ops import hip_ops
    ctx = rows + [n + p for n, p in zip(new, past)]
    q, kv, table, _, lens = _rows(ctx, hq, hkv, hd, dtype, cache or dtype)
    q = torch.randn(len(rows) + sum(new), hq, hd, device="cuda").to(dtype)
    qsl = torch.tensor([0] + [1] * len(rows) + new, device="cuda").cumsum(
        0).to(torch.int32)
    n = len(rows)
    none = q.new_empty(0, dtype=torch.float32)
    parts = hip_ops._decode_parts(n, hkv, max(rows), window)
    tmp = (torch.empty(n, hq, parts, hd, device="cuda"),
           torch.empty(n, hq, parts, 2, device="cuda")) if parts > 1 else (
               none, none)
    one, two = torch.empty_like(q), torch.empty_like(q)
    ops = hip_ops._C
    ops.mixed_attention(one, q, kv, table, qsl, lens, scale, n, max(rows),
                        max(new), window, *tmp)
    ops.paged_decode_attention(two[:n], q[:n], kv, table, lens, scale,
                               max(rows), window, *tmp)
    ops.prefill_attention(two, q, kv, table, qsl, lens, scale, n, max(new),
                          window)
    tol = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    torch.testing.assert_close(one.float(), two.float(), rtol=tol,
                               atol=1e-6)
