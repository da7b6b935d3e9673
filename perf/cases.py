"""The serving work that this framework is timed on.

Three kinds of pass, each one engine step's worth of work on one GPU:

"stack"    a dense decoder with grouped-query attention: the model's
           forward under a forward context and the logits of the rows
           that sample, exactly as the runner calls it. Four layers of
           a configured model at full width (one stage of its 8-way
           pipeline split, with embedding and head): every layer does
           the same work, so more of them only repeat it. A step holds
           decode rows, prompt portions, or both.
"experts"  the routed experts of one layer, called with the routing a
           router gave (given, because a tie in a router would make two
           correct implementations disagree).
"latent"   one attention block with compressed keys and values (MLA):
           projections, cache write, attention, output projection.

Contexts and prompt lengths are spread evenly between the stated ends
and shuffled by a fixed rule, so a case is the same amount of work
whatever the seed; the seed makes weights, tokens, cached keys and
values, the physical order of the cache blocks and the routing.
"""

import dataclasses
import math

import torch

from vllm_amd.config import ModelConfig, get_model_spec
from vllm_amd.layers.fused_moe import FusedMoE
from vllm_amd.models.deepseek import DeepseekMLAAttention
from vllm_amd.models.registry import get_model_class
from vllm_amd.worker.forward_context import (
    AttentionMetadata,
    ForwardContext,
    set_forward_context,
)

BLOCK = 64    # tokens per cache block, the framework's default
LAYERS = 4
DEV = "cuda"


def _stack(name, model="llama-3-8b", decodes=0, ctx_lo=0, ctx_hi=0,
           prompts=0, new_lo=0, new_hi=0, past_lo=0, past_hi=0,
           kv="bf16"):
    """decodes rows with contexts ctx_lo..ctx_hi (the new token
    included), then prompts portions of new_lo..new_hi tokens, each
    after past_lo..past_hi tokens that are cached already."""
    case = dict(kind="stack", model=model, decodes=decodes, ctx_lo=ctx_lo,
                ctx_hi=ctx_hi, prompts=prompts, new_lo=new_lo,
                new_hi=new_hi, past_lo=past_lo, past_hi=past_hi, kv=kv)
    return dict(name=name, **case) if name else case


def _latent(name, **kw):
    case = dict(_stack(None, model="deepseek-v3-lite", **kw), kind="latent")
    return dict(name=name, **case) if name else case


def _experts(name, model, tokens, skew):
    case = dict(kind="experts", model=model, tokens=tokens, skew=skew)
    return dict(name=name, **case) if name else case


def listed():
    return [
        # One user in a chat: nothing to batch, every launch is waited for.
        _stack("chat_1", decodes=1, ctx_lo=1000, ctx_hi=1000),
        # The latency suite's shape: batch 8, 32 in, 128 out.
        _stack("latency_8", decodes=8, ctx_lo=33, ctx_hi=160),
        # A busy server on the random 128/2048 serving shape.
        _stack("serve_256", decodes=256, ctx_lo=129, ctx_hi=2176),
        # bench.py's workload: 1024 running sequences, 128-token prompts.
        _stack("bench_1024", decodes=1024, ctx_lo=129, ctx_hi=176),
        # Long contexts on the half-size cache.
        _stack("long_64_fp8kv", decodes=64, ctx_lo=4096, ctx_hi=8192,
               kv="fp8"),
        # One prompt as long as the model takes.
        _stack("prompt_8k", prompts=1, new_lo=8192, new_hi=8192),
        # A burst of short prompts of uneven length (mean 128).
        _stack("prompts_64", prompts=64, new_lo=33, new_hi=223),
        # Chunked prefill: portions of prompts ride with decode rows.
        _stack("mixed", decodes=96, ctx_lo=100, ctx_hi=4000, prompts=3,
               new_lo=400, new_hi=1001, past_lo=0, past_hi=4096),
        # Routed experts, few large ones, a decode batch.
        _experts("experts_decode", "mixtral-8x7b", 48, 0.5),
        # Routed experts, many small ones, a prefill step.
        _experts("experts_prompt", "deepseek-v3-lite", 4096, 0.5),
        # Compressed-cache decode on a busy server.
        _latent("latent_decode", decodes=128, ctx_lo=129, ctx_hi=2176),
        # Compressed-cache prefill of a few uneven prompts.
        _latent("latent_prompts", prompts=3, new_lo=300, new_hi=2301),
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(
        rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    kind = rng.choice(("decode", "decode", "prompt", "mixed", "experts",
                       "latent"))
    model = rng.choice(("llama-3-8b", "llama-3-8b", "qwen2.5-7b",
                        "mistral-7b", "yi-6b"))
    limit = min(8192, get_model_spec(model).max_position_embeddings)
    if kind == "decode":
        n = _log(rng, 1, 1024)
        top = max(64, min(limit, 600000 // n))
        hi = _log(rng, 33, top)
        # The fp8 cache is for long contexts.
        kv = rng.choice(("bf16", "fp8")) if hi >= 1024 else "bf16"
        lo = rng.randint(512 if kv == "fp8" else 1, hi)
        return _stack(None, model=model, decodes=n, ctx_lo=lo, ctx_hi=hi,
                      kv=kv)
    if kind in ("prompt", "mixed"):
        n = _log(rng, 1, 48)
        hi = _log(rng, 17, min(limit, 8192 // n))
        past = rng.choice((0, _log(rng, 1, 4096)))
        past = max(0, min(past, limit - hi))
        dec = _log(rng, 1, 256) if kind == "mixed" else 0
        dhi = _log(rng, 33, min(4096, limit)) if dec else 0
        return _stack(None, model=model, decodes=dec,
                      ctx_lo=rng.randint(1, dhi) if dec else 0, ctx_hi=dhi,
                      prompts=n, new_lo=rng.randint(2, hi), new_hi=hi,
                      past_lo=rng.randint(0, past), past_hi=past)
    if kind == "experts":
        model = rng.choice(("mixtral-8x7b", "deepseek-v3-lite",
                            "qwen3-30b-a3b"))
        return _experts(None, model, _log(rng, 1, 4096),
                        rng.choice((0.0, 0.5, 1.0)))
    if rng.random() < 0.6:
        n = _log(rng, 1, 256)
        hi = _log(rng, 33, min(8192, 300000 // n))
        return _latent(None, decodes=n, ctx_lo=rng.randint(1, hi), ctx_hi=hi)
    n = rng.randint(1, 6)
    hi = _log(rng, 17, 3000 // n)
    return _latent(None, prompts=n, new_lo=rng.randint(2, hi), new_hi=hi,
                   past_lo=0, past_hi=rng.choice((0, 512)))


# ------------------------------------------------------------- lengths

def _spread(n, lo, hi):
    if n == 1:
        return [hi]
    vals = [lo + (hi - lo) * i // (n - 1) for i in range(n)]
    step = next(s for s in range(max(1, int(n * 0.618)), 2 * n + 2)
                if math.gcd(s, n) == 1)
    return [vals[i * step % n] for i in range(n)]


def _lengths(case):
    """[(new tokens, context with them)] per request, decodes first."""
    rows = [(1, c) for c in _spread(case["decodes"], case["ctx_lo"],
                                    case["ctx_hi"])] if case["decodes"] \
        else []
    if case["prompts"]:
        new = _spread(case["prompts"], case["new_lo"], case["new_hi"])
        past = _spread(case["prompts"], case["past_lo"], case["past_hi"])
        rows += [(n, n + p) for n, p in zip(new, past)]
    return rows


def _seen(case, window=0):
    """Sum over the new tokens of the keys each of them attends, and
    the cached positions that must be read at all."""
    pairs = keys = 0
    for new, ctx in _lengths(case):
        first = ctx - new
        if window and ctx > window:
            full = max(0, min(window, ctx) - first)
            pairs += sum(range(first + 1, first + full + 1))
            pairs += window * (new - full)
            keys += ctx - max(0, first + 1 - window)
        else:
            pairs += new * first + new * (new + 1) // 2
            keys += ctx
    return pairs, keys


# ------------------------------------------------------------- inputs

def _gen(seed, what):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 1000003 + what)
    return g


def _fill(t, bound, g):
    """Uniform in +-bound, in place."""
    return t.uniform_(-bound, bound, generator=g)


def _fill_module(module, g):
    """Dummy-weight scales: matrices uniform within 1/sqrt(fan_in), norm
    gains near 1, biases small."""
    for name, p in module.named_parameters():
        if p.dim() == 1:
            norm = "norm" in name
            _fill(p.data, 0.05 if norm else 1e-3, g)
            if norm:
                p.data.add_(1.0)
        else:
            _fill(p.data, p.shape[-1] ** -0.5, g)


def _meta(case, seed):
    rows = _lengths(case)
    g = _gen(seed, 1)
    need = [-(-ctx // BLOCK) for _, ctx in rows]
    order = torch.randperm(sum(need), generator=g, device=DEV)
    order = order.to(torch.int32).split(need)
    table = torch.nn.utils.rnn.pad_sequence(order, batch_first=True)
    starts = [0]
    for new, _ in rows:
        starts.append(starts[-1] + new)
    lens = torch.tensor([c for _, c in rows], dtype=torch.int32, device=DEV)
    qsl = torch.tensor(starts, dtype=torch.int32, device=DEV)
    total = starts[-1]
    req = torch.repeat_interleave(
        torch.arange(len(rows), device=DEV),
        torch.tensor([n for n, _ in rows], device=DEV), output_size=total)
    pos = (torch.arange(total, device=DEV) - qsl.long()[req]
           + (lens - (qsl[1:] - qsl[:-1])).long()[req])
    slots = table[req, pos // BLOCK].long() * BLOCK + pos % BLOCK
    meta = AttentionMetadata(
        query_start_loc=qsl, seq_lens=lens, block_table=table.contiguous(),
        slot_mapping=slots, num_reqs=len(rows), num_actual_tokens=total,
        max_query_len=max(n for n, _ in rows),
        max_seq_len=max(c for _, c in rows), num_decodes=case["decodes"])
    return meta, pos, sum(need)


def _spec(case):
    spec = get_model_spec(case["model"])
    if case["kind"] == "stack":
        spec = dataclasses.replace(spec, num_layers=LAYERS)
    return spec


def _cached(shape, bound, g, kv):
    t = _fill(torch.empty(shape, dtype=torch.bfloat16, device=DEV), bound, g)
    if kv == "bf16":
        return t
    out = torch.empty(shape, dtype=torch.float8_e4m3fn, device=DEV)
    return out.copy_(t)


def prepare(case, seed):
    with torch.inference_mode():
        return _PREPARE[case["kind"]](case, seed)


def _prepare_stack(case, seed):
    spec = _spec(case)
    config = ModelConfig(model=case["model"], dtype="bf16", spec=spec,
                         max_model_len=8192)
    with torch.device(DEV):
        model = get_model_class(spec.architecture)(config).eval()
    g = _gen(seed, 2)
    _fill_module(model, g)
    # A residual stream a few times each layer's contribution to it.
    _fill(model.model.embed_tokens.weight.data, 0.4, g)
    qk = (spec.num_heads + spec.num_kv_heads) * spec.head_dim
    for layer in model.model.layers:
        # Attention scores of a few units, as trained models have them,
        # rather than a nearly flat softmax.
        layer.self_attn.qkv_proj.weight.data[:qk].mul_(2.5)
    meta, pos, blocks = _meta(case, seed)
    shape = (blocks, spec.num_kv_heads, BLOCK, spec.head_dim)
    caches = []
    for _ in range(LAYERS):
        cache = torch.empty((2,) + shape, device=DEV, dtype=(
            torch.bfloat16 if case["kv"] == "bf16" else
            torch.float8_e4m3fn))
        # As the projections above make them: uniform inputs of a norm,
        # weights within 2.5 (keys) and 1 (values) over sqrt(fan_in).
        cache[0] = _cached(shape, 2.5, g, case["kv"])
        cache[1] = _cached(shape, 1.0, g, case["kv"])
        caches.append(cache)
    ids = torch.randint(0, spec.vocab_size, (meta.num_actual_tokens,),
                        generator=g, device=DEV)
    last = meta.query_start_loc[1:].long() - 1
    return dict(case=case, model=model, ids=ids, pos=pos, last=last,
                ctx=ForwardContext(attn_metadata=meta, kv_caches=caches))


def _prepare_latent(case, seed):
    spec = _spec(case)
    with torch.device(DEV):
        block = DeepseekMLAAttention(spec, 0, torch.bfloat16, 8192)
    g = _gen(seed, 2)
    _fill_module(block, g)
    block.q_b_proj.weight.data.mul_(6.0)  # scores of a few units
    meta, pos, blocks = _meta(case, seed)
    cache = torch.empty(blocks, BLOCK, spec.kv_lora_rank
                        + spec.qk_rope_head_dim, dtype=torch.bfloat16,
                        device=DEV).normal_(generator=g)
    cache[..., spec.kv_lora_rank:].mul_(0.58)
    hidden = torch.empty(meta.num_actual_tokens, spec.hidden_size,
                         dtype=torch.bfloat16, device=DEV)
    hidden.normal_(generator=g)
    return dict(case=case, block=block, pos=pos, hidden=hidden,
                ctx=ForwardContext(attn_metadata=meta, kv_caches=[cache]))


def _prepare_experts(case, seed):
    spec = _spec(case)
    with torch.device(DEV):
        moe = FusedMoE(spec.num_experts, spec.num_experts_per_tok,
                       spec.hidden_size, spec.moe_intermediate_size,
                       dtype=torch.bfloat16, learned_router=False)
    g = _gen(seed, 2)
    _fill_module(moe, g)
    hidden = torch.empty(case["tokens"], spec.hidden_size,
                         dtype=torch.bfloat16, device=DEV)
    hidden.normal_(generator=g)
    logits = torch.randn(case["tokens"], spec.num_experts, generator=g,
                         device=DEV)
    # Some experts are liked more than others.
    logits += case["skew"] * torch.randn(spec.num_experts, generator=g,
                                         device=DEV)
    w, ids = logits.softmax(-1).topk(spec.num_experts_per_tok, dim=-1)
    return dict(case=case, moe=moe, hidden=hidden,
                w=w / w.sum(-1, keepdim=True), ids=ids.to(torch.int32))


_PREPARE = {"stack": _prepare_stack, "latent": _prepare_latent,
            "experts": _prepare_experts}


# ---------------------------------------------------------------- pass

def _bytes_of(cache):
    return cache if cache.dtype == torch.bfloat16 else cache.view(
        torch.uint8)


def run(s):
    kind = s["case"]["kind"]
    with torch.inference_mode():
        if kind == "experts":
            return {"out": s["moe"].run_experts(s["hidden"], s["w"],
                                                s["ids"])}
        with set_forward_context(s["ctx"]):
            if kind == "latent":
                return {"out": s["block"](s["pos"], s["hidden"]),
                        "cache": s["ctx"].kv_caches[0]}
            hidden = s["model"](s["ids"], s["pos"])
            logits = s["model"].compute_logits(hidden[s["last"]])
        return {"logits": logits, "hidden": hidden,
                "caches": [_bytes_of(c) for c in s["ctx"].kv_caches]}


# ---------------------------------------------------------------- work

def work(case):
    spec = _spec(case)
    if case["kind"] == "experts":
        t, h, i = case["tokens"], spec.hidden_size, spec.moe_intermediate_size
        e, k = spec.num_experts, spec.num_experts_per_tok
        touched = e * (1 - (1 - k / e) ** t)
        return {"bytes": touched * 3 * h * i * 2 + 2 * t * h * 2 + t * k * 8,
                "flops": 6.0 * t * k * h * i}
    pairs, keys = _seen(case, spec.sliding_window)
    new = sum(n for n, _ in _lengths(case))
    h, heads = spec.hidden_size, spec.num_heads
    if case["kind"] == "latent":
        lora, rope = spec.kv_lora_rank, spec.qk_rope_head_dim
        nope, vd = spec.qk_nope_head_dim, spec.v_head_dim
        weights = (h * spec.q_lora_rank
                   + spec.q_lora_rank * heads * (nope + rope)
                   + h * (lora + rope) + heads * nope * lora
                   + heads * lora * vd + heads * vd * h)
        # Scores and values in the compressed space, or keys and values
        # of every head expanded first: whichever is less.
        absorbed = pairs * (2 * lora + rope) + new * lora * (nope + vd)
        expanded = pairs * (nope + rope + vd) + keys * lora * (nope + vd)
        weights -= heads * lora * (nope + vd)
        return {"bytes": 2 * (weights + heads * lora * (nope + vd)
                              + 2 * new * h + (keys + new) * (lora + rope)),
                "flops": 2.0 * new * weights
                + 2.0 * heads * min(absorbed, expanded)}
    kvw = 2 * spec.num_kv_heads * spec.head_dim
    qw = heads * spec.head_dim
    layer = (h * (qw + kvw) + qw * h + 3 * h * spec.intermediate_size)
    head = h * spec.vocab_size
    rows = len(_lengths(case))
    size = 2 if case["kv"] == "bf16" else 1
    return {"bytes": 2 * (LAYERS * layer + head + 2 * new * h
                          + rows * spec.vocab_size)
            + LAYERS * (keys + new) * kvw * size,
            "flops": 2.0 * LAYERS * new * layer + 2.0 * rows * head
            + 4.0 * LAYERS * pairs * qw}


def tolerance(case):
    # Up to four times the distance to exact() that was measured: 0.004
    # for the experts (hidden values rounded once between two products),
    # 0.006 to 0.007 for one block with its five projections, 0.007 to
    # 0.012 for four layers whose activations are rounded at every step.
    if case["kind"] == "experts":
        return {"rel": 0.015, "max": 0.2}
    if case["kind"] == "latent":
        return {"rel": 0.025, "max": 0.3}
    return {"rel": 0.03, "max": 0.5, "differ": 0.01}


# --------------------------------------------------------------- exact

def _norm64(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w


def _rotate64(x, pos, theta):
    """Halves of the last dimension turned by pos * theta^(-2i/d)."""
    d = x.shape[-1]
    f = theta ** (-torch.arange(0, d, 2, dtype=torch.float64, device=DEV)
                  / d)
    a = pos.double()[:, None, None] * f
    x1, x2 = x.chunk(2, -1)
    return torch.cat([x1 * a.cos() - x2 * a.sin(),
                      x2 * a.cos() + x1 * a.sin()], -1)


def _attend64(q, k, v, scale, window):
    """q [n, H, D], k [c, H, D], v [c, H, Dv]: the queries are the last
    n positions. Chunked over queries to bound the score matrix."""
    n, c = q.shape[0], k.shape[0]
    kt, vt = k.permute(1, 2, 0).contiguous(), v.transpose(0, 1).contiguous()
    kpos = torch.arange(c, device=DEV)
    out = []
    for at in range(0, n, 512):
        part = q[at:at + 512].transpose(0, 1)
        qpos = c - n + at + torch.arange(part.shape[1], device=DEV)
        hide = kpos[None] > qpos[:, None]
        if window:
            hide |= kpos[None] <= qpos[:, None] - window
        scores = torch.matmul(part, kt).mul_(scale)
        scores.masked_fill_(hide, float("-inf"))
        out.append(torch.matmul(scores.softmax(-1), vt).transpose(0, 1))
    return torch.cat(out)


def exact(case, seed):
    with torch.inference_mode():
        return _EXACT[case["kind"]](prepare(case, seed))


def _exact_experts(s):
    x, moe = s["hidden"].double(), s["moe"]
    out = torch.zeros_like(x)
    for e in range(moe.num_experts):
        t, k = (s["ids"] == e).nonzero(as_tuple=True)
        if len(t):
            gate, up = (x[t] @ moe.w13[e].double().t()).chunk(2, -1)
            y = (gate * torch.sigmoid(gate) * up) @ moe.w2[e].double().t()
            out.index_add_(0, t, y * s["w"][t, k].double()[:, None])
    return {"out": out}


def _exact_latent(s):
    b, x, meta = s["block"], s["hidden"].double(), s["ctx"].attn_metadata
    spec, lora = _spec(s["case"]), b.kv_lora
    t = x.shape[0]

    def lin(m, y):
        return y @ m.weight.double().t()

    q = lin(b.q_b_proj, _norm64(lin(b.q_a_proj, x),
                                b.q_a_layernorm.weight.double(),
                                spec.rms_norm_eps))
    q = q.view(t, b.num_heads, -1)
    q_pe = _rotate64(q[..., b.qk_nope:], s["pos"], spec.rope_theta)
    kv = lin(b.kv_a_proj_with_mqa, x)
    k_pe = _rotate64(kv[:, None, lora:], s["pos"], spec.rope_theta)[:, 0]
    new = torch.cat([_norm64(kv[:, :lora], b.kv_a_layernorm.weight.double(),
                             spec.rms_norm_eps), k_pe], -1)
    cache = s["ctx"].kv_caches[0].double()
    cache.view(-1, cache.shape[-1])[meta.slot_mapping] = new
    q_abs = torch.matmul(q[..., :b.qk_nope].transpose(0, 1).contiguous(),
                         b.w_uk.double()).transpose(0, 1)
    q_all = torch.cat([q_abs, q_pe], -1)
    out = []
    starts = meta.query_start_loc.tolist()
    for i, ctx in enumerate(meta.seq_lens.tolist()):
        blocks = meta.block_table[i, :-(-ctx // BLOCK)].long()
        rows = cache[blocks].flatten(0, 1)[:ctx, None]
        for h in range(0, b.num_heads, 32):
            k = rows.expand(-1, 32, -1)
            out.append(_attend64(q_all[starts[i]:starts[i + 1], h:h + 32],
                                 k, k[..., :lora], b.scale, 0))
    per = b.num_heads // 32
    o = torch.cat([torch.cat(out[i:i + per], 1)
                   for i in range(0, len(out), per)])
    o = torch.matmul(o.transpose(0, 1).contiguous(), b.w_uv.double())
    o = o.transpose(0, 1).reshape(t, -1)
    return {"out": lin(b.o_proj, o), "cache": cache}


def _rows64(plane, blocks):
    """[tokens, kv heads, D] of one request, from one plane of a cache."""
    raw = plane.view(torch.uint8)[blocks].view(plane.dtype)
    return raw.to(torch.float64).transpose(1, 2).flatten(0, 1)


def _exact_stack(s):
    model, meta, spec = s["model"], s["ctx"].attn_metadata, _spec(s["case"])
    fp8 = s["case"]["kv"] == "fp8"
    d, g = spec.head_dim, spec.num_heads // spec.num_kv_heads
    starts, lens = meta.query_start_loc.tolist(), meta.seq_lens.tolist()
    t = meta.num_actual_tokens

    def lin(m, y):
        w = m.weight.double()
        y = y @ w.t()
        return y if getattr(m, "bias", None) is None else y + m.bias.double()

    def norm(m, y):
        return _norm64(y, m.weight.double(), spec.rms_norm_eps)

    x = model.model.embed_tokens.weight[s["ids"]].double()
    caches = []
    for layer, cache in zip(model.model.layers, s["ctx"].kv_caches):
        a = layer.self_attn
        q, k, v = lin(a.qkv_proj, norm(layer.input_layernorm, x)).split(
            [a.qkv_proj.q_size, a.qkv_proj.kv_size, a.qkv_proj.kv_size], -1)
        q = _rotate64(q.reshape(t, -1, d), s["pos"], spec.rope_theta)
        k = _rotate64(k.reshape(t, -1, d), s["pos"], spec.rope_theta)
        v = v.reshape(t, -1, d)
        o = torch.empty_like(q)
        for i, ctx in enumerate(lens):
            at, to = starts[i], starts[i + 1]
            blocks = meta.block_table[i, :-(-ctx // BLOCK)].long()
            old = [_rows64(c, blocks)[:ctx - (to - at)] for c in cache]
            kk = torch.cat([old[0], k[at:to]])
            vv = torch.cat([old[1], v[at:to]])
            if to - at == 1:  # decode rows: groups as rows, no repeats
                w = spec.sliding_window
                kk, vv = (kk[-w:], vv[-w:]) if w else (kk, vv)
                sc = torch.matmul(q[at].view(-1, g, d),
                                  kk.permute(1, 2, 0).contiguous())
                p = (sc * d ** -0.5).softmax(-1)
                o[at] = torch.matmul(
                    p, vv.transpose(0, 1).contiguous()).view(-1, d)
                continue
            for h in range(spec.num_kv_heads):
                o[at:to, h * g:(h + 1) * g] = _attend64(
                    q[at:to, h * g:(h + 1) * g],
                    kk[:, h:h + 1].expand(-1, g, -1),
                    vv[:, h:h + 1].expand(-1, g, -1), d ** -0.5,
                    spec.sliding_window)
        if fp8:
            caches.append(None)
        else:
            c64 = cache.double()
            blk, off = meta.slot_mapping // BLOCK, meta.slot_mapping % BLOCK
            c64[0, blk, :, off] = k
            c64[1, blk, :, off] = v
            caches.append(c64)
        x = x + lin(a.o_proj, o.reshape(t, -1))
        gate, up = lin(layer.mlp.gate_up_proj, norm(
            layer.post_attention_layernorm, x)).chunk(2, -1)
        x = x + lin(layer.mlp.down_proj, gate * torch.sigmoid(gate) * up)
    hidden = norm(model.model.norm, x)
    logits = hidden[s["last"]] @ model.lm_head.weight.double().t()
    return {"logits": logits, "hidden": hidden, "caches": caches}


_EXACT = {"stack": _exact_stack, "latent": _exact_latent,
          "experts": _exact_experts}
