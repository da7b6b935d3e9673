"""GPU op wrappers backed by the hand-written CDNA4 HIP kernels.

Importing this module loads vllm_amd/_C.so (torch.library ops under
torch.ops.vllm_amd.*). If the extension is missing the import fails and
ops.get_backend() raises — the GPU path never silently falls back to
eager PyTorch.
"""

from __future__ import annotations

import functools
from pathlib import Path

import torch

_SO = Path(__file__).resolve().parent.parent / "_C.so"
if not _SO.exists():
    raise ImportError(
        f"vllm_amd HIP extension not found at {_SO}; "
        "run `python -m vllm_amd.build`"
    )
torch.ops.load_library(str(_SO))

_C = torch.ops.vllm_amd

# Decode attention: one workgroup takes at least this many keys (4 waves
# of 32), at most 16 times as many, and 2 workgroups fit on each of the
# 256 CUs.
_DEC_UNIT = 128
_DEC_MAX_UNITS = 16
_DEC_FILL = 512


def _decode_parts(rows, kv_heads, max_seq_len, sliding_window, head_dim=128,
                  kv_bytes=1):
    """Into how many partitions a row's keys are split. Every partition
    costs a pass over its fp32 partials, so no more than fill the chip:
    16 rows x 4096 keys (8 KV heads of 128) take 45.3 us in 4 partitions,
    50.3 in 16. Partitions of more than 2048 keys leave ragged batches
    waiting for their longest row; below that more partitions only
    cost: 256 rows x 129..2176 keys take 206 us in 2, 244 in 9; 64 rows
    x 4096..8192 fp8 keys 144 us in 4, 172 in 32. For one or two rows one
    workgroup a CU does: one x 8000 keys 13.2 us in 32, 16.3 in 63; two x
    8000 16.9 in 16, 18.5 in 32 (24 x 500..3000 45.1 in 2, 40.4 in 3). So
    it does for more rows with a cache of 16 bits, where partitions come out
    that 220 of the 256 CUs have one: us in one, and two, a CU, rows alike
    and from a fifth on (8 KV heads of 128) 4 x 2500 11.7 and 14.1, 10.7 and
    12.4; 8 x 4000 23.5 and 24.6, 17.5 and 19.5; 16 x 1200 16.7 and 18.0,
    13.5 and 15.2, x 4000 44.7 and 43.5, 30.7 and 33.2; 2 heads of 256, 6 x
    4000 17.2 and 21.5; 10 rows, 240 CUs, x 4000 29.7 and 30.2, 21.7 and 22.9;
    14, 224 CUs, x 2000 21.1 and 22.7, 17.5 and 18.4; of 9 rows, 216 CUs, x
    800..4000 21.4 and 20.3, of 13, 208 CUs, x 1200 14.8 and 17.2, 13.1 and
    12.7; with 8 bits 16 x 800..4000 23.9 and 20.2. (Of 148 shapes of 3 to 16
    rows in one a CU 9 lose more than 1 %, most of them uneven rows of 800 keys:
    5 x 160..800 8.8 and 8.5, with heads of 256 11.4 and 10.3.) At most 64, the
    lanes of the merging wave.

    Three steps of a workgroup's waves take no longer than to merge, two of
    twice the steps with heads of 256: us in one partition and in those of
    128 keys, 8 KV heads of 128, 1 x 160 4.9 and 6.5, 1 x 384 6.7 and 7.2, 1
    x 400 7.9 and 7.2, 16 x 256 6.3 and 8.5, 40 x 384 14.5 and 16.3; 2 of
    256, 1 x 256 8.8 and 10.3, 1 x 384 11.2 and 10.5."""
    span = max(max_seq_len, 1)
    if sliding_window > 0:
        span = min(span, sliding_window + 31)
    if span <= _DEC_UNIT * (3 if head_dim <= 128 else 2):
        return 1
    units = -(-span // _DEC_UNIT)
    groups = max(rows * kv_heads, 1)
    fill = _DEC_FILL // 2 if rows <= 2 else _DEC_FILL
    parts = -(-fill // groups)
    one = _DEC_FILL // 2 // groups
    if kv_bytes > 1 and groups <= 128 and one * groups >= 220:
        parts = one
    parts = max(parts, -(-units // _DEC_MAX_UNITS))
    return max(1, min(parts, units, 64))


def _aligned(*tensors):
    """Operands that kernels fill LDS from directly, 16 B at a time, must
    begin on 16 B; views into odd places take a form with plain loads."""
    return all(t.data_ptr() % 16 == 0 for t in tensors)


def rms_norm(x, weight, eps):
    return _C.rms_norm(x, weight, eps)


def fused_add_rms_norm(x, residual, weight, eps):
    # In-place: x <- norm(x + residual), residual <- x + residual.
    _C.fused_add_rms_norm(x, residual, weight, eps)
    return x, residual


def apply_rope(positions, q, k, cos_sin_cache, rotary_dim, is_neox=True):
    assert is_neox, "HIP rope kernel implements neox style"
    _C.rotary_embedding(positions, q, k, cos_sin_cache, rotary_dim)
    return q, k


def silu_and_mul(x):
    if x.dtype == torch.float32 or (x.shape[-1] // 2) % 8:
        # The 16-bit kernel is vectorized for 2-byte elements in groups
        # of 8; fp32 rows and other widths take the generic one.
        shape = list(x.shape)
        out = _C.silu_and_mul_any(x.reshape(-1, shape[-1]).contiguous())
        shape[-1] //= 2
        return out.reshape(shape)
    return _C.silu_and_mul(x)


def gelu_and_mul(x):
    return _C.gelu_and_mul(x)


def linear(x, weight, bias=None):
    # Few rows stream the weights (csrc/stream_linear.hip, tile_linear.hip),
    # others take a tuned hipBLASLt GEMM (per-shape algo search on first
    # use). Rows that are not 16-byte multiples fall outside the aligned
    # kernels: those shapes go to torch's vendor GEMM instead.
    per16 = 4 if x.dtype == torch.float32 else 8
    if weight.shape[0] % per16 or weight.shape[1] % per16:
        return torch.nn.functional.linear(x, weight, bias)
    return _C.lt_linear(x, weight, bias)


def linear_silu_and_mul(x, weight):
    # The activation as the product's epilogue where few rows stream the
    # weights (csrc/stream_linear.hip) and in tiles of up to 256 rows
    # (tile_linear.hip); other shapes take two launches.
    n2, k = weight.shape
    if (x.dtype == torch.float32 or n2 % 16 or k % 64
            or x.numel() > 256 * k or x.numel() == 0):
        return silu_and_mul(linear(x, weight))
    return _C.linear_silu_and_mul(x, weight)


def norm_linear(x, gain, eps, weight, bias=None, silu=False):
    return _C.norm_linear(x, gain, eps, weight, bias, silu)


def norm_qkv_rope_cache(x, gain, eps, weight, bias, positions, cos_sin_cache,
                        kv_cache, slot_mapping):
    kv_heads, head_dim = kv_cache.shape[2], kv_cache.shape[4]
    if head_dim % 16:
        # rope_and_cache knows what to do with these.
        qkv = norm_linear(x, gain, eps, weight, bias).view(
            x.shape[0], -1, head_dim)
        q, k, v = qkv.split([qkv.shape[1] - 2 * kv_heads, kv_heads, kv_heads],
                            dim=1)
        rope_and_cache(positions, q, k, v, cos_sin_cache, head_dim, True,
                       kv_cache, slot_mapping)
        return q
    return _C.norm_qkv_rope_cache(x, gain, eps, weight, bias, positions,
                                  slot_mapping, cos_sin_cache, kv_cache)


def linear_add(x, weight, bias, residual):
    return _C.linear_add(x, weight, bias, residual)


@functools.lru_cache(maxsize=1024)
def layer_streams(rows, hidden, qkv, heads, gate_up, inner, half):
    # Up to 64 rows (csrc/stream_linear.hip). (Prompts come in any number.)
    return _C.layer_streams(rows, hidden, qkv, heads, gate_up, inner, half)


def quant_fp8_dynamic(x):
    # Per-token dynamic quant (csrc/quant_fp8.hip): one workgroup/row.
    M, K = x.shape
    out = torch.empty(M, K, dtype=torch.float8_e4m3fn, device=x.device)
    scales = torch.empty(M, dtype=torch.float32, device=x.device)
    _C.dynamic_quant_fp8(out.view(torch.uint8), scales, x)
    return out, scales


def linear_fp8(x, w_fp8, w_scale, bias=None):
    """W8A8 fp8 linear: per-token activation quant -> fp8 MFMA GEMM
    (tuned hipBLASLt, raw bf16 out) -> fused rs[m]*cs[n] rescale + bias.
    ~2x bf16 GEMM rate on gfx950 and half the weight HBM traffic."""
    shape = list(x.shape)
    x2 = x.reshape(-1, shape[-1]).contiguous()
    x_fp8, x_scale = quant_fp8_dynamic(x2)
    y = _C.lt_linear_fp8(x_fp8, w_fp8)
    _C.scale_rows_cols(y, x_scale, w_scale, bias)
    shape[-1] = w_fp8.shape[0]
    return y.reshape(shape)


def reshape_and_cache(key, value, kv_cache, slot_mapping):
    _C.reshape_and_cache(key, value, kv_cache, slot_mapping)


def rope_and_cache(positions, q, k, v, cos_sin_cache, rotary_dim, is_neox,
                   kv_cache, slot_mapping):
    """One launch where heads split into 16 B pieces (csrc/elementwise.hip
    rope_cache_kernel), else rotation and cache write."""
    D = q.shape[2]
    if (is_neox and rotary_dim % 16 == 0 and D % 16 == 0
            and 16 <= rotary_dim <= D == v.shape[2]
            and q.dtype in (torch.bfloat16, torch.float16)
            and kv_cache.dtype in (q.dtype, torch.float8_e4m3fn)
            and kv_cache.is_contiguous()
            and all(x.data_ptr() % 16 == 0 and x.dtype == q.dtype
                    for x in (q, k, v))):
        _C.rope_and_cache(positions, q, k, v, cos_sin_cache, rotary_dim,
                          kv_cache, slot_mapping)
    else:
        apply_rope(positions, q, k, cos_sin_cache, rotary_dim, is_neox)
        reshape_and_cache(k, v, kv_cache, slot_mapping)


def _decode_waves(units, head_dim, parts, span):
    """Whether a wave takes a row of its own: plan_decode of
    csrc/attention_decode.hip, for rows * KV heads units."""
    return parts == 1 and (
        (span <= 128 and units >= (1536 if head_dim == 64 else 1024))
        or (span <= 512 and units >= 4096 and head_dim <= 128))


def _attention_mixes(rows, reqs, tokens, heads, head_dim, kv_heads, parts,
                     max_decode_len, max_seq_len, max_query_len,
                     window=0, kv_bytes=2):
    """Whether decode rows and portions of prompts run in one launch
    (csrc/attention_mixed.hip). Not rows that take a wave each (1024 x 64 keys
    and 8 portions of 128 tokens 58 us in turn, 74 as workgroups in one
    launch), heads that one of the two kernels does not take, nor grids past
    65535 units. Nor rows that read (5 TB/s) less than a twentieth of the time
    that the portions may take (0.8 PFLOP/s): they have hardly any effect (1
    row x 1000 keys and 8000 tokens 518 us in turn, 522 in one launch). A
    third where portions come after more cached tokens than they are long:
    their tiles are all of one length and fill the chip in step, which rows
    among them disturb (4 portions of 1000 after 4000 beside 8 x 4000 keys,
    16/2 heads, 177 and 200 us, one of 2000 after 6000 beside 32 x 1000, 32/8
    heads, 265 and 307; the 4 beside 64 x 2000, 8/8 heads, 182 and 144)."""
    if not 0 < rows < reqs or head_dim not in (64, 128):
        return False
    if heads % kv_heads or heads // kv_heads > 8:
        return False
    span = max_decode_len
    if window > 0:
        span = min(span, window + 31)
    if _decode_waves(rows * kv_heads, head_dim, parts, span):
        return False
    read_us = rows * span * kv_heads * head_dim * 2 * kv_bytes / 5e6
    # (Cached tokens of portions are known only where the longest context is
    # not a row's.)
    alike = (max_seq_len > max_decode_len
             and max_seq_len >= 2 * max_query_len)
    keys = max_seq_len - max_query_len / 2 if alike else max_seq_len / 2
    if window > 0:
        keys = min(keys, window)
    tile_us = (tokens - rows) * keys * heads * head_dim * 4 / 8e8
    tiles = -(-max_query_len * (heads // kv_heads) // 128)
    return (read_us * (3 if alike else 20) >= tile_us
            and tiles * (reqs - rows) + rows * parts < 65536)


def attention_unified(
    q,
    kv_cache,
    block_table,
    query_start_loc,
    seq_lens,
    scale,
    num_decodes=0,
    sliding_window=0,
    max_seq_len=0,
    max_query_len=0,
    max_decode_len=0,
):
    """Dispatch decode rows (first num_decodes, query_len==1) to the
    partitioned decode kernel and the rest to the MFMA prefill
    kernel. max_seq_len/max_query_len come from the scheduler (CPU) so
    no device sync is needed here. Decode rows are split by
    max_decode_len where it is known: by the length of a prompt beside
    them 64 rows x 1000 keys took 47 us (32768 tokens), by their own 41."""
    num_tokens, num_heads, head_dim = q.shape
    # q may be a strided head-slice of the fused QKV output; the kernels
    # take its row stride. The output is always freshly contiguous.
    out = torch.empty(
        (num_tokens, num_heads, head_dim), dtype=q.dtype, device=q.device
    )
    if max_seq_len <= 0:
        max_seq_len = int(seq_lens.max().item())
    num_reqs = seq_lens.shape[0]

    if num_decodes > 0:
        q_dec = q[:num_decodes]
        if max_decode_len <= 0:
            max_decode_len = max_seq_len
        num_parts = _decode_parts(num_decodes, kv_cache.shape[2],
                                  max_decode_len, sliding_window, head_dim,
                                  kv_cache.element_size())
        if num_parts > 1:
            tmp_out = torch.empty(
                num_decodes, num_heads, num_parts, head_dim,
                dtype=torch.float32, device=q.device,
            )
            tmp_lse = torch.empty(
                num_decodes, num_heads, num_parts, 2,
                dtype=torch.float32, device=q.device,
            )
        else:
            tmp_out = q.new_empty(0, dtype=torch.float32)
            tmp_lse = tmp_out
        if (max_query_len <= 0 and num_decodes < num_reqs
                and head_dim in (64, 128)):
            qsl = query_start_loc
            max_query_len = int((qsl[1:] - qsl[:-1]).max().item())
        if _attention_mixes(num_decodes, num_reqs, num_tokens, num_heads,
                            head_dim, kv_cache.shape[2], num_parts,
                            max_decode_len, max_seq_len, max_query_len,
                            sliding_window, kv_cache.element_size()):
            _C.mixed_attention(
                out, q, kv_cache, block_table, query_start_loc, seq_lens,
                scale, num_decodes, max_decode_len, max_query_len,
                sliding_window, tmp_out, tmp_lse,
            )
            return out
        _C.paged_decode_attention(
            out[:num_decodes], q_dec, kv_cache, block_table, seq_lens,
            scale, max_decode_len, sliding_window, tmp_out, tmp_lse,
        )

    if num_decodes < num_reqs:
        if head_dim not in (64, 128, 256):
            # Off-template head dims take an explicit torch path for the
            # prefill rows (decode runs the HIP kernel at any supported
            # head_dim). Gemma3 (256) and OPT (64) are on the MFMA
            # kernel since the head-dim templating.
            _warn_prefill_fallback(head_dim)
            from vllm_amd.ops import _torch_ref

            qsl = query_start_loc[num_decodes:] - num_decodes
            ref_out = _torch_ref.attention_unified(
                q[num_decodes:], kv_cache, block_table[num_decodes:],
                qsl, seq_lens[num_decodes:], scale, num_decodes=0,
                sliding_window=sliding_window,
            )
            out[num_decodes:] = ref_out
            return out
        if max_query_len <= 0:
            qsl = query_start_loc
            max_query_len = int((qsl[1:] - qsl[:-1]).max().item())
        _C.prefill_attention(
            out, q, kv_cache, block_table, query_start_loc, seq_lens,
            scale, num_decodes, max_query_len, sliding_window,
        )
    return out


_PREFILL_FALLBACK_WARNED = set()


def _warn_prefill_fallback(head_dim: int) -> None:
    if head_dim not in _PREFILL_FALLBACK_WARNED:
        _PREFILL_FALLBACK_WARNED.add(head_dim)
        import logging

        logging.getLogger(__name__).warning(
            "prefill head_dim=%d: off-template (64/128/256); prefill "
            "rows use the torch path (decode stays on the HIP kernel)",
            head_dim)


# MoE routing (small [T, E] tensors — torch ops are fine here).
from vllm_amd.ops import _torch_ref  # noqa: E402
from vllm_amd.ops._torch_ref import (  # noqa: E402,F401
    concat_and_cache_mla,
    grouped_topk,
    topk_softmax,
)

# MLA decode: one workgroup (128 heads of a row) fits on each of the 256
# CUs; a partition of its keys costs 256 KB of fp32 partials written and
# read.
_MLA_FILL = 256
_MLA_PART_MIN = 128


def _mla_parts(rows, heads, max_seq_len):
    """Into how many partitions a row's keys are split: as many as run at
    a time and no more (128 heads, us in 1 / 2 / 4 / 8: 200 rows x 129..2176
    keys 139 / 151 / 149; 128 rows 128 / 90 / 115; 32 rows x 8192 441 / 237
    / 134 / 105, 16 132), none shorter than two tiles (one row x 1000 keys
    24 in 8, 22 in 16; x 4000 31 in 16, 29 in 32, 35 in 63), at most 64."""
    groups = rows * -(-heads // 128)
    return max(1, min(_MLA_FILL // max(groups, 1),
                      -(-max_seq_len // _MLA_PART_MIN), 64))


def _mla_group_heads(pairs, heads):
    """Heads that a workgroup takes (csrc/mla.hip, group_heads) of so many
    rows and partitions: the fewest of 32, 64 and 128 that one round of
    workgroups has room for."""
    n = 128
    while n > 32 and heads > n // 2 and pairs * -(-heads // (n // 2)) <= _MLA_FILL:
        n //= 2
    return n


@functools.lru_cache(maxsize=1024)
def _mla_split(rows, heads, max_seq_len):
    """Into how many partitions the kernel splits a row's keys: as
    _mla_parts says or, where that is 5 % less by an estimate, as many as
    leave room for workgroups of fewer heads. The estimate, in us: a start and the queries' way in,
    tiles of 64 keys, and with partitions a launch and their traffic. Its
    coefficients come from a fit of 528 times at 16, 64 and 128 heads, 1 to
    200 rows and 60 to 16000 keys, which they meet within 5 %.
    max_seq_len is a bound, for captured steps the longest that rows may
    become: longer partitions must not be behind either where rows have a
    quarter or a sixteenth of it (4 rows, 64 heads, told 8192: of 491 keys
    16.0 in 64 partitions, 20.4 in 32). Of 820 times at 16 to 128 heads, 1 to
    160 rows, told 100 to 16384 keys and having all, 0.6, a quarter or 0.06
    of them, 0.89 of _mla_parts' on average; 26 above 1.02, all at less than
    35 us, the worst 1.09 (64 rows, 16 heads, 120 keys told 200: 11.5)."""
    first = _mla_parts(rows, heads, max_seq_len)

    def us(parts, keys):
        wide = _mla_group_heads(rows * parts, heads)
        took = min(wide, heads)
        part_tiles = max(1, -(-max_seq_len // (64 * parts)))
        used = min(parts, -(-keys // (64 * part_tiles)))
        groups = rows * used * -(-heads // wide)
        tile = 2.1 if took <= 32 else 2.3 if took <= 64 else 3.15
        tiles = min(part_tiles, -(-keys // 64)) * -(-groups // _MLA_FILL)
        t = (3.8 + 9.8 * took / 128
             + tiles * tile * (1 + 0.25 * min(groups / _MLA_FILL, 1)))
        if parts > 1:
            t += 2.2 + 0.16 * used + rows * used * heads * 4.5e-4
        return t

    shorter = [max(1, max_seq_len // n) for n in (4, 16)]
    limits = [us(first, keys) for keys in shorter]
    best, least = first, us(first, max_seq_len) * 0.95
    for n in (32, 64):
        room = _MLA_FILL // max(1, rows * -(-heads // n))
        parts_of = [min(room, -(-max_seq_len // keys), 64)
                    for keys in (64, 128)] + [1] * (room > 0)
        for parts in parts_of:
            if parts > 0 and us(parts, max_seq_len) < least and all(
                    us(parts, k) <= u for k, u in zip(shorter, limits)):
                best, least = parts, us(parts, max_seq_len)
    return best


def _mla_scratch(q, max_seq_len):
    """Partials of the partitions of q's rows [T, Hq, lora]; empty for one
    partition."""
    T, Hq, lora = q.shape
    parts = _mla_split(T, Hq, max_seq_len)
    if parts == 1:
        none = q.new_empty(0, dtype=torch.float32)
        return none, none
    return (q.new_empty(T, Hq, parts, lora, dtype=torch.float32),
            q.new_empty(T, Hq, parts, 2, dtype=torch.float32))


def mla_decode(q_nope, q_pe, kv_cache, block_table, seq_lens, scale,
               max_seq_len):
    """Absorbed-MQA MLA decode on the MFMA kernel (csrc/mla.hip);
    kv_lora_rank 512 + rope 64 latent cache."""
    T, Hq, lora = q_nope.shape
    out = torch.empty(T, Hq, lora, dtype=q_nope.dtype, device=q_nope.device)
    if max_seq_len <= 0:
        max_seq_len = int(seq_lens.max().item())
    _C.mla_decode(out, q_nope, q_pe, kv_cache, block_table, seq_lens,
                  scale, max_seq_len, *_mla_scratch(q_nope, max_seq_len))
    return out


def mla_attention(q_nope, q_pe, kv_cache, block_table, query_start_loc,
                  seq_lens, scale, num_decodes=0, max_seq_len=0,
                  max_prompt_len=0):
    """Decode rows (query_len==1, first num_decodes) and prompt rows on
    the MFMA kernel (csrc/mla.hip). Other latent widths, types or cache
    types take the torch composition. max_prompt_len bounds the prompts'
    contexts (0: max_seq_len does, or they are not split)."""
    T = q_nope.shape[0]
    use_hip = (q_nope.shape[2] == 512 and q_pe.shape[2] == 64
               and q_nope.dtype in (torch.bfloat16, torch.float16)
               and q_pe.dtype == q_nope.dtype
               and kv_cache.dtype == q_nope.dtype and _aligned(kv_cache))
    if not use_hip:
        return _torch_ref.mla_attention(
            q_nope, q_pe, kv_cache, block_table, query_start_loc, seq_lens,
            scale)
    q_nope, q_pe = q_nope.contiguous(), q_pe.contiguous()
    if num_decodes == T:
        return mla_decode(q_nope, q_pe, kv_cache, block_table,
                          seq_lens[:num_decodes], scale, max_seq_len)
    out = torch.empty_like(q_nope)
    if num_decodes > 0:
        out[:num_decodes] = mla_decode(
            q_nope[:num_decodes], q_pe[:num_decodes], kv_cache,
            block_table, seq_lens[:num_decodes], scale, max_seq_len)
    bound = max_prompt_len or max_seq_len
    _C.mla_prefill(out, q_nope, q_pe, kv_cache, block_table,
                   query_start_loc, seq_lens, scale, num_decodes, bound,
                   *_mla_scratch(q_nope[num_decodes:], bound))
    return out


def head_matmul(x, w):
    """out[t, h] = x[t, h] @ w[h], fp32 sums, result in x's type."""
    if (x.dtype in (torch.bfloat16, torch.float16) and x.dtype == w.dtype
            and w.shape[1] % 128 == 0 and w.shape[2] % 128 == 0
            and w.is_contiguous() and x.stride(2) == 1
            and x.stride(0) % 8 == 0 and x.stride(1) % 8 == 0
            and _aligned(x, w)):
        return _C.head_matmul(x, w)
    return _torch_ref.head_matmul(x, w)


def mla_prepare(positions, q_pe, kv_a, weight, eps, cos_sin_cache, kv_cache,
                slot_mapping):
    """Norm, rotations and cache write of an MLA block's projections in
    one launch where rows are 16 B aligned and everything has one 16-bit
    type; else step by step."""
    aligned = all(
        x.stride(-1) == 1 and x.data_ptr() % 16 == 0
        and all(n % 8 == 0 for n in x.stride()[:-1])
        for x in (q_pe, kv_a, weight))
    if (aligned and q_pe.shape[2] == 64 and weight.shape[0] == 512
            and kv_a.shape[1] == 576 and kv_cache.shape[2] == 576
            and kv_cache.is_contiguous() and cos_sin_cache.shape[-1] == 64
            and q_pe.dtype in (torch.bfloat16, torch.float16)
            and all(x.dtype == q_pe.dtype
                    for x in (kv_a, weight, kv_cache))):
        return _C.mla_prepare(positions, q_pe, kv_a, weight, eps,
                              cos_sin_cache, kv_cache, slot_mapping)
    lora = weight.shape[0]
    c_kv = rms_norm(kv_a[:, :lora].contiguous(), weight, eps)
    q_pe = q_pe.contiguous()
    k_pe = kv_a[:, lora:].unsqueeze(1).contiguous()
    apply_rope(positions, q_pe, k_pe, cos_sin_cache, k_pe.shape[-1])
    concat_and_cache_mla(c_kv, k_pe.squeeze(1), kv_cache, slot_mapping)
    return q_pe


_MLA_PROMPT_SCRATCH = 512 << 20   # bytes


def _mla_prompt_heads(q_nope, w_uk, w_uv, kv_cache, reqs, scale,
                      num_decodes, max_query_len, max_seq_len):
    """How many heads at a time prompt portions attend with keys and
    values carried out of the latent space (csrc/mla_prompt.hip); 0:
    in it (csrc/mla.hip). Carrying them out costs by context row, the
    latent form by query (a part for each and a part per key; 200 at
    least, which fill the chip, or 256 pieces of queries whose keys are
    split), so the line is a number of queries per request that grows with
    the context. us per head / latent, 8 requests: 96 tokens of 512 260 /
    261, 128 267 / 342; 192 of 2048 1233 / 1181, 256 of 4096 2492 / 2786;
    32 requests: 32 of 128 265 / 242, 64 of 256 521 / 552; one: 64 of 512
    54 / 62, 128 of 2048 150 / 136, 160 154 / 175, 192 of 8192 655 / 623,
    256 629 / 692. Only the longest context is known here: shorter ones
    cost less than this says, most so per head."""
    T, Hq, nope = q_nope.shape
    rows, reqs = T - num_decodes, reqs - num_decodes
    S = max(max_seq_len, 128)
    parts = _mla_parts(rows, Hq, S)
    cost = (max(rows, 200) * (800 + S) if parts == 1 else
            256 * (800 + S // parts))
    if (nope != 128 or w_uk.shape[2] != 512 or w_uv.shape[2] != 128
            or kv_cache.shape[2] != 576 or scale <= 0 or max_query_len <= 0
            or max_seq_len <= 0 or not 0 < reqs < 65536 or rows <= 0
            or cost < reqs * 255 * S
            or q_nope.dtype not in (torch.bfloat16, torch.float16)
            or any(t.dtype != q_nope.dtype for t in (w_uk, w_uv, kv_cache))
            or not all(t.is_contiguous() for t in (w_uk, w_uv, kv_cache))
            or q_nope.stride(2) != 1 or q_nope.stride(0) % 8
            or q_nope.stride(1) % 8
            or not _aligned(q_nope, w_uk, w_uv, kv_cache)):
        return 0
    heads = min(Hq, _MLA_PROMPT_SCRATCH // (reqs * max_seq_len * 512))
    # The kernel deals eight heads at a time to the eight XCDs.
    return heads if heads < 8 or heads == Hq else heads // 8 * 8


def mla_heads(q_nope, q_pe, w_uk, w_uv, kv_cache, block_table,
              query_start_loc, seq_lens, scale, num_decodes=0,
              max_query_len=0, max_seq_len=0, max_decode_len=0,
              max_prompt_len=0):
    """MLA attention from per-head queries to per-head results. Decode
    rows and short portions work on the latent rows themselves; portions
    of many tokens carry their context's keys and values out of the latent
    space first. Decode rows are split by max_decode_len where it is
    known (32 rows x 1000 keys beside a prompt of 8192: 68 us by the
    prompt's length, 45 by their own); form and scratch of the portions go
    by max_prompt_len (20 portions of 400 beside a row of 8192 keys: 3.1
    ms in 22 passes over the heads by the row's length, 0.98 by their own)."""
    T = q_nope.shape[0]
    reqs = seq_lens.shape[0]

    def latent(n, reqs):
        o = mla_attention(head_matmul(q_nope[:n], w_uk), q_pe[:n], kv_cache,
                          block_table[:reqs], query_start_loc[:reqs + 1],
                          seq_lens[:reqs], scale, num_decodes=num_decodes,
                          max_seq_len=max_decode_len or max_seq_len,
                          max_prompt_len=max_prompt_len or max_seq_len)
        return head_matmul(o, w_uv)

    S = max_prompt_len or max_seq_len
    heads = _mla_prompt_heads(q_nope, w_uk, w_uv, kv_cache, reqs, scale,
                              num_decodes, max_query_len, S)
    if heads == 0:
        return latent(T, reqs)
    out = torch.empty(T, q_nope.shape[1], w_uv.shape[2], dtype=q_nope.dtype,
                      device=q_nope.device)
    if num_decodes > 0:
        out[:num_decodes] = latent(num_decodes, num_decodes)
    rows = (reqs - num_decodes) * S
    scratch = torch.empty(rows * (64 + heads * 256), dtype=q_nope.dtype,
                          device=q_nope.device)
    exps = torch.empty(heads * (reqs - num_decodes) * -(-S // 64) * 2,
                       dtype=torch.int32, device=q_nope.device)
    _C.mla_prompt_attention(out, q_nope, q_pe.contiguous(), w_uk, w_uv,
                            kv_cache, block_table, query_start_loc, seq_lens,
                            scale, num_decodes, max_query_len, S, scratch,
                            exps)
    return out


# Form of the expert products by the average number of rows an expert gets:
# below 24 weights are streamed past at most 64 rows, below 192 tiles of 128
# rows, from there 256 (in which an expert of at most 32 rows is streamed as
# well). ms streamed / 128 / 256, chosen evenly: 8 experts of 4096 x 14336, 12
# rows 0.44 / 0.49 / 0.49, 32 rows 0.47 / 0.54 / 0.54 (0.61 / 0.53 / 0.53
# where half of the tokens agree), 64 rows 0.76 / 0.57 / 0.57, 100 rows 0.94 /
# 0.60 / 0.60; 64 experts of 7168 x 2048, 16 rows 0.87 / 0.86 / 0.87, 64 rows
# 1.43 / 1.03 / 1.03.
# Where one tile per expert leaves more than half of the chip idle, tiles are
# worth it from 48 rows only: 16 experts of 1024 x 3584 without a gate, us
# streamed / 128, 24 rows 70 / 82 (76 / 78 where half agree), 38 rows 76 / 82
# (80 / 95), 50 rows 89 / 82 (85 / 94), 64 rows 96 / 63; 8 of 1024 x 2048, 32
# rows 34 / 57, 48 rows 36 / 41, 64 rows 56 / 45.
_MOE_TILES_FROM = 24
_MOE_FEW_TILES_FROM = 48
_MOE_WIDE_TILES_FROM = 192
# The average says little where rows meet in few experts (equal prompts,
# padded rows of a captured step): weights of an expert with more than 64
# rows are streamed once per 64. So tiles also from 4 rows an expert where
# an expert may get more than 64 (the batch holds more tokens) and one tile
# per expert fills the chip. us streamed / 128, experts chosen evenly | by
# half of the tokens | all the same: 64 experts of 7168 x 2048, 8 a token,
# 80 tokens 856 / 858 | 858 / 846 | 267 / 197, 191 tokens 923 / 888 | 959 /
# 900 | 342 / 212; 128 of 2048 x 768, 65 tokens 209 / 218 | 210 / 220 | 51 /
# 46. Not filled: 8 experts of 4096 x 14336, 2 a token, 65 tokens 439 / 516 |
# 452 / 504 | 281 / 299.
_MOE_STREAM_ROWS = 64
_MOE_CHIP_TILES = 256


def _moe_form(tokens, total, E, H):
    """0 streamed, 1 and 2 tiles of 128 and 256 rows, for total (token,
    expert) pairs of tokens rows of H, no pair twice."""
    if total >= _MOE_WIDE_TILES_FROM * E:
        return 2
    chip = E * -(-H // 256) / _MOE_CHIP_TILES
    if total >= (_MOE_TILES_FROM if chip >= 0.5 else _MOE_FEW_TILES_FROM) * E:
        return 1
    return int(tokens > _MOE_STREAM_ROWS and total >= 4 * E and chip >= 1)


def _moe_hip_ok(hidden, w13, w2, activation):
    if activation not in ("silu", "relu2"):
        return False
    if hidden.dtype not in (torch.bfloat16, torch.float16):
        return False
    H = hidden.shape[1]
    n1 = w13.shape[1]
    if activation == "relu2":
        # Ungated: GEMM1 K=H%64, N=I%128; GEMM2 K=I%64, N=H%128.
        return H % 128 == 0 and n1 % 128 == 0
    # GEMM1: K=H%64, N=2I%128; GEMM2: K=I%64, N=H%128.
    return H % 128 == 0 and n1 % 128 == 0 and (n1 // 2) % 64 == 0


def moe_shuffle_weights(w):
    """Pre-shuffle expert weights [E, N, K] into MFMA fragment-major
    order [E][N/16][K/32][64 lanes][8 elems]: each wave's B-fragment
    becomes one coalesced 16B/lane HBM read (csrc/moe.hip
    moe_stream_kernel). One-time cost at weight load."""
    E, N, K = w.shape
    v = w.view(E, N // 16, 16, K // 32, 4, 8)
    v = v.permute(0, 1, 3, 4, 2, 5)
    return v.reshape(E, (N // 16) * (K // 32) * 512).contiguous()


def fused_moe_hip(hidden, w13, w2, topk_weights, topk_ids,
                  w13_shuf=None, w2_shuf=None, activation="silu"):
    """Grouped-GEMM MFMA MoE (csrc/moe.hip): on-device token->expert
    sort into BM tiles, two MFMA GEMMs streaming each expert's weights,
    deterministic weighted combine. No host sync — hipGraph-capturable
    (role of the reference's fused_moe.py:299 + moe_align_sum_kernels.cu).
    """
    T, H = hidden.shape
    E, n1, _ = w13.shape
    I = w2.shape[2]
    k = topk_ids.shape[1]
    total = T * k
    dev = hidden.device
    form = _moe_form(T, total, E, H)
    if (max(T * H, (total + E * 256) * I, n1 * H) >= 1 << 31
            or not _aligned(hidden, w13, w2)):
        form = 0    # tiles address 4 GB, by 16 B
    if form > 0:    # (they take the weights in their own order)
        w13_shuf = w2_shuf = None
    bm = _C.moe_tile_rows(form)
    tiles = (total + min(E, total) * (bm - 1)) // bm
    em = tiles * bm
    ids32 = topk_ids.to(torch.int32).contiguous()
    blocks = -(-total // 2048)
    scratch = torch.empty(
        em + tiles + 1 + total + (blocks * E if blocks > 1 else 0)
        + (2 * E if E > 1024 else 0),
        dtype=torch.int32, device=dev)
    sorted_ids, expert_tiles, inv_perm, part = scratch.split(
        [em, tiles + 1, total, scratch.numel() - em - tiles - 1 - total])
    _C.moe_align(ids32, E, bm, sorted_ids, expert_tiles, inv_perm, part)
    act_kind = 2 if activation == "relu2" else 1
    act = torch.empty(em, I, dtype=hidden.dtype, device=dev)
    if w13_shuf is not None:
        _C.moe_gemm_shuf(hidden, w13_shuf, act, sorted_ids, expert_tiles,
                         n1, H, k, total, act_kind)
    else:
        _C.moe_gemm(hidden, w13, act, sorted_ids, expert_tiles, k, total,
                    act_kind, form)
    y = torch.empty(em, H, dtype=hidden.dtype, device=dev)
    if w2_shuf is not None:
        _C.moe_gemm_shuf(act, w2_shuf, y, sorted_ids, expert_tiles,
                         H, I, 0, total, 0)
    else:
        _C.moe_gemm(act, w2, y, sorted_ids, expert_tiles, 0, total, 0, form)
    out = torch.empty(T, H, dtype=hidden.dtype, device=dev)
    _C.moe_combine(out, y, topk_weights.float().contiguous(), inv_perm)
    return out


def fused_moe(hidden, w13, w2, topk_weights, topk_ids, activation="silu",
              w13_shuf=None, w2_shuf=None):
    """MoE expert MLP on GPU. Primary path: the grouped-GEMM MFMA kernel
    (fused_moe_hip, no host sync; fragment-major weight stream when the
    layer provides pre-shuffled copies). Fallback for unsupported shapes
    or activations: tokens sorted by expert, one tuned hipBLASLt GEMM
    pair per non-empty expert (one D2H sync per call), weighted
    scatter-add combine.

    hidden: [T, H]; w13: [E, 2I, H]; w2: [E, H, I].
    """
    if _moe_hip_ok(hidden, w13, w2, activation):
        return fused_moe_hip(hidden, w13, w2, topk_weights, topk_ids,
                             w13_shuf=w13_shuf, w2_shuf=w2_shuf,
                             activation=activation)
    T, H = hidden.shape
    E = w13.shape[0]
    k = topk_ids.shape[1]
    flat = topk_ids.long().flatten()
    order = torch.argsort(flat, stable=True)
    token_of = order // k
    counts = torch.bincount(flat, minlength=E).cpu().tolist()
    x = hidden[token_of].contiguous()
    out_sorted = torch.empty(T * k, H, dtype=hidden.dtype,
                             device=hidden.device)
    act = {"silu": silu_and_mul, "gelu": gelu_and_mul,
           "relu2": lambda v: _C.relu2(v.contiguous())}[activation]
    offset = 0
    for e in range(E):
        c = counts[e]
        if c == 0:
            continue
        seg = x[offset:offset + c]
        h = act(linear(seg, w13[e]))
        out_sorted[offset:offset + c] = linear(h, w2[e])
        offset += c
    w = topk_weights.flatten()[order].unsqueeze(1).float()
    out = torch.zeros(T, H, dtype=torch.float32, device=hidden.device)
    out.index_add_(0, token_of, out_sorted.float() * w)
    return out.to(hidden.dtype)


# ---------------------------------------------------------------------
# fp32 residual stream / token shift / scalar-gain norm / windowed
# attention with pooled far blocks (csrc/pooled_attention*.hip).

def scalar_rms_norm(x, gain, eps, out_dtype=None):
    return _C.scalar_rms_norm(x.contiguous(), gain, eps,
                              out_dtype or torch.float32)


def add_scaled_scalar_norm(residual, y, gain, eps, mult, out_dtype=None):
    return _C.add_scaled_scalar_norm(residual, y.contiguous(), gain, eps,
                                     mult, out_dtype)


def token_shift(x, shift, state, state_rows, query_start_loc, out_dtype):
    return _C.token_shift(x, shift, state,
                          state_rows if state is not None else None,
                          query_start_loc, out_dtype)


def norm_qk_cache_write(q, k, v, q_w, k_w, eps, k_cache, v_cache,
                        slot_mapping):
    return _C.norm_qk_cache_write(q, k, v, q_w, k_w, eps, k_cache, v_cache,
                                  slot_mapping)


def split_cache_write(key, value, k_cache, v_cache, slot_mapping):
    # Same kernel without norms; the normed-q output is unused here.
    _C.norm_qk_cache_write(key[:, :0], key, value, None, None, 0.0,
                           k_cache, v_cache, slot_mapping)


def pool_update(k_cache, v_cache, pool_k, pool_v, block_table,
                query_start_loc, seq_lens, pool, max_query_len=0):
    if max_query_len <= 0:
        qsl = query_start_loc
        max_query_len = int((qsl[1:] - qsl[:-1]).max().item())
    _C.pool_update(k_cache, v_cache, pool_k, pool_v, block_table,
                   query_start_loc, seq_lens, pool, max_query_len)


def pooled_window_attention(q, k_cache, v_cache, pool_k, pool_v,
                            block_table, query_start_loc, seq_lens, scale,
                            window, pool, gate=None, num_decodes=0,
                            max_seq_len=0, max_query_len=0):
    """Decode rows (the first num_decodes requests, one token each) run
    on the split-key decode kernel in 16-bit dtypes; prefill chunks run
    on the MFMA tile kernel in bf16. fp32 (and fp16 prefill rows) use
    the row-wise kernel, which VLLM_AMD_PWA_ROWWISE=1 forces for all."""
    import os

    T, H, _ = q.shape
    q = q.contiguous()
    out = torch.empty(T, H, v_cache.shape[3], dtype=q.dtype,
                      device=q.device)
    num_reqs = seq_lens.shape[0]
    rowwise = os.environ.get("VLLM_AMD_PWA_ROWWISE", "0") == "1"
    half = q.dtype in (torch.bfloat16, torch.float16) and not rowwise
    tiled = q.dtype == torch.bfloat16 and not rowwise
    row0 = 0
    if half and num_decodes > 0:
        if max_seq_len <= 0:
            max_seq_len = int(seq_lens[:num_decodes].max().item())
        _C.pooled_window_attention_decode(
            out, q, k_cache, v_cache, pool_k, pool_v, block_table,
            query_start_loc, seq_lens, gate, scale, window, pool,
            num_decodes, max_seq_len)
        row0 = num_decodes
    n_rows = (num_decodes if tiled else T) - row0
    if n_rows > 0:
        _C.pooled_window_attention_rows(
            out, q, k_cache, v_cache, pool_k, pool_v, block_table,
            query_start_loc, seq_lens, gate, scale, window, pool, row0,
            n_rows)
    if tiled and num_decodes < num_reqs:
        if max_query_len <= 0:
            qsl = query_start_loc
            max_query_len = int((qsl[1:] - qsl[:-1]).max().item())
        _C.pooled_window_attention_prefill(
            out, q, k_cache, v_cache, pool_k, pool_v, block_table,
            query_start_loc, seq_lens, gate, scale, window, pool,
            num_decodes, max_query_len)
    return out


# ---------------------------------------------------------------------
# fp32 residual stream with weighted output norms (csrc/residual_ops.hip),
# latent attention with a softmax sink (csrc/latent_attention*.hip),
# state-space-duality mixers (csrc/ssd.hip).

from vllm_amd.ops._torch_ref import softmax_topk_scaled  # noqa: E402,F401


def scaled_embedding(input_ids, table, scale):
    return _C.scaled_embedding(input_ids.contiguous(), table, float(scale))


def rms_norm_cast(x, weight, eps, out_dtype):
    return _C.rms_norm_cast(x.contiguous(), weight, eps, out_dtype)


def add_rms_norm(residual, y, weight, eps, out_dtype=None):
    return _C.add_rms_norm(residual, y.contiguous(), weight, eps, out_dtype)


def relu2(x):
    return _C.relu2(x.contiguous())


def logit_softcap(logits, cap):
    return _C.logit_softcap(logits.contiguous(), float(cap))


def sigmoid_gate_mul(x, gate):
    return _C.sigmoid_gate_mul(x, gate)


def latent_rope_cache_write(q, dkv, norm_w, eps, positions, inv_freq,
                            nope_dim, kv_rank, cache, slot_mapping):
    _C.latent_rope_cache_write(q, dkv, norm_w, eps, positions, inv_freq,
                               nope_dim, kv_rank, cache, slot_mapping)


def latent_attention(q_abs, q_rot, cache, block_table, query_start_loc,
                     seq_lens, scale, sink=None, num_decodes=0,
                     max_seq_len=0, max_query_len=0):
    """bf16 batches whose (kv_rank, rot_dim) the MFMA tile kernel is
    built for run there (prefill chunks and decode rows alike); every
    other dtype and shape runs on the row-wise kernel, which
    VLLM_AMD_LATENT_ROWWISE=1 forces for all."""
    import os

    T, H, L = q_abs.shape
    R = q_rot.shape[2]
    out = torch.empty(T, H, L, dtype=q_abs.dtype, device=q_abs.device)
    if (q_abs.dtype == torch.bfloat16
            and _C.latent_attention_tiles_supported(L, R)
            and os.environ.get("VLLM_AMD_LATENT_ROWWISE", "0") != "1"):
        def aligned(t):
            return (t.stride(0) % 8 == 0 and t.stride(1) % 8 == 0
                    and t.storage_offset() % 8 == 0 and t.stride(2) == 1)
        if not aligned(q_abs):
            q_abs = q_abs.contiguous()
        if R and not aligned(q_rot):
            q_rot = q_rot.contiguous()
        if max_seq_len <= 0:
            max_seq_len = int(seq_lens.max().item())
        _C.latent_attention_tiles(out, q_abs, q_rot, cache, block_table,
                                  query_start_loc, seq_lens, sink, scale,
                                  num_decodes, max_seq_len)
        return out
    _C.latent_attention_rows(out, q_abs, q_rot, cache, block_table,
                             query_start_loc, seq_lens, sink, scale)
    return out


def causal_conv_silu(x, weight, bias, conv_state, state_rows,
                     query_start_loc, out_dtype=None):
    return _C.causal_conv_silu(
        x, weight, bias, conv_state,
        state_rows if conv_state is not None else None, query_start_loc,
        out_dtype or x.dtype)


def ssd_scan(xbc, heads, head_dim, groups, state, dt, dt_bias, a_log,
             d_skip, ssm_state, state_rows, query_start_loc,
             max_query_len=0):
    """max_query_len (a host-side bound on the longest portion) lets
    long portions run as parallel segments; 0 = unknown, sequential."""
    return _C.ssd_scan(
        xbc, heads, head_dim, groups, state, dt.float(), dt_bias, a_log,
        d_skip, ssm_state,
        state_rows if ssm_state is not None else None, query_start_loc,
        max_query_len)


def gated_group_rms_norm(y, z, weight, eps, groups, out_dtype):
    return _C.gated_group_rms_norm(y, z, weight, eps, groups, out_dtype)
