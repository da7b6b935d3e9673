"""Experts of few rows: weights streamed past them (csrc/moe_rows.h), by
themselves and among tiles, against 64 bits."""

import pytest
import torch

pytestmark = pytest.mark.gpu


# Rows of each expert: ends of the 8-, 16-, 32- and 64-row forms, none, more
# than a tile; a last row group that ends within a tile of an expert.
@pytest.mark.parametrize("counts,H,I,act", [
    ([1, 0, 0], 64, 64, "silu"),                  # one step, narrow
    ([8, 9, 16, 17, 0, 32, 33, 64], 576, 320, "silu"),
    ([65, 1, 64, 0], 128, 192, "relu2"),
    ([3] * 40, 512, 1024, "silu"),                # wide
    ([7, 20, 2, 64], 2048, 4096, "relu2"),
    ([32, 33, 1, 200, 31], 256, 192, "silu"),     # 128-row tiles
    ([30, 600, 290, 0, 17], 256, 192, "silu"),    # 256-row tiles
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_rows(counts, H, I, act, dtype):
    from vllm_amd.ops import hip_ops
    torch.manual_seed(len(counts) + H)
    E = len(counts)
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))
    ids = ids[torch.randperm(len(ids))].to(torch.int32).cuda()[:, None]
    T, g = len(ids), 2 if act == "silu" else 1
    x = torch.randn(T, H, device="cuda", dtype=dtype)
    w13 = torch.randn(E, g * I, H, device="cuda", dtype=dtype) * H ** -0.5
    w2 = torch.randn(E, H, I, device="cuda", dtype=dtype) * I ** -0.5
    tw = torch.rand(T, 1, device="cuda")
    out = hip_ops.fused_moe_hip(x, w13, w2, tw, ids, activation=act).double()
    # Rounding to p significant bits is off by 2^-p of the value (p = 8, 11):
    # the activation, the expert's output and the weighted result.
    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    for e in range(E):
        t = (ids[:, 0] == e).nonzero()[:, 0]
        y = x[t].double() @ w13[e].double().T
        a = (torch.nn.functional.silu(y[:, :I]) * y[:, I:] if g == 2
             else y.relu() ** 2)
        w = tw[t].double()
        y, mag = a @ w2[e].double().T, a.abs() @ w2[e].double().abs().T
        bound = 1.1 * eps * w * (mag + 2 * y.abs()) + 2.0 ** -20
        assert ((out[t] - w * y).abs() <= bound).all(), e
