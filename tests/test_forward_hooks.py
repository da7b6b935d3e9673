"""Forward hooks fire on modules that a fused pass would otherwise leave
out, and results stay what they are without hooks."""

import pytest
import torch

from vllm_amd.config import ModelConfig, get_model_spec
from vllm_amd.models.registry import get_model_class
from vllm_amd.worker.forward_context import (
    AttentionMetadata,
    ForwardContext,
    set_forward_context,
)

DEVICES = ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)]


def _run(model, spec, device, dtype):
    """A prompt of 5 tokens beside a row that decodes its 4th."""
    torch.manual_seed(1)
    if spec.is_mla:
        shape = (3, 64, spec.kv_lora_rank + spec.qk_rope_head_dim)
    else:
        shape = (2, 3, spec.num_kv_heads, 64, spec.head_dim)
    caches = [torch.randn(shape).to(device, dtype)
              for _ in range(spec.num_layers)]

    def ints(x, dtype=torch.int32):
        return torch.tensor(x, dtype=dtype, device=device)

    meta = AttentionMetadata(
        query_start_loc=ints([0, 1, 6]), seq_lens=ints([4, 5]),
        block_table=ints([[1], [2]]),
        slot_mapping=ints([64 + 3] + [128 + i for i in range(5)],
                          torch.int64),
        num_reqs=2, num_actual_tokens=6, max_query_len=5, max_seq_len=5,
        num_decodes=1)
    ids = ints([7, 3, 1, 4, 1, 5], torch.int64)
    pos = ints([3, 0, 1, 2, 3, 4], torch.int64)
    ctx = ForwardContext(attn_metadata=meta, kv_caches=caches)
    with torch.inference_mode(), set_forward_context(ctx):
        return model(ids, pos), caches


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("name,modules", [
    ("tiny-llama-128", ["rotary_emb"]),
    ("tiny-deepseek", ["rotary_emb", "kv_a_layernorm", "q_a_proj",
                       "kv_a_proj_with_mqa"]),
])
def test_hooks_fire(name, modules, device):
    """Every named module of a layer is called once a pass. The modules
    compute what the fused pass does: CPU results are the same to the last
    bit, 16-bit ones within a few roundings (2^-8 each) of activations."""
    dtype = torch.float32 if device == "cpu" else torch.bfloat16
    spec = get_model_spec(name)
    config = ModelConfig(model=name, dtype="fp32" if device == "cpu"
                         else "bf16", max_model_len=64)
    torch.manual_seed(0)
    with torch.device(device):
        model = get_model_class(spec.architecture)(config).eval()
    for p in model.parameters():
        torch.nn.init.normal_(p, std=0.05)
    plain, plain_caches = _run(model, spec, device, dtype)
    for module in modules:
        calls = []
        handles = [m.register_forward_hook(lambda *a: calls.append(1))
                   for n, m in model.named_modules()
                   if n.split(".")[-1] == module]
        out, caches = _run(model, spec, device, dtype)
        assert len(calls) == len(handles) > 0, module
        for h in handles:
            h.remove()
        tol = 0 if device == "cpu" else 2**-5
        for a, b in [(out, plain), *zip(caches, plain_caches)]:
            torch.testing.assert_close(a, b, rtol=tol, atol=tol)


def test_bias_of_joined_projections():
    """A bias on one of the two projections of an MLA block's hidden state
    is added, wherever their weights lie."""
    from vllm_amd.models.deepseek import DeepseekMLAAttention

    spec = get_model_spec("tiny-deepseek")
    block = DeepseekMLAAttention(spec, 0, torch.float32, 64)
    for p in block.parameters():
        torch.nn.init.normal_(p)
    block.kv_a_proj_with_mqa.bias = torch.nn.Parameter(
        torch.ones(block.kv_a_proj_with_mqa.weight.shape[0]),
        requires_grad=False)
    assert block._joined_a_projs() is not None

    class OnGpu(torch.Tensor):
        """Takes the path that GPU tensors take."""
        is_cuda = True

    x = torch.randn(3, spec.hidden_size)
    _, kv = block._a_projs(x.as_subclass(OnGpu))
    expect = x @ block.kv_a_proj_with_mqa.weight.T + 1
    torch.testing.assert_close(kv.as_subclass(torch.Tensor), expect)
