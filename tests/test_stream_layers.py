"""Small steps pass by the modules of a layer only where these do what their
classes say: anything replaced, wrapped or added is called as before."""

import pytest
import torch
import torch.nn as nn

from vllm_amd import ops
from vllm_amd.config import ModelConfig, get_model_spec
from vllm_amd.models.registry import get_model_class
from vllm_amd.worker.forward_context import (
    AttentionMetadata,
    ForwardContext,
    set_forward_context,
)


@pytest.fixture
def net(monkeypatch):
    """A model on the CPU whose steps are all small enough."""
    monkeypatch.setattr(ops, "layer_streams", lambda *args: True)
    name = "tiny-llama-128"
    spec = get_model_spec(name)
    torch.manual_seed(0)
    model = get_model_class(spec.architecture)(
        ModelConfig(model=name, dtype="bf16", max_model_len=64)).eval()
    for p in model.parameters():
        nn.init.normal_(p, std=0.05)
    return model


def _step(model):
    """Three rows that decode, with a hook-free count of fused layers."""
    spec = model.config.spec
    torch.manual_seed(1)
    caches = [torch.randn(2, 3, spec.num_kv_heads, 64,
                          spec.head_dim).bfloat16()
              for _ in range(spec.num_layers)]
    lens = torch.tensor([4, 9, 30], dtype=torch.int32)
    meta = AttentionMetadata(
        query_start_loc=torch.arange(4, dtype=torch.int32), seq_lens=lens,
        block_table=torch.arange(3, dtype=torch.int32)[:, None],
        slot_mapping=torch.arange(3) * 64 + lens.long() - 1, num_reqs=3,
        num_actual_tokens=3, max_query_len=1, max_seq_len=30, num_decodes=3)
    fused = []
    inner = ops.linear_add
    ops.linear_add = lambda *args: fused.append(1) or inner(*args)
    try:
        with torch.inference_mode(), set_forward_context(
                ForwardContext(attn_metadata=meta, kv_caches=caches)):
            out = model(torch.tensor([7, 3, 1]), lens.long() - 1)
    finally:
        ops.linear_add = inner
    return out, caches, len(fused)


def _by_modules(model, monkeypatch):
    """The step as all modules' calls."""
    with monkeypatch.context() as m:
        m.setattr(ops, "layer_streams", lambda *args: False)
        return _step(model)


def _same(got, expect):
    assert got[2] == expect[2] == 0
    assert torch.equal(got[0], expect[0])
    for a, b in zip(got[1], expect[1]):
        assert torch.equal(a, b)


class Wrapped(nn.Module):
    def __init__(self, inner):
        super().__init__()
        self.inner = inner
        self.calls = 0

    def forward(self, *args, **kwargs):
        self.calls += 1
        return self.inner(*args, **kwargs)

    def split_qkv(self, qkv):
        return self.inner.split_qkv(qkv)


PROJECTIONS = ["self_attn.qkv_proj", "self_attn.o_proj", "mlp.gate_up_proj",
               "mlp.down_proj"]


def test_plain_layers_are_passed_by(net, monkeypatch):
    out, caches, fused = _step(net)
    assert fused == 2 * net.config.spec.num_layers
    expect = _by_modules(net, monkeypatch)
    for a, b in [(out, expect[0]), *zip(caches, expect[1])]:
        # A few roundings of 2^-8 apart.
        assert (a - b).norm() <= 2.0 ** -5 * b.norm()


@pytest.mark.parametrize("name", PROJECTIONS)
def test_wrapped_projections_are_called(net, monkeypatch, name):
    layer = net.model.layers[0]
    parent, attr = name.split(".")
    wrapped = Wrapped(layer.get_submodule(name))
    setattr(getattr(layer, parent), attr, wrapped)
    assert not layer.streams()
    got = _step(net)
    assert wrapped.calls == 1
    _same(got, _by_modules(net, monkeypatch))


def test_a_wrapped_rotation_is_called(net, monkeypatch):
    attn = net.model.layers[0].self_attn
    expect = _by_modules(net, monkeypatch)
    attn.rotary_emb = wrapped = Wrapped(attn.rotary_emb)
    got = _by_modules(net, monkeypatch)
    assert wrapped.calls == 1
    _same(got, expect)
    _step(net)
    assert wrapped.calls == 2


@pytest.mark.parametrize("name", PROJECTIONS)
def test_parametrized_weights_are_asked_for(net, monkeypatch, name):
    class Twice(nn.Module):
        def forward(self, w):
            return w * 2

    layer = net.model.layers[0]
    nn.utils.parametrize.register_parametrization(
        layer.get_submodule(name), "weight", Twice())
    assert not layer.streams()
    _same(_step(net), _by_modules(net, monkeypatch))


@pytest.mark.parametrize("name", PROJECTIONS)
def test_adapters_and_fp8_weights_are_not_plain(net, name):
    layer = net.model.layers[0]
    proj = layer.get_submodule(name)
    assert layer.streams()
    proj.lora_slices = [(0, 8, "a")]
    assert not layer.streams()
    proj.lora_slices = None
    assert layer.streams()
    proj.quantize_fp8()
    assert not layer.streams()


@pytest.mark.parametrize("name", PROJECTIONS + [
    "self_attn", "mlp", "mlp.act_fn", "input_layernorm",
    "post_attention_layernorm"])
def test_functions_in_the_place_of_modules_are_called(net, monkeypatch, name):
    layer = net.model.layers[0]
    parent, _, attr = name.rpartition(".")
    parent = layer.get_submodule(parent)
    module, calls = layer.get_submodule(name), []
    class Function:
        def __call__(self, *args, **kwargs):
            calls.append(1)
            return module(*args, **kwargs)

        def __getattr__(self, what):
            return getattr(module, what)

    delattr(parent, attr)
    setattr(parent, attr, Function())
    got = _step(net)
    assert len(calls) == 1
    _same(got, _by_modules(net, monkeypatch))


MODULES = PROJECTIONS + ["", "self_attn", "self_attn.attn",
                         "self_attn.rotary_emb", "mlp", "mlp.act_fn",
                         "input_layernorm", "post_attention_layernorm"]
# Called with what they are called with by the layer's modules, beside
# products that take norms and sums along.
BESIDE = ["self_attn.attn", "self_attn.rotary_emb"]


@pytest.mark.parametrize("name", MODULES)
def test_replaced_forwards_are_called(net, monkeypatch, name):
    module = net.model.layers[0].get_submodule(name)
    calls, inner = [], module.forward
    module.forward = lambda *a, **kw: calls.append(1) or inner(*a, **kw)
    got = _step(net)
    assert len(calls) == 1
    if name not in BESIDE:
        _same(got, _by_modules(net, monkeypatch))


@pytest.mark.parametrize("name", MODULES)
def test_replaced_forwards_of_classes_are_called(net, monkeypatch, name):
    cls = type(net.model.layers[0].get_submodule(name))
    calls, inner = [], cls.forward
    monkeypatch.setattr(
        cls, "forward", lambda *a, **kw: calls.append(1) or inner(*a, **kw))
    got = _step(net)
    assert len(calls) >= net.config.spec.num_layers
    if name not in BESIDE:
        _same(got, _by_modules(net, monkeypatch))


def test_layers_of_other_classes_are_called(net, monkeypatch):
    from vllm_amd.models.llama import LlamaDecoderLayer

    class Scaled(LlamaDecoderLayer):
        def forward(self, positions, hidden, residual):
            hidden, residual = super().forward(positions, hidden, residual)
            return hidden * 0.5, residual

    net.model.layers[0].__class__ = Scaled
    _same(_step(net), _by_modules(net, monkeypatch))
    wrapped = net.model.layers[0] = Wrapped(net.model.layers[0])
    _same(_step(net), _by_modules(net, monkeypatch))
    assert wrapped.calls == 2


@pytest.mark.parametrize("change", ["hook", "forward", "wrap"])
def test_the_last_norm_is_called_as_before(net, monkeypatch, change):
    """With the sublayer's output and the residual apart."""
    seen = []
    norm = net.model.norm
    if change == "hook":
        norm.register_forward_pre_hook(lambda m, args: seen.append(len(args)))
    elif change == "forward":
        norm.forward = lambda *args: seen.append(len(args)) or type(
            norm).forward(norm, *args)
    else:
        net.model.norm = Wrapped(norm)
        norm.register_forward_pre_hook(lambda m, args: seen.append(len(args)))
    got = _step(net)
    assert seen == [2]
    _same(got, _by_modules(net, monkeypatch))


@pytest.mark.parametrize("name", ["q_a_proj", "kv_a_proj_with_mqa",
                                  "kv_a_layernorm", "rotary_emb"])
def test_wrapped_modules_of_latent_attention_are_called(name):
    from vllm_amd.models.deepseek import DeepseekMLAAttention

    spec = get_model_spec("tiny-deepseek")
    torch.manual_seed(0)
    block = DeepseekMLAAttention(spec, 0, torch.float32, 64)
    for p in block.parameters():
        nn.init.normal_(p, std=0.05)

    def step():
        torch.manual_seed(1)
        cache = torch.randn(2, 64, spec.kv_lora_rank + spec.qk_rope_head_dim)
        meta = AttentionMetadata(
            query_start_loc=torch.arange(3, dtype=torch.int32),
            seq_lens=torch.tensor([4, 9], dtype=torch.int32),
            block_table=torch.tensor([[0], [1]], dtype=torch.int32),
            slot_mapping=torch.tensor([3, 64 + 8]), num_reqs=2,
            num_actual_tokens=2, max_query_len=1, max_seq_len=9,
            num_decodes=2)
        x = torch.randn(2, spec.hidden_size)
        with torch.inference_mode(), set_forward_context(
                ForwardContext(attn_metadata=meta, kv_caches=[cache])):
            return block(torch.tensor([3, 8]), x), cache

    expect = step()
    wrapped = Wrapped(getattr(block, name))
    setattr(block, name, wrapped)
    got = step()
    assert wrapped.calls == 1
    for a, b in zip(got, expect):
        torch.testing.assert_close(a, b)

    class OnGpu(torch.Tensor):
        """Takes the path that GPU tensors take."""
        is_cuda = True

    block._a_projs(torch.randn(2, spec.hidden_size).as_subclass(OnGpu))
    block.double()
