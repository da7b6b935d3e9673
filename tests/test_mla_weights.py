"""The MLA block keeps the weights of its two projections of the hidden
state one behind the other; what a model's user does to its parameters
works as for any other."""

import pytest
import torch

from vllm_amd.config import get_model_spec
from vllm_amd.models.deepseek import DeepseekMLAAttention


@pytest.fixture
def block():
    b = DeepseekMLAAttention(get_model_spec("tiny-deepseek"), 0,
                             torch.float32, 64)
    for p in b.parameters():
        torch.nn.init.normal_(p)
    return b


def _weights(b):
    return b.q_a_proj.weight, b.kv_a_proj_with_mqa.weight


def test_moves_that_change_nothing_keep_storage(block):
    before = [w.data_ptr() for w in _weights(block)]
    block.to("cpu")
    block.to(torch.float32)
    block.float()
    assert [w.data_ptr() for w in _weights(block)] == before


def test_shared_memory_is_kept(block):
    values = [w.clone() for w in _weights(block)]
    block.share_memory()
    for w, v in zip(_weights(block), values):
        assert w.is_shared() and torch.equal(w, v)
    assert block._joined_a_projs() is not None


def test_other_types_are_joined_again(block):
    values = [w.clone() for w in _weights(block)]
    block.to(torch.bfloat16)
    both = block._joined_a_projs()
    assert torch.equal(both, torch.cat(values).to(torch.bfloat16))
    q, kv = _weights(block)
    kv.data = kv.data.clone()
    assert block._joined_a_projs() is None
