"""Which blocks may run a decode step's linear layers through the fused calls
(TransformerBlock._plain_decode): a predicate over the modules, so it is checked
without a GPU."""
from __future__ import annotations

import pytest

from minivllm.block import TransformerBlock
from minivllm.model import MiniGPT


@pytest.fixture
def block():
    return TransformerBlock(64, 2, 32).eval()


def test_switch_keeps_the_pytorch_calls(block):
    assert block._plain_decode(64)
    block.fused_decode_linears = False
    assert not block._plain_decode(64)
    block.fused_decode_linears = True
    assert block._plain_decode(64) and not block._plain_decode(128)


@pytest.mark.parametrize("backend", ["reference", "hip", "triton_v0"])
def test_the_attention_backend_does_not_choose(backend):
    model = MiniGPT(n_embd=64, n_head=2, vocab_size=16, block_size=32, n_layer=2).eval()
    model.set_decode_attention_backend(backend)
    assert all(b._plain_decode(64) for b in model.blocks)
    assert not any("fused_decode" in k for k in model.state_dict())
