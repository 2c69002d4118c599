"""Which blocks may run a decode step's linear layers through the fused calls
(TransformerBlock._plain_decode): a predicate over the modules, so it is checked
without a GPU."""
from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F
from torch import nn

from minivllm import decode_fused
from minivllm.attention import KVCacheCausalSelfAttention
from minivllm.block import TransformerBlock
from minivllm.decode_batch_metadata import DecodeBatchMetadata
from minivllm.feed_forward import FeedForward
from minivllm.kv_block_pool import KVBlockPool
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


@pytest.mark.parametrize("cls", [nn.Linear, nn.LayerNorm, nn.GELU, nn.Dropout, nn.Sequential, FeedForward])
def test_a_replaced_class_method_is_called(cls, monkeypatch):
    """A forward replaced on the class (as quantisers and profilers do) runs in
    a decode step; so does a replaced __call__."""
    forward = cls.forward
    assert decode_fused.unpatched()
    monkeypatch.setattr(cls, "forward", lambda self, *a, **kw: forward(self, *a, **kw))
    assert not decode_fused.unpatched()
    monkeypatch.undo()
    assert decode_fused.unpatched()
    monkeypatch.setattr(cls, "__call__", lambda self, *a, **kw: forward(self, *a, **kw), raising=False)
    assert not decode_fused.unpatched()
    monkeypatch.undo()
    assert decode_fused.unpatched()


@pytest.mark.parametrize("owner,name", [
    (F, "linear"), (F, "layer_norm"), (F, "gelu"), (F, "dropout"), (nn.Module, "_call_impl"), (nn.Module, "__call__"),
    (TransformerBlock, "_mlp"), (TransformerBlock, "forward_decode_batch"), (KVCacheCausalSelfAttention, "_qkv_heads"),
    (KVCacheCausalSelfAttention, "_finish"), (KVCacheCausalSelfAttention, "forward_decode_batch")])
def test_a_replaced_function_is_called(owner, name, monkeypatch):
    assert decode_fused.unpatched()
    function = getattr(owner, name)
    monkeypatch.setattr(owner, name, lambda *a, **kw: function(*a, **kw))
    assert not decode_fused.unpatched()
    monkeypatch.undo()
    assert decode_fused.unpatched()


@pytest.mark.parametrize("path,name", [("attn.project", "forward"), ("ffn", "forward"), ("attn", "_finish"), ("", "_mlp")])
def test_a_method_replaced_on_one_module_is_called(block, path, name):
    m = block.get_submodule(path)
    assert block._plain_decode(64)
    setattr(m, name, lambda *a, **kw: None)
    assert not block._plain_decode(64)
    delattr(m, name)
    assert block._plain_decode(64)


@pytest.mark.parametrize("path", ["attn.project", "ffn.network.0", "ffn.network.2", "layer_norm_1", "layer_norm_2"])
@pytest.mark.parametrize("name", ["weight", "bias"])
def test_attributes_in_place_of_parameters_are_used(block, path, name):
    """A weight or bias taken out of the parameters and set as a plain tensor
    (or put over the parameter in the module's dict) is what the module's
    forward reads; a bias so placed must not be taken for none."""
    m = block.get_submodule(path)
    p = m._parameters.pop(name)
    object.__setattr__(m, name, p.detach() + 1)
    assert not block._plain_decode(64)
    m._parameters[name] = p
    assert not block._plain_decode(64)
    object.__delattr__(m, name)
    assert block._plain_decode(64)
    m._parameters.pop(name)
    m.register_buffer(name, p.detach() + 1)
    assert not block._plain_decode(64)


def test_a_linear_without_bias_stays_plain(block):
    block.attn.project = nn.Linear(64, 64, bias=False)
    assert block._plain_decode(64)
    block.attn.project.bias = nn.Parameter(torch.zeros(64))
    assert block._plain_decode(64)


class TorchOps:
    """The binding's two calls in PyTorch, refusing those whose weight is in ``refused``."""

    def __init__(self, refused=()):
        self.refused = {id(w) for w in refused}

    def decode_linear(self, x, w, bias, gelu):
        if id(w) in self.refused:
            return None
        y = F.linear(x, w, bias)
        return F.gelu(y) if gelu else y

    def decode_linear_norm(self, x, w, bias, residual, ln_w, ln_b, eps):
        if id(w) in self.refused:
            return None
        h = residual if x is None else F.linear(x, w, bias) + residual
        return h, None if ln_w is None else F.layer_norm(h, (h.shape[-1],), ln_w, ln_b, eps)


@pytest.mark.parametrize("refused", [(), ("attn.qkv",), ("attn.project",), ("ffn.network.0",), ("ffn.network.2",),
                                     ("attn.qkv", "ffn.network.0", "ffn.network.2")])
def test_step_with_layers_the_kernels_do_not_take(block, refused):
    """A block's fused step, each of its layers refused in turn, against the
    block's own PyTorch calls: the same output and appended KV, and no layer
    made twice."""
    g = torch.Generator().manual_seed(1)
    x = torch.randn((3, 1, 64), generator=g)
    ctx, tables = torch.tensor([5, 9, 1]), torch.tensor([[2, -1], [0, 3], [1, -1]])
    slots = tables[torch.arange(3), (ctx - 1) // 8] * 8 + (ctx - 1) % 8
    meta = DecodeBatchMetadata(positions=ctx - 1, context_lengths=ctx, block_tables=tables, slot_mapping=slots)
    pools = [KVBlockPool(1, 4, 8, 2, 32) for _ in range(2)]
    for p in pools:
        p.k.copy_(torch.randn(p.k.shape, generator=torch.Generator().manual_seed(2)))
        p.v.copy_(torch.randn(p.v.shape, generator=torch.Generator().manual_seed(3)))
    after = nn.LayerNorm(64)
    ops = TorchOps([block.get_submodule(p).weight for p in refused])
    calls = []
    for p in ("attn.qkv", "attn.project", "ffn.network.0", "ffn.network.2"):
        block.get_submodule(p).register_forward_hook(lambda *a, p=p: calls.append(p))
    with torch.no_grad():
        want = block.forward_decode_batch(x, metadata=meta, kv_pool=pools[0], layer_idx=0)
        assert calls == ["attn.qkv", "attn.project", "ffn.network.0", "ffn.network.2"]
        calls.clear()
        out, normed = block._decode_step(ops, x, None, after, meta, pools[1], 0)
    torch.testing.assert_close(out, want, rtol=1e-6, atol=1e-6)
    assert torch.equal(pools[0].k, pools[1].k) and torch.equal(pools[0].v, pools[1].v)
    if normed is not None:
        torch.testing.assert_close(normed, after(out), rtol=1e-6, atol=1e-6)
    # Without the fused sum after the attention, the MLP is the block's own.
    assert calls == (["attn.project", "ffn.network.0", "ffn.network.2"] if refused == ("attn.project",) else list(refused))
