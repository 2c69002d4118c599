"""Pre-LN transformer block of MiniGPT (minivllm/block.py:6-102):
x + attn(LN1(x)), then x + ffn(LN2(x)), for each execution mode."""
from __future__ import annotations

from torch import Tensor, nn

from . import decode_fused
from .attention import KVCacheCausalSelfAttention, plain_decode_attention
from .decode_batch_metadata import DecodeBatchMetadata
from .feed_forward import FeedForward
from .kv_block_pool import KVBlockPool
from .kv_runtime import KVRuntimeContext, PrefillChunkContext, PrefillRuntimeContext


class TransformerBlock(nn.Module):
    def __init__(self, n_embd: int, n_head: int, block_size: int, dropout: float = 0.0):
        super().__init__()
        if n_embd <= 0:
            raise ValueError("n_embd must be > 0")
        if n_head <= 0:
            raise ValueError("n_head must be > 0")
        self.attn = KVCacheCausalSelfAttention(n_embd, n_head, block_size, dropout)
        self.ffn = FeedForward(n_embd, dropout)
        self.layer_norm_1 = nn.LayerNorm(n_embd)
        self.layer_norm_2 = nn.LayerNorm(n_embd)

    # False: decode steps make the PyTorch calls for this block's norms, projections and MLP (and, on a model's last
    # block, for the final norm and the LM head), whatever the attention backend.
    fused_decode_linears = True

    def _mlp(self, x: Tensor) -> Tensor:
        return x + self.ffn(self.layer_norm_2(x))

    def forward_prefill(self, x: Tensor, context: PrefillRuntimeContext) -> Tensor:
        return self._mlp(x + self.attn.forward_prefill(self.layer_norm_1(x), context))

    def forward_prefill_chunk(self, x: Tensor, context: PrefillChunkContext) -> Tensor:
        return self._mlp(x + self.attn.forward_prefill_chunk(self.layer_norm_1(x), context))

    def forward_decode(self, x: Tensor, kv_context: KVRuntimeContext) -> Tensor:
        return self._mlp(x + self.attn.forward_decode(self.layer_norm_1(x), kv_context=kv_context))

    def forward_decode_batch(self, x: Tensor, metadata: DecodeBatchMetadata, kv_pool: KVBlockPool,
                             layer_idx: int) -> Tensor:
        ops = decode_fused.ops_for(x)
        if ops is not None and self._plain_decode(x.shape[2]):
            fused = self._decode_step(ops, x, None, None, metadata, kv_pool, layer_idx)
            if fused is not None:
                return fused[0]
        h = self.attn.forward_decode_batch(self.layer_norm_1(x), metadata=metadata, kv_pool=kv_pool,
                                           layer_idx=layer_idx)
        return self._mlp(x + h)

    def _plain_decode(self, width: int) -> bool:
        """Whether forward_decode_batch is this module's own code over plain
        submodules (decode_fused)."""
        m = self._modules
        if not self.fused_decode_linears or type(self) is not TransformerBlock \
                or not self.__dict__.keys().isdisjoint(_DECODE_METHODS) \
                or not plain_decode_attention(m["attn"]) or m["attn"].n_embd != width:
            return False
        ffn = m["ffn"]
        net = ffn._modules["network"] if decode_fused.plain(ffn, FeedForward) else None
        if net is None or not decode_fused.plain(net, nn.Sequential) or len(net) != 4:
            return False
        up, act, down, drop = (net._modules.get(i) for i in "0123")
        return decode_fused.plain_norm(m["layer_norm_1"], width) and decode_fused.plain_norm(m["layer_norm_2"], width) \
            and decode_fused.plain_linear(up) and decode_fused.plain(act, nn.GELU) and act.approximate == "none" \
            and decode_fused.plain_linear(down) and decode_fused.idle_dropout(drop)

    def _decode_step(self, ops, x: Tensor, normed: Tensor | None, next_norm: nn.LayerNorm | None,
                     metadata: DecodeBatchMetadata, kv_pool: KVBlockPool, layer_idx: int):
        """forward_decode_batch through the fused linear calls: (output,
        next_norm(output) or None). ``normed`` is layer_norm_1(x) when the caller
        has it. None, with nothing done, when the kernels do not take x; a layer
        they do not take is made with PyTorch."""
        m = self._modules
        attn = m["attn"]
        n1, n2 = m["layer_norm_1"], m["layer_norm_2"]
        net = m["ffn"]._modules["network"]._modules
        up, down = net["0"]._parameters, net["2"]._parameters
        project = attn._modules["project"]._parameters
        if normed is None:
            p = n1._parameters
            first = ops.decode_linear_norm(None, None, None, x, p["weight"], p["bias"], n1.eps)
            if first is None:
                return None
            normed = first[1]
        qkv = attn._modules["qkv"]
        heads = ops.decode_linear(normed, qkv._parameters["weight"], qkv._parameters["bias"], False)
        if heads is None:
            heads = qkv(normed)
        q, k, v = heads.view(-1, 3, attn.n_head, attn.head_size).unbind(1)
        a = attn._decode_attend(q, k, v, metadata, kv_pool, layer_idx)
        p = n2._parameters
        pair = ops.decode_linear_norm(a, project["weight"], project["bias"], x, p["weight"], p["bias"], n2.eps)
        if pair is None:
            return self._mlp(x + attn._finish(a)), None
        h, y = pair
        u = ops.decode_linear(y, up["weight"], up["bias"], True)
        if u is None:
            u = net["1"](net["0"](y))
        if next_norm is None:
            pair = ops.decode_linear_norm(u, down["weight"], down["bias"], h, None, None, 0.0)
        else:
            p = next_norm._parameters
            pair = ops.decode_linear_norm(u, down["weight"], down["bias"], h, p["weight"], p["bias"], next_norm.eps)
        return (h + net["3"](net["2"](u)), None) if pair is None else pair

    def forward(self, x: Tensor) -> Tensor:
        return self._mlp(x + self.attn(self.layer_norm_1(x)))


_DECODE_METHODS = ("forward_decode_batch", "_mlp", "_plain_decode", "_decode_step")
decode_fused.own_methods(TransformerBlock, _DECODE_METHODS)
