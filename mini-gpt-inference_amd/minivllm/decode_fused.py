"""A decode step's linear layers through the HIP kernels of decode_linear.hip.

The reference runs LayerNorm, each projection, GELU and the residual sums as
separate PyTorch calls (minivllm/block.py:72-93, minivllm/feed_forward.py:3-28).
For up to 64 rows of a bf16 or f16 model on a GPU these are launch- and
weight-bandwidth-bound, so TransformerBlock.forward_decode_batch and
MiniGPT.decode_batch hand them to four calls per block (six launches):
QKV projection; output projection + residual + LayerNorm; first MLP layer +
GELU; second MLP layer + residual + the next LayerNorm. Sums are fp32 and each
stored tensor is rounded once, so nothing is less precise than the PyTorch
calls; the bits differ.

Whether a call may take this route is decided on every call from the tensors
(in the binding, which returns None for what the kernels do not take) and the
modules: only the plain module classes, without hooks, replaced methods (the
module's, its class's or the torch functions' they end in), active dropout,
autocast, gradients, tracing or transforms. Everything else makes the PyTorch
calls, and so does a block whose ``fused_decode_linears`` is False. The choice
does not depend on the attention backend, so that switching the backend changes
the attention alone.
"""
from __future__ import annotations

import torch
import torch.nn.functional as F
from torch import Tensor, nn
from torch.autograd import forward_ad
from torch.nn.modules import module as _nn_module

from . import _native
from .feed_forward import FeedForward

MAX_ROWS = 64
_DTYPES = (torch.bfloat16, torch.float16)


def ops_for(x: Tensor):
    """The binding, when a decode step on x may use it; else None."""
    if type(x) is not Tensor or x.dtype not in _DTYPES or not x.is_cuda or x.dim() != 3 or x.shape[1] != 1 \
            or not 1 <= x.shape[0] <= MAX_ROWS:
        return None
    if torch.is_grad_enabled() or torch.is_autocast_enabled("cuda") or torch.jit.is_tracing() \
            or torch.compiler.is_compiling() or forward_ad._current_level >= 0 \
            or torch._C._len_torch_dispatch_stack() or torch._C._len_torch_function_stack() \
            or torch._C._functorch.peek_interpreter_stack() is not None \
            or _nn_module._global_forward_hooks or _nn_module._global_forward_pre_hooks or not unpatched():
        return None
    try:
        ops = _native.ops()
    except RuntimeError:
        return None  # no library: the attention backend says so if it needs one
    return ops if hasattr(ops, "decode_linear") else None


def unpatched() -> bool:
    """Whether the methods and torch functions the fused calls stand for are the
    ones this package was imported with (once per step: they belong to classes
    and modules, not to a model)."""
    for owner, name, function in _OWN:
        if getattr(owner, name) is not function:
            return False
    return True


def own_methods(cls: type, names: tuple[str, ...]) -> None:
    """Adds cls's methods to what unpatched checks."""
    _OWN.extend((cls, n, getattr(cls, n)) for n in names)


def plain(m: nn.Module, cls: type) -> bool:
    """Whether calling m runs cls's forward and nothing else, on parameters where
    it has any: no hooks, and no forward, weight or bias in m's own dict."""
    d = m.__dict__
    return type(m) is cls and not d["_forward_hooks"] and not d["_forward_pre_hooks"] \
        and "forward" not in d and "weight" not in d and "bias" not in d


def plain_linear(m: nn.Module) -> bool:
    if not plain(m, nn.Linear):
        return False
    p = m._parameters
    return type(p.get("weight")) is nn.Parameter and "bias" in p and type(p["bias"]) in _PARAMS


def plain_norm(m: nn.Module, width: int) -> bool:
    if not plain(m, nn.LayerNorm) or m.normalized_shape != (width,):
        return False
    p = m._parameters
    return type(p.get("weight")) is nn.Parameter and type(p.get("bias")) is nn.Parameter


def idle_dropout(m: nn.Module) -> bool:
    return plain(m, nn.Dropout) and not (m.training and m.p > 0.0)


_PARAMS = (nn.Parameter, type(None))
_OWN = [(nn.Module, "__call__", nn.Module.__call__), (nn.Module, "_call_impl", nn.Module._call_impl)]
_OWN += [(F, n, getattr(F, n)) for n in ("linear", "layer_norm", "gelu", "dropout")]
for _cls in (nn.Linear, nn.LayerNorm, nn.GELU, nn.Dropout, nn.Sequential, FeedForward):
    # A forward from elsewhere than its class's module was patched before this import: nothing is None.
    _OWN += [(_cls, "forward", _cls.forward if _cls.forward.__module__ == _cls.__module__ else None),
             (_cls, "__call__", nn.Module.__call__)]
