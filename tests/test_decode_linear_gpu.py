"""The decode step's linear kernels (decode_linear.hip) on the MI355X against
float64, at the sizes where their division can go wrong: row counts around the
16-row blocks, column counts around a tile and a split's 64, K from one unit
to the widest, odd column counts; the block and model steps they make against
the PyTorch calls; and the modules and contexts that must keep those calls."""
from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F
from torch import nn

from minivllm import _native, decode_fused
from minivllm.block import TransformerBlock
from minivllm.decode_batch_metadata import DecodeBatchMetadata
from minivllm.kv_block_pool import KVBlockPool
from minivllm.model import MiniGPT

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
# One rounding of the stored result (half an ulp, 2^-9 and 2^-12 relative) plus f32
# sums of K products in another order (K 2^-24 of the terms' magnitude): together
# below one ulp of the largest output, 2^-8 and 2^-11. A LayerNorm is compared with
# the float64 one of the row as it was stored, so it is one rounding too.
ULP = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}
DTYPES = [torch.bfloat16, torch.float16]


def rnd(g, *shape, dtype, scale=1.0, shift=0.0):
    return (torch.randn(shape, generator=g, device=DEV) * scale + shift).to(dtype)


def close(got, want, ulps, dtype):
    assert got.dtype == dtype
    err = (got.double() - want).abs().max().item()
    assert err <= ulps * ULP[dtype] * max(1.0, want.abs().max().item()), err


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("K,N", [(64, 16), (128, 17), (512, 1536), (768, 100), (1280, 4099), (2048, 8192), (2560, 48)])
def test_decode_linear(K, N, dtype):
    ops = _native.ops()
    g = torch.Generator(device=DEV).manual_seed(K + N)
    w = rnd(g, N, K, dtype=dtype, scale=K ** -0.5)
    bias = rnd(g, N, dtype=dtype)
    for B in (1, 15, 16, 17, 32, 33, 48, 64):
        x = rnd(g, B, 1, K, dtype=dtype)
        for b, gelu in ((bias, True), (None, False)):
            print(f"  linear B={B} K={K} N={N} {dtype} gelu={gelu}", flush=True)
            y = ops.decode_linear(x, w, b, gelu)
            if B > 48 and K > 1536 and not gelu:
                assert y is None
                continue
            assert _native.lib().mgi_decode_linear_pays(B, N, K, gelu) == 1
            want = x.double() @ w.double().t().contiguous() + (0 if b is None else b.double())
            close(y, F.gelu(want) if gelu else want, 1, dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("K,N", [(64, 64), (576, 68), (512, 512), (3072, 768), (8192, 2048), (10240, 2560), (1024, 4096)])
def test_decode_linear_norm(K, N, dtype):
    ops = _native.ops()
    g = torch.Generator(device=DEV).manual_seed(K + N)
    w = rnd(g, N, K, dtype=dtype, scale=K ** -0.5)
    bias, lw, lb = rnd(g, N, dtype=dtype), rnd(g, N, dtype=dtype), rnd(g, N, dtype=dtype)
    for B in (1, 16, 17, 33, 64):
        print(f"  linear+norm B={B} K={K} N={N} {dtype}", flush=True)
        x, r = rnd(g, B, 1, K, dtype=dtype), rnd(g, B, 1, N, dtype=dtype, shift=3.0)
        h, y = ops.decode_linear_norm(x, w, bias, r, lw, lb, 1e-5)
        want = x.double() @ w.double().t().contiguous() + bias.double() + r.double()
        close(h, want, 1, dtype)
        close(y, F.layer_norm(h.double(), (N,), lw.double(), lb.double(), 1e-5), 1, dtype)
        again, none = ops.decode_linear_norm(x, w, bias, r, None, None, 0.0)
        assert none is None and torch.equal(again, h)
        same, alone = ops.decode_linear_norm(None, None, None, r, lw, lb, 1e-5)
        assert same.data_ptr() == r.data_ptr()
        close(alone, F.layer_norm(r.double(), (N,), lw.double(), lb.double(), 1e-5), 1, dtype)


def test_calls_the_kernels_do_not_take_return_none():
    ops = _native.ops()
    x, w = torch.zeros(4, 1, 128, device=DEV, dtype=torch.bfloat16), torch.zeros(64, 128, device=DEV, dtype=torch.bfloat16)
    assert ops.decode_linear(x, w, None, False) is not None
    for bx, bw in ((x.float(), w.float()), (x, w.half()), (x.expand(4, 2, 128), w), (x[..., :96], w[:, :96]),
                   (x, w.t().contiguous().t()), (torch.zeros(65, 1, 128, device=DEV, dtype=torch.bfloat16), w),
                   (x.cpu(), w), (x, w.cpu()), (x[..., :64], w[:, :64]), (x.flatten()[4:].clone().view(-1, 1, 127), w)):
        assert ops.decode_linear(bx, bw, None, False) is None
    assert ops.decode_linear(x, w, torch.zeros(63, device=DEV, dtype=torch.bfloat16), False) is None
    r = torch.zeros(4, 1, 64, device=DEV, dtype=torch.bfloat16)
    assert ops.decode_linear_norm(x, w, None, r, None, None, 0.0) is not None
    assert ops.decode_linear_norm(x, w, None, r[:3], None, None, 0.0) is None
    assert ops.decode_linear_norm(x, w, None, r, torch.zeros(64, device=DEV), torch.zeros(64, device=DEV), 1e-5) is None


def _step(B, H, D, dtype, layers=2, vocab=333, seed=1):
    torch.manual_seed(seed)
    model = MiniGPT(n_embd=H * D, n_head=H, vocab_size=vocab, block_size=256, n_layer=layers).eval().to(DEV, dtype)
    model.set_decode_attention_backend("hip")
    S, M = 16, 8
    tables = torch.randperm(B * M, generator=torch.Generator().manual_seed(seed)).view(B, M)
    ctx = torch.randint(1, M * S, (B,), generator=torch.Generator().manual_seed(seed + 1))
    slots = tables[torch.arange(B), (ctx - 1) // S] * S + (ctx - 1) % S
    meta = DecodeBatchMetadata(positions=(ctx - 1).to(DEV), context_lengths=ctx.to(DEV), block_tables=tables.to(DEV),
                               slot_mapping=slots.to(DEV))
    ids = torch.randint(0, vocab, (B, 1), generator=torch.Generator().manual_seed(seed + 2)).to(DEV)

    def run():
        pool = KVBlockPool(layers, B * M, S, H, D, device=DEV, dtype=dtype)
        g = torch.Generator(device=DEV).manual_seed(seed)
        pool.k.normal_(generator=g)
        pool.v.normal_(generator=g)
        return model.decode_batch(ids, meta, pool), pool

    return model, run, (ids, meta)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("B,H,D", [(1, 4, 64), (17, 6, 128), (64, 8, 64), (65, 4, 64), (50, 16, 128)])
def test_model_step_matches_pytorch_calls(B, H, D, dtype, monkeypatch):
    """Logits and appended KV against the PyTorch calls in f32 with the same
    weights and pool: no further from them than the PyTorch calls in dtype,
    which round more often (1.5 for the spread between two roundings)."""
    print(f"  step B={B} H={H} D={D} {dtype}", flush=True)
    model, run, _ = _step(B, H, D, dtype)
    calls = []
    ops = _native.ops()
    with torch.inference_mode():
        fused, pool = run()
        monkeypatch.setattr(decode_fused, "ops_for", lambda x: calls.append(1))
        plain, pool1 = run()
        model.float()
        monkeypatch.setattr(KVBlockPool, "__init__", _f32_pool(KVBlockPool.__init__, dtype))
        exact, pool2 = run()
    assert calls and hasattr(ops, "decode_linear")
    if B > decode_fused.MAX_ROWS:
        assert torch.equal(fused, plain) and torch.equal(pool.k, pool1.k)
    rel = lambda t: ((t.double() - exact.double()).norm() / exact.double().norm()).item()
    print(f"    error: fused {rel(fused):.2e}, PyTorch calls {rel(plain):.2e}", flush=True)
    assert rel(fused) <= 1.5 * rel(plain)
    far = lambda p: (p.k.double() - pool2.k.double()).norm() + (p.v.double() - pool2.v.double()).norm()
    assert far(pool) <= 1.5 * far(pool1)


def _f32_pool(init, dtype):
    def make(self, *a, **kw):
        kw["dtype"] = torch.float32
        init(self, *a, **kw)
    return make


def test_modules_and_contexts_that_keep_the_pytorch_calls(monkeypatch):
    """Each change below must be honoured: the fused calls are not made."""
    model, run, (ids, meta) = _step(3, 4, 64, torch.bfloat16)
    used = []
    ops = _native.ops()

    class Spy:
        def decode_linear(self, *a):
            used.append("linear")
            return ops.decode_linear(*a)

        def decode_linear_norm(self, *a):
            used.append("norm")
            return ops.decode_linear_norm(*a)

        def __getattr__(self, name):
            return getattr(ops, name)

    monkeypatch.setattr(_native, "ops", lambda: Spy())

    def fused_calls():
        used.clear()
        with torch.inference_mode():
            out, _ = run()
        assert torch.isfinite(out).all()
        return len(used)

    full = fused_calls()
    assert full == 2 * 4 + 2  # per block: two linears and two with norm; the first LayerNorm and the head
    b = model.blocks[0]
    seen = []
    for m in (b.layer_norm_1, b.layer_norm_2, b.attn.qkv, b.attn.project, b.attn.resid_dropout, b.ffn, b.ffn.network,
              *b.ffn.network):
        h = m.register_forward_hook(lambda *a: seen.append(1))
        assert fused_calls() < full and seen
        h.remove()
        seen.clear()
    for m in (model.layer_norm, model.language_model_head):
        h = m.register_forward_pre_hook(lambda *a: seen.append(1))
        assert fused_calls() < full and seen
        h.remove()
        seen.clear()
    b.attn._finish = lambda out: out
    assert fused_calls() < full
    del b.attn._finish
    with monkeypatch.context() as mp:
        mp.setattr(TransformerBlock, "_mlp", lambda self, x: x)
        assert fused_calls() == 0
    for blk in model.blocks:
        blk.fused_decode_linears = False
    assert fused_calls() == 0
    with torch.inference_mode():
        off, _ = run()
        monkeypatch.setattr(decode_fused, "ops_for", lambda x: None)
        plain, _ = run()
    assert torch.equal(off, plain)
    monkeypatch.undo()
    monkeypatch.setattr(_native, "ops", lambda: Spy())
    for blk in model.blocks:
        blk.fused_decode_linears = True
    assert fused_calls() == full
    b.ffn.network[1].approximate = "tanh"
    assert fused_calls() < full
    b.ffn.network[1].approximate = "none"
    b.attn.resid_dropout.p, b.attn.resid_dropout.training = 0.5, True
    assert fused_calls() < full
    b.attn.resid_dropout.training = False
    assert fused_calls() == full
    with torch.autocast("cuda", dtype=torch.float16), torch.inference_mode():
        assert decode_fused.ops_for(torch.zeros(1, 1, 64, device=DEV, dtype=torch.bfloat16)) is None
    x = torch.zeros(1, 1, 64, device=DEV, dtype=torch.bfloat16)
    assert decode_fused.ops_for(x) is None  # gradients enabled
    with torch.no_grad():
        assert decode_fused.ops_for(x) is not None
        assert torch.func.vmap(lambda t: t if decode_fused.ops_for(t.view(1, 1, 64)) is None else None)(x[0]) is not None
        assert decode_fused.ops_for(nn.Parameter(x)) is None
        with torch.device("cuda"):
            assert decode_fused.ops_for(x) is None  # a function mode is active
