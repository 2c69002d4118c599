"""The fp32 paged prefill's key split on the MI355X: where the cost rule takes
it, against the float64 oracle and against the same call unsplit, over tile and
partition edges, ragged chunks, every padded head dim, two-wavefront chunks, odd
block sizes and masked table entries; and the C entry without a workspace."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from minivllm import _native
from test_paged_prefill_gpu import check, prefill_case, run_hip

DEV = torch.device("cuda:0")
CASES = [  # start, T, H, D, S
    (450, 700, 8, 64, 16), (0, 512, 4, 32, 16), (512, 64, 8, 128, 16), (255, 65, 4, 128, 16), (1000, 100, 3, 96, 5),
    (2000, 20, 4, 24, 16), (383, 33, 2, 40, 32), (0, 515, 2, 8, 4), (1, 191, 5, 72, 16)]


def ws_bytes(start, T, H, D):
    return int(_native.lib().mgi_paged_prefill_workspace_bytes(start, T, H, D, _native.MGI_F32))


@pytest.mark.gpu
@pytest.mark.parametrize("start,T,H,D,S", CASES)
def test_split_matches_oracle_and_unsplit(start, T, H, D, S, monkeypatch):
    assert ws_bytes(start, T, H, D) > 0
    qkv, pool, table, layer = prefill_case(start, T, H, D, S, torch.float32, seed=T)
    q = qkv.to(DEV)[:, 0]
    torch.cuda.empty_cache()
    torch.empty(1 << 24, device=DEV).fill_(float("nan"))  # freed: the workspace may reuse it
    out = run_hip(q, pool, table, start, layer)
    check(out, q, pool, table, start, layer)
    monkeypatch.setenv("MINIVLLM_HIP_PREFILL_SPLIT_KEYS", "-1")
    assert ws_bytes(start, T, H, D) == 0
    whole = run_hip(q, pool, table, start, layer)
    # two orders of the same f32 sums: 2^-24 per term of up to start + T keys of weight about 1 / (start + T)
    torch.testing.assert_close(out, whole, atol=1e-5, rtol=1e-5)


@pytest.mark.gpu
def test_masked_entries_and_no_workspace():
    start, T, H, D, S = 450, 200, 4, 64, 16
    qkv, pool, table, layer = prefill_case(start, T, H, D, S, torch.float32, seed=3)
    q = qkv.to(DEV)[:, 0]
    out = run_hip(q, pool, table, start, layer)
    lib, check_status = _native.lib(), _native.check
    got = torch.empty_like(out)
    t = table.to(DEV)
    args = (got.data_ptr(), _native.strides(got), q.data_ptr(), _native.strides(q), pool.k.data_ptr(),
            pool.v.data_ptr(), _native.strides(pool.k), _native.strides(pool.v), _native.MGI_F32, t.data_ptr(),
            t.stride(0), _native.MGI_I64, t.numel(), start, T, H, D, S, pool.num_blocks, pool.n_layer, layer, D ** -0.5,
            None, 0, torch.cuda.current_stream().cuda_stream)
    check_status(lib.mgi_paged_prefill(*args))  # fp32 needs no workspace: it runs unsplit
    torch.testing.assert_close(out, got, atol=1e-5, rtol=1e-5)
    table[:3] = -1
    table[20] = pool.num_blocks
    masked = run_hip(q, pool, table, start, layer)
    # float64 over the keys that are left
    pos = torch.arange(start + T)
    phys = table[pos // S]
    ok = (phys >= 0) & (phys < pool.num_blocks)
    k = pool.k[layer].cpu()[phys.clamp(0, pool.num_blocks - 1), pos % S].double()
    v = pool.v[layer].cpu()[phys.clamp(0, pool.num_blocks - 1), pos % S].double()
    k[~ok], v[~ok] = 0, 0
    s = torch.einsum("thd,khd->htk", q.cpu().double(), k) * D ** -0.5
    s = s.masked_fill(~(ok[None] & (pos[None] <= start + torch.arange(T)[:, None]))[None], -np.inf)
    want = torch.einsum("htk,khd->thd", torch.softmax(s, -1), v)
    np.testing.assert_allclose(masked.cpu().numpy(), want.numpy(), atol=2e-5, rtol=2e-4)


def test_rule_on_the_host(monkeypatch):
    monkeypatch.delenv("MINIVLLM_HIP_PREFILL_SPLIT_KEYS", raising=False)
    assert ws_bytes(0, 64, 8, 64) == 0            # one key tile
    assert ws_bytes(0, 4096, 64, 64) == 0         # query tiles enough
    assert ws_bytes(450, 700, 8, 20) == 0         # the merge's lane layout
    assert ws_bytes(450, 700, 8, 136) == 0        # no matrix-core variant
    assert ws_bytes(15360 - 100, 100, 4, 64) > 0
    assert ws_bytes(15360 - 100, 101, 4, 64) == 0
    for start, T, H, D in ((450, 700, 8, 64), (0, 512, 4, 32), (4096, 256, 16, 128), (3000, 32, 8, 32)):
        n = ws_bytes(start, T, H, D)
        parts = [p for p in range(2, 300) if -(-T * H * p * D * 4 // 256) * 256 + T * H * p * 8 == n]
        assert len(parts) == 1


@pytest.mark.gpu
@pytest.mark.parametrize("start,T,H", [(3000, 900, 16), (15000, 300, 32)])
def test_bf16_workspace_too_small_for_the_priced_split(start, T, H):
    """A workspace that holds less than the priced split's partials: the call
    falls back to the plain split or refuses, as it did before, and never writes
    past what it was given."""
    lib, D, S = _native.lib(), 128, 16
    n = -(-(start + T) // S)
    pool_k = torch.randn((1, n, S, H, D), device=DEV).to(torch.bfloat16)
    q = torch.randn((T, H, D), device=DEV).to(torch.bfloat16)
    table = torch.randperm(n, device=DEV)
    need = int(lib.mgi_paged_prefill_workspace_bytes(start, T, H, D, _native.MGI_BF16))
    assert need > 0
    outs = []
    for nbytes in (need, need - 256):
        ws = torch.full((need,), 77, dtype=torch.uint8, device=DEV)
        out = torch.empty_like(q)
        rc = lib.mgi_paged_prefill(
            out.data_ptr(), _native.strides(out), q.data_ptr(), _native.strides(q), pool_k.data_ptr(), pool_k.data_ptr(),
            _native.strides(pool_k), _native.strides(pool_k), _native.MGI_BF16, table.data_ptr(), 1, _native.MGI_I64, n,
            start, T, H, D, S, n, 1, 0, D ** -0.5, ws.data_ptr(), nbytes, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        assert rc in (_native.MGI_OK, _native.MGI_EWORKSPACE) and (nbytes < need or rc == _native.MGI_OK)
        assert (ws[nbytes:] == 77).all()
        if rc == _native.MGI_OK:
            outs.append(out.double())
    if len(outs) == 2:
        assert ((outs[0] - outs[1]).norm() / outs[0].norm()).item() <= 2.0 ** -8
