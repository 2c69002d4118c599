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


def plain_bytes(start, T, H, D):
    """Workspace of the 2-byte types' plain split on 256 CUs (0: none), by the
    rule written out."""
    tiles = [-(-(start + min(T, r + 64)) // 64) for r in range(0, T, 64)]
    k = max(2, -(-sum(tiles) * H // 512))
    if len(tiles) * H >= 512 or start < T or k >= tiles[-1]:
        return 0
    spans = sum(p for p in (-(-(start + i + 1) // (64 * k)) for i in range(T)) if p > 1)
    tile_us = 1.5 * max(D, 64) / 128
    if k * tile_us + 8.0 + 2.0 * spans * H * (4 * D + 8) / 5.0e6 >= tiles[-1] * tile_us:
        return 0
    n = T * H * -(-(start + T) // (64 * k))
    return -(-n * D * 4 // 256) * 256 + n * 8


def prefill_with_workspace(start, T, H, D, dtype):
    """A bf16, f16 or fp32 call of fixed inputs as a function of its workspace
    (bytes, and how many bytes off alignment; None for no workspace): (status,
    output), with the bytes past the workspace checked untouched."""
    lib, S = _native.lib(), 16
    n = -(-(start + T) // S)
    g = torch.Generator(device=DEV).manual_seed(T)
    pool_k, pool_v = (torch.randn((1, n, S, H, D), generator=g, device=DEV).to(dtype) for _ in range(2))
    q = torch.randn((T, H, D), generator=g, device=DEV).to(dtype)
    table = torch.randperm(n, device=DEV, generator=g)

    def call(nbytes, off=0):
        print(f"  prefill start={start} T={T} H={H} D={D} {dtype} workspace {nbytes} bytes off {off}", flush=True)
        out = torch.full_like(q, float("nan"))
        ws = None if nbytes is None else torch.full((nbytes + 512,), 77, dtype=torch.uint8, device=DEV)
        rc = lib.mgi_paged_prefill(
            out.data_ptr(), _native.strides(out), q.data_ptr(), _native.strides(q), pool_k.data_ptr(), pool_v.data_ptr(),
            _native.strides(pool_k), _native.strides(pool_v), _native.DTYPE_CODES[dtype], table.data_ptr(), 1,
            _native.MGI_I64, n, start, T, H, D, S, n, 1, 0, D ** -0.5, None if ws is None else ws.data_ptr() + off,
            0 if nbytes is None else nbytes, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        assert ws is None or ((ws[:off] == 77).all() and (ws[off + nbytes:] == 77).all())
        return rc, out
    return call


@pytest.mark.gpu
@pytest.mark.parametrize("start,T,H", [(3000, 900, 16), (15000, 300, 32)])
def test_bf16_workspace_too_small_for_the_priced_split(start, T, H, monkeypatch):
    """A workspace below what the query asks for: the plain split where its
    partials fit, with that split's own bits, else a refusal, as before there
    were prices; never a byte past what was given."""
    D = 128
    need = int(_native.lib().mgi_paged_prefill_workspace_bytes(start, T, H, D, _native.MGI_BF16))
    plain = plain_bytes(start, T, H, D)
    assert 0 < plain <= need
    call = prefill_with_workspace(start, T, H, D, torch.bfloat16)
    rc, full = call(need)
    assert rc == _native.MGI_OK and torch.isfinite(full).all()
    rc, out = call(plain)
    assert rc == _native.MGI_OK
    rows = (out.double() - full.double()).norm(dim=-1) / full.double().norm(dim=-1)
    assert rows.max().item() <= 2.0 ** -6  # every row and head: a few half-ulps (2^-9) of outputs and weights
    for nbytes in (plain - 256 if need > plain else 4096, 16, None):  # need == plain: the priced split wants less
        rc, out = call(nbytes)
        assert rc == _native.MGI_EWORKSPACE and torch.isnan(out).all()
    rc, out = call(need, off=8)
    assert rc == _native.MGI_EINVAL and torch.isnan(out).all()


@pytest.mark.gpu
@pytest.mark.parametrize("start,T,H,D,dtype", [(8000, 900, 32, 64, torch.bfloat16), (8000, 900, 32, 64, torch.float16),
                                               (450, 700, 8, 64, torch.float32)])
def test_calls_without_a_plain_split_run_unsplit_without_room(start, T, H, D, dtype, monkeypatch):
    """No workspace, too small or misaligned a one, where only the priced split
    wants any: the unsplit call's bits, as before there were prices."""
    need = int(_native.lib().mgi_paged_prefill_workspace_bytes(start, T, H, D, _native.DTYPE_CODES[dtype]))
    assert need > 0 and (dtype == torch.float32 or plain_bytes(start, T, H, D) == 0)
    call = prefill_with_workspace(start, T, H, D, dtype)
    rc, split = call(need)
    assert rc == _native.MGI_OK
    outs = [call(None), call(need - 256), call(need, off=8)]
    monkeypatch.setenv("MINIVLLM_HIP_PREFILL_SPLIT_KEYS", "-1")
    rc, whole = call(None)
    assert rc == _native.MGI_OK and not torch.equal(split, whole)
    for rc, out in outs:
        assert rc == _native.MGI_OK and torch.equal(out, whole)
    rows = (split.double() - whole.double()).norm(dim=-1) / whole.double().norm(dim=-1)
    assert rows.max().item() <= {torch.bfloat16: 2.0 ** -6, torch.float16: 2.0 ** -9, torch.float32: 1e-5}[dtype]
