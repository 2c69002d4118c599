"""The one-launch decode kernel (one workgroup per (sequence, head)) on the
MI355X: against float64 softmax over the gathered tokens, and its fused append against the split kernels,
at the sizes where its work division can go wrong -- contexts around a granule
(4 tokens, 2 in f32), around one and two steps of four and of eight
wavefronts, empty and one-token contexts, head dims below and at every lane
layout, block sizes that are not a power of two, masked table entries, and
NaN in every slot outside a context."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import _fixtures as fx
from minivllm import _native
from minivllm import hip_paged_decode as hpd
from test_decode_append_gpu import bits, step_case
from test_paged_decode_gpu import _small_case, hip

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
# The suite's decode tolerances: f32 sums in another order; one rounding of a
# 2-byte output of magnitude about one (2^-9 and 2^-12) with room for the order.
TOL = {torch.float32: 1e-5, torch.bfloat16: 2e-2, torch.float16: 2e-3}
DTYPES = [torch.float32, torch.bfloat16, torch.float16]


def edges(D: int, dtype, waves: int, cap: int) -> list[int]:
    lph = 4 if D <= 32 else 8 if D <= 64 else 16 if D <= 128 else 32
    gt = 2 if dtype == torch.float32 else 4
    step = waves * (64 // lph) * gt
    ctx = {0, 1, gt - 1, gt, gt + 1, step - 1, step, step + 1, 2 * step, 2 * step + gt + 1, 3 * step - 1, cap}
    return sorted(c for c in ctx if c <= cap)


def reference(q, pool, tables, lens, layer) -> np.ndarray:
    """softmax(q K^T / sqrt(D)) V in float64 over each row's tokens whose table entry is a block."""
    S, out = pool.block_size, torch.zeros(q.shape, dtype=torch.float64)
    for b, n in enumerate(lens.tolist()):
        phys = tables[b].repeat_interleave(S)[:n]
        keep = (phys >= 0) & (phys < pool.num_blocks)
        if not keep.any():
            continue
        idx, off = phys[keep], (torch.arange(n) % S)[keep]
        k, v = pool.k[layer, idx, off].double(), pool.v[layer, idx, off].double()
        p = torch.softmax((k * q[b].double()).sum(-1) / q.shape[-1] ** 0.5, 0)
        out[b] = (p.unsqueeze(-1) * v).sum(0)
    return out.numpy()


@pytest.mark.parametrize("waves", [4, 8])
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("D,S,H", [(8, 16, 3), (32, 16, 8), (64, 8, 5), (80, 24, 2), (128, 16, 4), (256, 40, 1)])
def test_matches_reference_at_step_edges(D, S, H, dtype, waves, monkeypatch):
    monkeypatch.setenv("MINIVLLM_HIP_DECODE_WG", str(waves))
    print(f"  D={D} S={S} H={H} {dtype} waves={waves}", flush=True)
    ctx = edges(D, dtype, waves, 1100)
    N = sum((c + S - 1) // S for c in ctx) + 4
    q, pool, tables, lens, layer = _small_case(len(ctx), H, D, S, ctx, dtype, seed=D + waves, N=N)
    tables[-1, 1] = -1       # a masked block in the longest context
    tables[-2, 0] = N + 3    # and an entry past the pool
    got = hip(q, fx.pool_to_device(pool, DEV), tables, lens, layer)
    want = reference(q, pool, tables, lens, layer)
    np.testing.assert_allclose(got, want, atol=TOL[dtype], rtol=TOL[dtype])
    assert (got[np.array(ctx) == 0] == 0).all()


@pytest.mark.parametrize("waves", [4, 8])
@pytest.mark.parametrize("dtype", DTYPES)
def test_scores_of_minus_infinity(dtype, waves, monkeypatch):
    """A score of -inf is a weight of 0 wherever it stands -- alone in the last
    granule, filling the first one, a row's only one, or all but one token of the
    context -- and a context of nothing else is NaN, as softmax has it."""
    monkeypatch.setenv("MINIVLLM_HIP_DECODE_WG", str(waves))
    ctx = [5, 17, 40, 40, 3, 300, 8]
    print(f"  -inf scores {dtype} waves={waves}", flush=True)
    q, pool, tables, lens, layer = _small_case(len(ctx), 3, 32, 16, ctx, dtype, seed=21)
    q = q.abs() + 0.5
    # the -inf tokens of each sequence: its last, its first granule, two granules, all but one, all, every second
    # one, the first half
    gone = [[4], range(4), range(8, 16), [i for i in range(40) if i != 23], range(3), range(0, 300, 2), range(4)]
    for b, tokens in enumerate(gone):
        for i in tokens:
            pool.k[layer, tables[b, i // 16], i % 16, :, 7] = -float("inf")
    got = hip(q, fx.pool_to_device(pool, DEV), tables, lens, layer)
    want = reference(q, pool, tables, lens, layer)
    assert np.isnan(want[4]).all() and np.isfinite(np.delete(want, 4, 0)).all()
    np.testing.assert_allclose(got, want, atol=TOL[dtype], rtol=TOL[dtype])


@pytest.mark.parametrize("waves", [4, 8])
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("D", [32, 96, 128])
def test_fused_append_matches_two_calls(D, dtype, waves, monkeypatch):
    """Same pools and outputs, bit for bit, as the append kernel followed by
    the same attention kernel; the split kernels agree within tolerance."""
    print(f"  append D={D} {dtype} waves={waves}", flush=True)
    c = step_case(24, 4, D, 16, 1, 700, dtype, seed=D + waves)
    pools = [fx.pool_to_device(c["pool"], DEV) for _ in range(2)]
    monkeypatch.setenv("MINIVLLM_HIP_DECODE_WG", str(waves))
    fused = hpd.paged_attention_batch_append_hip(c["q"], pools[0], c["tables"], c["ctx"], 1, c["k"], c["v"], c["slots"])
    hpd.kv_append(pools[1], 1, c["k"], c["v"], c["slots"])
    two = hpd.paged_attention_batch_hip(c["q"], pools[1], c["tables"], c["ctx"], 1)
    monkeypatch.setenv("MINIVLLM_HIP_DECODE_WG", "0")
    split = hpd.paged_attention_batch_hip(c["q"], pools[1], c["tables"], c["ctx"], 1)
    assert torch.equal(bits(pools[0].k), bits(pools[1].k)) and torch.equal(bits(pools[0].v), bits(pools[1].v))
    assert torch.equal(bits(fused), bits(two))
    torch.testing.assert_close(fused, split, atol=TOL[dtype], rtol=TOL[dtype])


@pytest.mark.parametrize("dtype", DTYPES)
def test_split_kernels_still_match_where_the_rule_leaves_them(dtype, monkeypatch):
    """The shapes the one-launch kernel now takes, on the balanced split."""
    monkeypatch.setenv("MINIVLLM_HIP_DECODE_WG", "0")
    ctx = [0, 1, 17, 255, 256, 640]
    q, pool, tables, lens, layer = _small_case(6, 8, 128, 16, ctx, dtype, seed=9, N=90)
    got = hip(q, fx.pool_to_device(pool, DEV), tables, lens, layer)
    want = reference(q, pool, tables, lens, layer)
    np.testing.assert_allclose(got, want, atol=TOL[dtype], rtol=TOL[dtype])


@pytest.mark.parametrize("B,H,D,width,want", [(4, 8, 32, 16, 8), (22, 22, 128, 4, 4), (8, 4, 128, 128, 0)])
def test_query_names_the_route_a_call_takes(B, H, D, width, want, monkeypatch):
    """The call's bits are those of the route mgi_paged_decode_workgroup_waves
    reports, and not those of the others: a table with one full row."""
    monkeypatch.delenv("MINIVLLM_HIP_DECODE_WG", raising=False)
    assert hpd._native.lib().mgi_paged_decode_workgroup_waves(B, H, D, 16, width, _native.MGI_F32, 0) == want
    ctx = [16 * width] + [1 + (7 * b) % min(48, 16 * width) for b in range(1, B)]
    q, pool, tables, lens, layer = _small_case(B, H, D, 16, ctx, torch.float32, seed=B)
    pool, auto = fx.pool_to_device(pool, DEV), {}
    auto["call"] = hip(q, pool, tables, lens, layer)
    for w in (0, 4, 8):
        monkeypatch.setenv("MINIVLLM_HIP_DECODE_WG", str(w))
        auto[w] = hip(q, pool, tables, lens, layer)
    assert [w for w in (0, 4, 8) if np.array_equal(auto[w], auto["call"])] == [want]
