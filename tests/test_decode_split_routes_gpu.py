"""The decode tests whose small shapes the one-launch kernel takes, run once more
on the split kernels (partitions, even split) of those shapes on the MI355X: lane
layouts and partial head groups, strides, index types, scales, empty and one-token
contexts, the fused append in each, and the even split's fused append with its
ticket claims."""
from __future__ import annotations

import pytest
import torch

import test_decode_append_gpu as app
import test_paged_decode_gpu as dec

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("split_kernels")]
F32, BF16, F16 = torch.float32, torch.bfloat16, torch.float16
DTYPES = [F32, BF16, F16]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("D", [32, 64, 128, 256])
@pytest.mark.parametrize("S,H", [(16, 32), (8, 3), (32, 5)])
def test_lane_layouts_and_head_groups(dtype, D, S, H):
    assert dec.takes_balanced_split(6, H, D, S, -(-513 // S), dtype)
    dec.test_fast_path_shapes(dtype, D, S, H, 0)


@pytest.mark.parametrize("dtype", DTYPES)
def test_int32_indices_strided_q_and_short_contexts(dtype):
    assert dec.takes_balanced_split(3, 8, 128, 16, 40, dtype)
    dec.test_int32_indices_and_strided_q(dtype, 0)
    dec.test_single_token_context_returns_value_row_exactly(dtype)
    dec.test_zero_context_row_gives_zeros()


@pytest.mark.parametrize("scale", [-0.3, 0.0], ids=["neg", "zero"])
@pytest.mark.parametrize("dtype", [F32, BF16], ids=["f32", "bf16"])
def test_scales_and_strided_outputs(dtype, scale):
    assert dec.takes_balanced_split(24, 8, 128, 16, 37, dtype)
    dec.test_any_finite_scale_matches_c_oracle(dtype, 0, scale)
    dec.test_strided_outputs_match_contiguous(dtype, 0)


@pytest.mark.parametrize("dtype", [BF16, F16, F32], ids=["bf16", "f16", "f32"])
@pytest.mark.parametrize("B,H,D,S,lo,hi,split", [c for c in app.CASES if c[-1] == 0])
def test_fused_append(dtype, B, H, D, S, lo, hi, split):
    app.test_fused_matches_append_then_decode(dtype, B, H, D, S, lo, hi, split)


@pytest.mark.parametrize("tiers", dec.TIERS)
@pytest.mark.parametrize("dtype", [BF16, F32], ids=["bf16", "f32"])
@pytest.mark.parametrize("B,H,D", [(40, 6, 96), (33, 4, 64), (21, 8, 128)])
def test_fused_append_with_ticket_claims(B, H, D, dtype, tiers, monkeypatch):
    """Rows of every kind, empty sequences among them, in wide enough tables that
    the even split divides them, under each setting of its claims."""
    dec._set_tiers(monkeypatch, tiers)
    c = app.step_case(B, H, D, 16, 1, 900, dtype, seed=B + D)
    assert "empty" in c["kinds"] and "tail" in c["kinds"]
    assert dec.takes_balanced_split(B, H, D, 16, c["tables"].shape[1], dtype)
    app.assert_identical(*app.run_both(c))


@pytest.mark.parametrize("dtype", [BF16, F32], ids=["bf16", "f32"])
def test_fused_append_index_types_views_and_steps(dtype):
    app.test_int32_tables_lengths_and_slots(dtype, 0)
    app.test_every_row_kind_lands_in_the_fused_write()
    app.test_rows_from_a_fused_qkv_view()
    app.test_repeated_fused_steps_match_repeated_separate_steps()
