"""Which decode calls run as one workgroup per (sequence, head): the rule reads
only the table's width, so it must hold for any contexts in it. Host queries
(256 CUs when no device is visible, as on MI355X)."""
from __future__ import annotations

import pytest

from minivllm import _native

F32, BF16, F16 = _native.MGI_F32, _native.MGI_BF16, _native.MGI_F16


def waves(B, H, D, tokens, dtype=BF16, S=16, split_tokens=0):
    return int(_native.lib().mgi_paged_decode_workgroup_waves(B, H, D, S, -(-tokens // S), dtype, split_tokens))


@pytest.mark.parametrize("B,H,D,tokens,dtype", [
    # one long context in the table would take its workgroup longer than the split takes for the call, measured 1.5-3
    # times as long, also where partial head groups slow the split down on full tables
    (64, 4, 32, 32768, BF16), (190, 4, 64, 131072, BF16), (64, 2, 128, 8192, BF16), (32, 4, 64, 8192, F32),
    (13, 4, 32, 8192, F32), (64, 4, 64, 8192, BF16), (64, 2, 128, 4096, F32), (1, 32, 128, 2000, BF16),
    (4, 32, 128, 4000, BF16), (190, 4, 64, 9728, F16),
    # head dims that leave lanes empty cost as much as those that fill them: 31 us against 62, 69 against 173
    (13, 32, 8, 8192, BF16), (13, 32, 8, 4096, F32), (64, 16, 8, 4096, BF16), (13, 32, 16, 2048, F32),
    (32, 8, 40, 2048, BF16), (13, 20, 80, 2048, BF16), (4, 8, 24, 2048, BF16),
    # half of the rows long: 55 us against 65
    (256, 4, 128, 1024, BF16), (64, 16, 128, 1024, BF16), (128, 8, 128, 1024, BF16),
    # too many workgroups for short contexts: 5.4 us against 12 or more
    (128, 16, 128, 256, BF16), (64, 32, 32, 256, BF16), (256, 8, 64, 256, F32), (256, 16, 64, 112, BF16),
])
def test_left_to_the_split(B, H, D, tokens, dtype, monkeypatch):
    monkeypatch.delenv("MINIVLLM_HIP_DECODE_WG", raising=False)
    assert waves(B, H, D, tokens, dtype) == 0
    assert waves(B, H, D, 2 * tokens, dtype) == 0


@pytest.mark.parametrize("B,H,D,tokens,dtype,want", [
    (4, 8, 32, 256, F32, 8), (13, 16, 128, 1008, BF16, 8), (16, 16, 128, 768, BF16, 8), (32, 8, 128, 1024, F16, 8),
    (22, 22, 128, 64, BF16, 4), (64, 16, 128, 256, BF16, 4), (1, 1, 8, 16, F32, 4), (20, 16, 96, 256, BF16, 4)])
def test_small_calls(B, H, D, tokens, dtype, want, monkeypatch):
    monkeypatch.delenv("MINIVLLM_HIP_DECODE_WG", raising=False)
    assert waves(B, H, D, tokens, dtype) == want


def test_one_long_context_never_outlasts_the_split(monkeypatch):
    """Over the ranges calls come in: a full row's K and V per workgroup, at a
    CU's own rate, stay below what the split takes for such a row (27 us at the
    most, plus the row's bytes at the split's lowest rate)."""
    monkeypatch.delenv("MINIVLLM_HIP_DECODE_WG", raising=False)
    taken = 0
    for dtype, eb in ((BF16, 2), (F32, 4)):
        for H in (1, 2, 4, 5, 8, 16, 20, 32):
            for D in (8, 32, 64, 80, 96, 128, 256):
                for B in (1, 3, 8, 22, 64, 256, 1000, 4096, 4100):
                    for tokens in (16, 64, 256, 512, 1024, 2048, 4096, 8192, 32768, 131072):
                        if waves(B, H, D, tokens, dtype):
                            taken += 1
                            mb = 2e-6 * tokens * D * eb
                            assert 4.2 + 23.5 * mb <= 27.0 + H * mb / 0.8, (B, H, D, tokens, dtype)
    assert taken > 1000


def test_explicit_splits_and_other_paths(monkeypatch):
    monkeypatch.delenv("MINIVLLM_HIP_DECODE_WG", raising=False)
    assert waves(4, 8, 32, 256, split_tokens=64) == 0
    assert waves(4, 8, 12, 256) == 0 and waves(4, 8, 264, 256) == 0 and waves(4, 8, 32, 256, S=4) == 0
    assert waves(4, 8, 32, 256, F32, S=4) == 8 and waves(0, 8, 32, 256) == 0 and waves(4, 8, 32, 256, 7) == 0
    for value, want in (("0", 0), ("4", 4), ("8", 8)):
        monkeypatch.setenv("MINIVLLM_HIP_DECODE_WG", value)
        assert waves(4, 8, 32, 256) == want and waves(64, 4, 32, 32768) == want
        assert waves(4, 8, 32, 256, split_tokens=64) == 0
