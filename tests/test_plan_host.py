"""The launch plan of a decode call (split counts and waves), from its sizes alone."""

from __future__ import annotations

import pytest


@pytest.fixture(autouse=True)
def _cus(monkeypatch):
    from tritonkv_amd.kernels import fused_decode_attn as fda

    monkeypatch.setattr(fda, "compute_units", lambda device=None: 256)


@pytest.mark.parametrize("B,S,splits", [
    (16, 8192, 2), (16, 16384, 2), (16, 32768, 8),          # half a unit per CU
    (17, 2048, 1), (17, 4096, 4), (20, 4096, 4),            # up to five eighths
    (24, 4096, 1), (24, 8192, 5),                           # up to three quarters
    (28, 8192, 1), (31, 8192, 1), (31, 16384, 4),           # up to one
    (32, 16384, 2), (32, 65535, 2), (32, 65536, 2), (40, 98304, 3), (64, 131072, 4),
])
def test_ragged_batches_are_cut_where_that_was_measured_to_pay(B, S, splits):
    from tritonkv_amd.kernels.fused_decode_attn import plan_splits

    assert plan_splits(S, 64, None, B, 8, 4, ragged=True)[1] == splits
    # the fp16 control and per-channel keys keep the even cut
    even = plan_splits(S, 64, None, B, 8, 4, ragged=True, fine=False)[1]
    assert even == {16: 2}.get(B, 1) if B < 32 else even == splits
