"""The launch plan of a decode call (split counts and waves), from its sizes alone."""

from __future__ import annotations

import pytest


@pytest.fixture(autouse=True)
def _cus(monkeypatch):
    from tritonkv_amd.kernels import fused_decode_attn as fda

    monkeypatch.setattr(fda, "compute_units", lambda device=None: 256)


@pytest.mark.parametrize("B,S,splits", [
    (16, 4095, 2), (16, 4096, 4), (16, 8192, 8), (16, 16384, 4), (16, 32768, 8),  # half a unit per CU
    (17, 2048, 1), (17, 4096, 4), (20, 4096, 4),            # up to five eighths
    (24, 4096, 1), (24, 8192, 5),                           # up to three quarters
    (28, 8192, 1), (31, 8192, 1), (31, 16384, 4),           # up to one
    (32, 16384, 2), (32, 65535, 2), (32, 65536, 6), (40, 98304, 9), (64, 131072, 4),
])
def test_ragged_batches_are_cut_where_that_was_measured_to_pay(B, S, splits):
    from tritonkv_amd.kernels.fused_decode_attn import plan_splits

    assert plan_splits(S, 64, None, B, 8, 4, ragged=True, fine=True)[1] == splits
    # the fp16 control, per-channel keys and callers with partials of their own keep the even cut
    even = plan_splits(S, 64, None, B, 8, 4, ragged=True)[1]
    assert even == ({16: 2}.get(B, 1) if B < 32 else max(2, S // 32768))


def test_the_plan_of_other_callers_fits_the_static_scratch():
    """48 rows of 64 query heads and up to 131072 tokens: the partials of the plan
    a caller without a workspace makes (tkv_fused_decode_attention_noalloc)."""
    from tritonkv_amd import _lib
    from tritonkv_amd.kernels import plan_splits

    _, ns, _ = plan_splits(131072, 64, None, 48, 8, 8, ragged=True)
    assert ns == 4 and 48 * 64 * ns * (128 + 2) * 4 <= _lib.NOALLOC_SCRATCH_BYTES


FP16, K4, K2, K42 = (16, 16, 0), (4, 4, 32), (2, 2, 32), (4, 2, 32)
ONE4, ONE2 = (4, 4, 128), (2, 2, 128)


@pytest.mark.parametrize("fmt,D,B,S,ns,ragged,waves", [
    (K4, 128, 47, 1024, 1, False, 8), (K4, 128, 48, 1024, 1, False, 4), (K4, 128, 64, 32768, 1, False, 4),
    (K2, 128, 64, 32768, 1, False, 4), (K2, 128, 64, 40960, 1, False, 12),
    (ONE4, 128, 64, 32768, 1, False, 4),
    (FP16, 128, 64, 8192, 1, False, 4), (FP16, 128, 128, 16384, 1, False, 8), (FP16, 64, 64, 1024, 1, False, 8),
    (K4, 64, 64, 16384, 1, False, 4), (K2, 64, 64, 4096, 1, False, 8), (K2, 64, 128, 4096, 1, False, 4),
    (K42, 64, 64, 16384, 1, False, 8),
    (K4, 128, 64, 3072, 1, True, 4), (K4, 128, 64, 4096, 1, True, 8), (K4, 128, 128, 4096, 1, True, 4),
    (K4, 128, 24, 4096, 4, True, 4), (K4, 128, 128, 8192, 1, True, 4), (K4, 128, 64, 16384, 2, True, 8),
    (K2, 128, 64, 16384, 2, True, 4), (K4, 128, 64, 32768, 3, True, 4),
    (ONE4, 128, 128, 8192, 1, True, 4), (ONE4, 128, 64, 16384, 2, True, 12), (ONE4, 128, 96, 16384, 2, True, 4),
    (ONE4, 128, 64, 32768, 3, True, 12), (ONE2, 128, 64, 32768, 2, True, 4),
    (FP16, 128, 64, 512, 1, True, 4), (FP16, 128, 64, 1024, 1, True, 8), (FP16, 64, 64, 512, 1, True, 8),
    (K2, 64, 64, 2048, 1, True, 8), (K2, 64, 128, 2048, 1, True, 4), (K4, 64, 128, 8192, 1, True, 8),
])
def test_four_waves_run_where_they_were_measured_to_pay(fmt, D, B, S, ns, ragged, waves):
    from tritonkv_amd.kernels.fused_decode_attn import choose_waves

    k, v, gs = fmt
    assert choose_waves(B, 8, 4, S, ns, D=D, k_nbits=k, v_nbits=v, group_size=gs, ragged=ragged) == waves


def test_per_channel_keys_keep_larger_workgroups_on_long_pieces():
    from tritonkv_amd.kernels.fused_decode_attn import choose_waves

    kw = dict(D=128, k_nbits=2, v_nbits=2, group_size=32, ragged=True)
    assert choose_waves(64, 8, 4, 16384, 2, **kw) == 4
    assert choose_waves(64, 8, 4, 16384, 2, per_channel=True, **kw) == 12
    assert choose_waves(128, 8, 4, 4096, 1, per_channel=True, **kw) == 4
    assert choose_waves(128, 8, 4, 8192, 1, per_channel=True, **kw) == 12
    kw["ragged"] = False
    assert choose_waves(64, 8, 4, 16384, 1, per_channel=True, **kw) == 4
    assert choose_waves(64, 8, 4, 24576, 1, per_channel=True, **kw) == 12


def test_page_pools_of_head_dim_64_keep_larger_workgroups():
    from tritonkv_amd.kernels.fused_decode_attn import choose_waves

    kw = dict(D=64, k_nbits=4, v_nbits=4, group_size=64, paged=True)
    assert [choose_waves(B, 8, G, 4096, 1, **kw) for B, G in ((64, 4), (128, 4), (64, 16))] == [8, 4, 4]
