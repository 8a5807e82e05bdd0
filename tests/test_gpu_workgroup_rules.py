"""Decode at the sizes where the wave, split, tile and order rules change.

Batches on both sides of one and a half workgroups per compute unit, pieces on
both sides of the paired-tile and order thresholds, with equal and different
lengths: sampled units against the oracle, and the paged call bit for bit.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import attention as oatt
from oracle import quant as oq
from tests.helpers import MAX_ABS_TOL, MEAN_ABS_TOL

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _row(t, b, h, n):
    return t[b, h, :n].cpu().numpy()[None, None]


def _check(out, q, kq, vq, lens, units, G):
    for b, h in units:
        n = int(lens[b])
        k, v = (oq.dequantize_groupwise(oq.QuantNP(_row(t.packed, b, h, n), _row(t.scale, b, h, n),
                                                   _row(t.zero, b, h, n), t.nbits, t.group_size, 128))
                for t in (kq, vq))
        qn = q[b, h * G:(h + 1) * G].float().cpu().numpy()[None]
        m = oatt.metrics(out[b, h * G:(h + 1) * G].cpu().numpy()[None],
                         oatt.reference_decode_attention(qn, k, v))
        assert m["max_abs_err"] <= MAX_ABS_TOL and m["mean_abs_err"] <= MEAN_ABS_TOL, (b, h, n, m)


@pytest.mark.parametrize("B,S,kb,vb,G,lengths", [
    (24, 1000, 4, 4, 4, "full"),      # under one and a half workgroups per CU: 8 waves
    (50, 1000, 4, 4, 4, "full"),      # 4 waves, one tile at a time
    (50, 2113, 2, 2, 4, "full"),      # 4 waves, paired tiles
    (33, 2113, 4, 2, 8, "full"),      # 8 waves, paired tiles
    (50, 4097, 4, 4, 4, "ragged"),    # 4 waves, ordered, one tile at a time, then paired
    (50, 3000, 4, 2, 8, "ragged"),    # 4 waves, no order
    (50, 8300, 2, 2, 4, "ragged"),    # 8 waves, ordered
    (16, 4097, 4, 4, 4, "ragged"),    # below a unit per CU: cut finely
    (20, 9001, 4, 2, 8, "ragged"),
    (32, 66000, 4, 2, 8, "ragged"),   # one unit per CU, long rows cut finely
])
def test_rules_match_the_oracle(B, S, kb, vb, G, lengths):
    from tritonkv_amd.kernels import fused_decode_attention
    from tritonkv_amd.quantize import append_kv, empty_cache

    HKV, gs = 8, 32
    g = torch.Generator(device=DEV).manual_seed(B + S)
    kq, vq = empty_cache(B, HKV, S, 128, kb, gs, DEV), empty_cache(B, HKV, S, 128, vb, gs, DEV)
    x = torch.randn(1, HKV, S, 128, device=DEV, generator=g, dtype=torch.float16)
    for c in (kq, vq):  # every row the same tokens, rotated
        for b in range(B):
            row = type(c)(c.packed[b:b + 1], c.scale[b:b + 1], c.zero[b:b + 1], c.nbits, gs, 128)
            append_kv(row, torch.roll(x, 37 * b + c.nbits, 2))
    q = torch.randn(B, HKV * G, 128, device=DEV, generator=g, dtype=torch.float16)
    lens = np.full(B, S)
    if lengths == "ragged":
        lens = np.random.default_rng(B).integers(1, S + 1, B)
        lens[:4] = (1, 31, S, S // 2)
    kw = dict(allow_mixed_bits=kb != vb, _workspace={})
    if lengths == "ragged":
        kw["seq_lens"] = torch.tensor(lens, dtype=torch.int32, device=DEV)
    out = fused_decode_attention(q, kq, vq, **kw)
    _check(out, q, kq, vq, lens, [(0, 0), (1, 3), (2, 7), (3, 5), (B - 1, 2)], G)
    order = fused_decode_attention(q, kq, vq, dispatch_order=False, **dict(kw, _workspace=None))
    # the order may change the tile form (rounding), never which tokens are read
    assert float((out - order).abs().max()) <= MAX_ABS_TOL
