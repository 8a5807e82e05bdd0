"""Decode at the sizes where the wave, split, tile and order rules change.

Batches on both sides of one and a half workgroups per compute unit, pieces on
both sides of the paired-tile and order thresholds, with equal and different
lengths: sampled units against the oracle, the call in grid order bit for bit,
and the paged call bit for bit.  Each case states the plan it is there for.
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


def _caches(B, S, kb, vb, G, seed, HKV=8, gs=32):
    """q, K and V: every row the same tokens, rotated."""
    from tritonkv_amd.quantize import append_kv, empty_cache

    g = torch.Generator(device=DEV).manual_seed(seed)
    kq, vq = empty_cache(B, HKV, S, 128, kb, gs, DEV), empty_cache(B, HKV, S, 128, vb, gs, DEV)
    x = torch.randn(1, HKV, S, 128, device=DEV, generator=g, dtype=torch.float16)
    for c in (kq, vq):
        for b in range(B):
            row = type(c)(c.packed[b:b + 1], c.scale[b:b + 1], c.zero[b:b + 1], c.nbits, gs, 128)
            append_kv(row, torch.roll(x, 37 * b + c.nbits, 2))
    return torch.randn(B, HKV * G, 128, device=DEV, generator=g, dtype=torch.float16), kq, vq


def _lengths(B, S, lengths):
    if lengths == "full":
        return np.full(B, S)
    lens = np.random.default_rng(B).integers(1, S + 1, B)
    lens[:4] = (1, 31, S, S // 2)
    return lens


def _check_plan(B, S, kb, vb, G, lengths, plan, order):
    """(waves, splits) of the call, and whether it takes an order, on 256 compute units."""
    from tritonkv_amd.kernels import fused_decode_attn as fda

    if fda.compute_units() != 256:
        return
    ragged = lengths == "ragged"
    _, ns, split = fda.plan_splits(S, 64, None, B, 8, G, ragged=ragged, fine=True)
    waves = fda.choose_waves(B, 8, G, split, ns, k_nbits=kb, v_nbits=vb, group_size=32, ragged=ragged)
    assert (waves, ns, order) == plan


@pytest.mark.parametrize("B,S,kb,vb,G,lengths,plan", [
    (24, 1000, 4, 4, 4, "full", (8, 1, False)),    # under one and a half workgroups per CU
    (50, 1000, 4, 4, 4, "full", (4, 1, False)),    # one tile at a time
    (50, 2113, 2, 2, 4, "full", (4, 1, False)),    # paired tiles
    (33, 2113, 4, 2, 8, "full", (8, 1, False)),    # one tile at a time
    (33, 4113, 4, 2, 8, "full", (8, 1, False)),    # paired tiles, aligned chunks
    (50, 4097, 4, 4, 4, "ragged", (8, 1, True)),   # paired tiles, aligned chunks
    (50, 3000, 4, 2, 8, "ragged", (4, 1, False)),  # paired tiles, too short for an order
    (50, 8300, 2, 2, 4, "ragged", (12, 1, True)),
    (64, 20000, 2, 2, 4, "ragged", (4, 2, True)),  # four workgroups per CU
    (16, 4000, 4, 4, 4, "ragged", (8, 2, False)),  # half a unit per CU
    (16, 4097, 4, 4, 4, "ragged", (4, 4, False)),
    (16, 12321, 4, 2, 8, "ragged", (4, 4, False)),
    (20, 9001, 4, 2, 8, "ragged", (4, 6, False)),  # below a unit per CU: cut finely
    (32, 66000, 4, 2, 8, "ragged", (4, 6, True)),  # one unit per CU, long rows cut finely
])
def test_rules_match_the_oracle(B, S, kb, vb, G, lengths, plan):
    from tritonkv_amd.kernels import fused_decode_attention

    print(f"rules B={B} S={S} K{kb}V{vb} G={G} {lengths}", flush=True)
    q, kq, vq = _caches(B, S, kb, vb, G, B + S)
    lens, ws = _lengths(B, S, lengths), {}
    kw = dict(allow_mixed_bits=kb != vb)
    if lengths == "ragged":
        kw["seq_lens"] = torch.tensor(lens, dtype=torch.int32, device=DEV)
    out = fused_decode_attention(q, kq, vq, _workspace=ws, **kw)
    _check_plan(B, S, kb, vb, G, lengths, plan, "work_order" in ws)
    _check(out, q, kq, vq, lens, [(0, 0), (1, 3), (2, 7), (3, 5), (B - 1, 2)], G)
    assert torch.equal(out, fused_decode_attention(q, kq, vq, dispatch_order=False, **kw))


@pytest.mark.parametrize("B,S,kb,vb,G,lengths,plan", [
    (50, 1024, 4, 4, 4, "full", (4, 1, False)),    # one tile at a time
    (50, 2112, 2, 2, 4, "full", (4, 1, False)),    # paired tiles
    (33, 4096, 4, 2, 8, "full", (8, 1, False)),    # paired tiles, 8 waves
    (50, 4160, 4, 4, 4, "ragged", (8, 1, True)),
    (64, 10048, 4, 2, 8, "ragged", (8, 1, True)),
    (128, 4096, 4, 4, 4, "ragged", (4, 1, True)),
    (20, 9024, 4, 2, 8, "ragged", (4, 6, False)),
])
def test_paged_calls_follow_the_same_rules_bit_for_bit(B, S, kb, vb, G, lengths, plan):
    from tests.test_gpu_paged import _random_table, _scatter_to_pool
    from tritonkv_amd.kernels import fused_decode_attention
    from tritonkv_amd.paged import paged_decode_attention

    print(f"paged rules B={B} S={S} K{kb}V{vb} G={G} {lengths}", flush=True)
    page = 64
    q, kq, vq = _caches(B, S, kb, vb, G, B + S)
    pages = B * S // page
    table = _random_table(B, S // page, pages + 3, seed=B)
    kp, vp = (_scatter_to_pool(t, table, pages + 3, page) for t in (kq, vq))
    lens = torch.tensor(_lengths(B, S, lengths), dtype=torch.int32, device=DEV) if lengths == "ragged" else None
    ws, kw = {}, dict(allow_mixed_bits=kb != vb)
    want = fused_decode_attention(q, kq, vq, seq_lens=lens, **kw)
    got = paged_decode_attention(q, kp, vp, table, lens, _workspace=ws, **kw)
    _check_plan(B, S, kb, vb, G, lengths, plan, "work_order" in ws)
    assert torch.isfinite(got).all() and torch.equal(got, want)
    if lens is not None:
        for order in (False, True):
            assert torch.equal(got, paged_decode_attention(q, kp, vp, table, lens, dispatch_order=order, **kw))
