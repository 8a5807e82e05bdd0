"""Decode over caches whose blocks start inside a cache line (S no multiple of 32).

Splits of 4096 tokens or more of the long-split forms (paired tiles, which small
grids run from 8192 tokens, and one tile at a time above 8 query heads) then count
their chunks from a multiple of 32 rows of the tensor and mask the rows before the
split: the chunk before the block's start (read as zeros), before a later split's
start (the previous split's rows), and a first chunk that is also the last, with
and without the appended token in it.  Against the oracle's fp32 attention over
the same codes.
"""

from __future__ import annotations

import pytest
import torch

from tests.helpers import assert_close_to_reference, make_case, oracle_attention_on_quant

pytestmark = pytest.mark.gpu
DEV = "cuda"

CASES = [  # nbits, gs, HQ, HKV, D, S, num_splits
    (4, 32, 8, 2, 128, 4127, 1),     # one tile at a time: not aligned
    (4, 32, 8, 2, 128, 8250, 2),     # ... and a second split that starts at a block of 64
    (4, 32, 12, 2, 128, 8251, 1),    # paired tiles
    (2, 32, 8, 2, 128, 8263, 1),     # 12 waves
    (2, 128, 8, 2, 128, 8250, 1),    # one group per row: not aligned
    (2, 128, 8, 2, 128, 8251, 1),    # ... odd S
    (4, 16, 32, 2, 128, 4099, 1),    # 16 head columns
    (2, 64, 4, 2, 64, 8199, 1),      # one group per row
    (4, 32, 8, 2, 128, 16451, 2),    # paired tiles, a second split
    (2, 32, 8, 2, 128, 16469, 2),    # ... in 12 waves
    (4, 16, 32, 2, 128, 8251, 2),    # 16 head columns, a second split
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c)))
def test_unaligned_blocks_match_the_oracle(case):
    from tritonkv_amd.kernels import fused_decode_attention

    nbits, gs, HQ, HKV, D, S, ns = case
    q, _, _, kq, vq = make_case(2, HQ, HKV, D, S, nbits, gs, seed=S + gs, outlier_frac=0.0)
    out = fused_decode_attention(q, kq, vq, num_splits=ns)
    assert_close_to_reference(out, oracle_attention_on_quant(q, kq, vq), str(case))


@pytest.mark.parametrize("nbits,HQ,S", [(4, 8, 4127), (2, 8, 8263), (4, 12, 8251)])
@pytest.mark.parametrize("append", [False, True])
def test_short_rows_of_unaligned_blocks(nbits, HQ, S, append):
    """Rows that end in the first chunk, just past it, and at the capacity (4-bit at
    4127 not aligned)."""
    from tritonkv_amd.kernels import fused_decode_attention
    from tritonkv_amd.quantize import append_kv

    B, HKV, D, gs = 6, 2, 128, 32
    q, k, v, kq, vq = make_case(B, HQ, HKV, D, S, nbits, gs, seed=S, outlier_frac=0.0)
    lens = torch.tensor([1, 3, 31, 33, 290, S], dtype=torch.int32, device=DEV)
    new = {}
    want_k, want_v = kq.contiguous(), vq.contiguous()
    if append:
        g = torch.Generator().manual_seed(1)
        kn, vn = (torch.randn(B, HKV, D, generator=g).to(torch.float16).to(DEV) for _ in range(2))
        want_k, want_v = kq._map(torch.Tensor.clone), vq._map(torch.Tensor.clone)
        append_kv(want_k, kn[:, :, None], lens - 1)
        append_kv(want_v, vn[:, :, None], lens - 1)
        new = dict(k_new=kn, v_new=vn)
    out = fused_decode_attention(q, kq, vq, seq_lens=lens, num_splits=1, **new)
    for got, want in ((kq, want_k), (vq, want_v)):
        assert torch.equal(got.packed, want.packed)
        assert torch.equal(got.scale.view(torch.int16), want.scale.view(torch.int16))
    ref = oracle_attention_on_quant(q, want_k, want_v, seq_lens=lens.cpu().numpy())
    assert_close_to_reference(out, ref, f"nbits={nbits} append={append}")


@pytest.mark.parametrize("nbits,gs,HQ,S", [(4, 32, 8, 4127), (2, 32, 8, 8263), (4, 16, 32, 4099),
                                           (2, 128, 8, 8250), (4, 32, 12, 8251)])
def test_rows_before_the_block_do_not_show_what_lds_held(nbits, gs, HQ, S):
    """The rows masked before a block's start are not loaded: a launch over a
    cache of NaN scales and zero points leaves NaNs in every CU's LDS, and the
    next launch must not see them."""
    from tritonkv_amd.kernels import fused_decode_attention

    B, HKV = 160, 2  # more workgroups than compute units
    q, _, _, kq, vq = make_case(2, HQ, HKV, 128, S, nbits, gs, seed=S, outlier_frac=0.0)
    wide = [t._map(lambda x: x[:1].expand(B, *x.shape[1:]).contiguous()) for t in (kq, vq)]
    nan = [t._map(lambda x: x if x.dtype == torch.uint8 else torch.full_like(x, float("nan"))) for t in wide]
    qs = q[:1].expand(B, -1, -1).contiguous()
    want = fused_decode_attention(q[:1].contiguous(), *(t._map(lambda x: x[:1].contiguous())
                                                        for t in (kq, vq)), num_splits=1)
    assert not bool(want.isnan().any())
    assert bool(fused_decode_attention(qs, *nan, num_splits=1).isnan().all())
    got = fused_decode_attention(qs, *wide, num_splits=1)
    assert not bool(got.isnan().any())
    assert float((got - want).abs().max()) <= 2e-3


@pytest.mark.parametrize("fused_combine,ns", [(False, 1), (True, 2)])
def test_empty_rows_and_splits_of_unaligned_blocks(fused_combine, ns):
    """A row or split with no tokens runs no chunk, as where S is a multiple of 32."""
    from tritonkv_amd.kernels import fused_decode_attention

    B, S = 4, 8251
    q, _, _, kq, vq = make_case(B, 8, 2, 128, S, 4, 32, seed=5, outlier_frac=0.0)
    lens = torch.tensor([0, 4000, 0, S], dtype=torch.int32, device=DEV)
    even = [t._map(lambda x: torch.cat([x, x[:, :, :-S % 32]], 2).contiguous()) for t in (kq, vq)]
    got, want = (fused_decode_attention(q, *c, seq_lens=lens, num_splits=ns, fused_combine=fused_combine)
                 for c in ((kq, vq), even))
    assert torch.equal(got[::2].isnan(), want[::2].isnan())
    assert torch.equal(got[::2].nan_to_num(), want[::2].nan_to_num())
    assert float((got[1::2] - want[1::2]).abs().max()) <= 2e-3


@pytest.mark.parametrize("kb,vb,gs,HQ,S", [
    (4, 4, 32, 8, 16411),   # paired tiles, two splits of 8256
    (2, 2, 32, 8, 16417),   # 12 waves; S % 32 == 1, so unit 1 starts one row into its chunk
    (4, 2, 32, 16, 16385),  # 8 head columns
    (4, 4, 16, 40, 8225),   # two blocks of 16 query heads, one tile at a time, splits of 4160
    (2, 4, 64, 2, 16390),   # one query head
])
def test_later_splits_and_ordered_launches_of_unaligned_blocks(kb, vb, gs, HQ, S):
    """Second splits that start inside a chunk, rows that end in that chunk, at
    its start and one row past it; the ordered kernels bit for bit the same."""
    from tritonkv_amd.kernels import fused_decode_attention
    from tritonkv_amd.kernels.fused_decode_attn import plan_splits
    from tritonkv_amd.quantize import quantize_groupwise

    HKV = 2
    print(f"aligned splits K{kb}V{vb} gs{gs} HQ={HQ} S={S}", flush=True)
    q, _, v, kq, _ = make_case(5, HQ, HKV, 128, S, kb, gs, seed=S, outlier_frac=0.0)
    vq = quantize_groupwise(v, vb, gs)
    lo = plan_splits(S, 64, 2, 5, HKV, HQ // HKV)[2]
    lens = torch.tensor([S, lo, lo + 1, lo + 3, lo + 40], dtype=torch.int32, device=DEV)
    outs = [fused_decode_attention(q, kq, vq, seq_lens=lens, num_splits=2, allow_mixed_bits=kb != vb,
                                   dispatch_order=order, _workspace={}) for order in (False, True)]
    torch.cuda.synchronize()
    assert torch.equal(*outs)
    assert_close_to_reference(outs[0], oracle_attention_on_quant(q, kq, vq, seq_lens=lens.cpu().numpy()),
                              f"K{kb}V{vb} gs{gs} S={S}")
