"""The prompt quantizer (one head's tokens per workgroup) against the oracle, bit for bit.

Token counts sit on both sides of a workgroup's rows, with start positions
that leave the first and last rows outside the cache; the values hold what the
quotient by a corrected reciprocal must get right: ties, constant groups, and
scales that are fp16-subnormal, zero or infinite.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import quant as oq

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _values(shape, gs, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(shape, generator=g).view(*shape[:-1], -1, gs)
    kinds = torch.randint(0, 8, x.shape[:-1], generator=g)
    small = torch.tensor([1.0, 1e-4, 3e-7, 2e4])[torch.randint(0, 4, x.shape[:-1], generator=g)]
    x = torch.where((kinds == 1)[..., None], x * small[..., None], x)
    x = torch.where((kinds == 2)[..., None], torch.round(x * 2) / 2, x)  # ties
    x = torch.where((kinds == 3)[..., None], x[..., :1].expand_as(x), x)  # constant
    if dtype == torch.float32:
        x = torch.where((kinds == 4)[..., None], x * 1e-30 + 1.0, x)
        x = torch.where((kinds == 5)[..., None], x * 1e5 - 4.0, x)
    return x.reshape(shape).to(dtype)


@pytest.mark.parametrize("D,nbits,gs", [(128, 4, 32), (128, 2, 32), (128, 2, 128), (128, 4, 16),
                                        (64, 2, 16), (64, 4, 64)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("N", [32, 33, 161])
def test_tokens_at_positions_match_the_oracle_bitwise(D, nbits, gs, dtype, N):
    from tritonkv_amd.quantize import append_kv, empty_cache

    B, HKV, cap = 4, 3, 200
    x = _values((B, HKV, N, D), gs, dtype, D + nbits + gs + N)
    pos = [0, 7, cap - N + 5, -3]  # the third row's end and the fourth row's start do not fit
    cache = empty_cache(B, HKV, cap, D, nbits, gs, DEV)
    for t in (cache.packed, cache.scale, cache.zero):
        t.view(torch.uint8).fill_(0xA5)
    append_kv(cache, x.to(DEV), torch.tensor(pos, dtype=torch.int32, device=DEV))
    ref = oq.quantize_groupwise(x.numpy(), nbits, gs)
    for got, want in ((cache.packed, ref.packed), (cache.scale, ref.scale), (cache.zero, ref.zero)):
        got = got.cpu().numpy().view(np.uint8)
        want = np.ascontiguousarray(want).view(np.uint8)
        full = np.full_like(got, 0xA5)
        for b, p in enumerate(pos):
            t = [i for i in range(N) if 0 <= p + i < cap]
            full[b, :, p + t[0]:p + t[-1] + 1] = want[b, :, t[0]:t[-1] + 1]
        assert np.array_equal(got, full)


@pytest.mark.parametrize("nbits,gs", [(4, 32), (2, 128)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_several_steps_per_wave_match_the_oracle_bitwise(nbits, gs, dtype):
    """65536 rows or more: several steps per wave, the last tile of a head partly empty."""
    from tritonkv_amd.quantize import quantize_groupwise

    x = _values((1, 1, 65536 + 77, 128), gs, dtype, nbits)
    qt = quantize_groupwise(x.to(DEV), nbits, gs)
    ref = oq.quantize_groupwise(x.numpy(), nbits, gs)
    assert np.array_equal(qt.packed.cpu().numpy(), ref.packed)
    assert np.array_equal(qt.scale.cpu().numpy().view(np.uint16), ref.scale.view(np.uint16))
    assert np.array_equal(qt.zero.cpu().numpy().view(np.uint16), ref.zero.view(np.uint16))


@pytest.mark.parametrize("nbits,gs,D", [(4, 32, 128), (2, 64, 128), (2, 32, 64)])
@pytest.mark.parametrize("B,HKV,N", [(2, 3, 15), (2, 3, 31), (2, 3, 57), (2, 3, 65),  # small workgroups
                                     (512, 4, 32), (512, 4, 33), (256, 4, 64), (256, 4, 96),
                                     (256, 4, 111), (256, 4, 112), (256, 4, 129), (128, 4, 256)])
def test_prompts_on_both_sides_of_the_fill_rule(nbits, gs, D, B, HKV, N):
    """By head or all heads together: the same rows as one long run of them."""
    from tritonkv_amd.quantize import append_kv, empty_cache, quantize_groupwise

    print(f"fill rule {nbits}-bit gs{gs} D={D} B={B} HKV={HKV} N={N}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(N)
    x = torch.randn(B, HKV, N, D, device=DEV, generator=g, dtype=torch.float16)
    got = append_kv(empty_cache(B, HKV, N, D, nbits, gs, DEV), x)
    want = quantize_groupwise(x.view(1, 1, -1, D), nbits, gs)
    for a, b in ((got.packed, want.packed), (got.scale, want.scale), (got.zero, want.zero)):
        assert torch.equal(a.view(-1, a.shape[-1]), b.view(-1, b.shape[-1]))
