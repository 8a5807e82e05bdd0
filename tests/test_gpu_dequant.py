"""GPU parity of the whole-cache dequantizer and code unpacker -- bit-exact.

``code * scale + zero`` is one rounding in fp32 (the product is exact) and one
more into a 16-bit dtype, so every value is determined to the bit.  Row counts
sit on both sides of a wave's batch of rows; metadata includes infinities, NaN
and zero scales, as a cache of non-finite input holds them.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import quant as oq

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _cache(rows, D, nbits, gs, seed):
    g = torch.Generator().manual_seed(seed)
    packed = torch.randint(0, 256, (rows, D * nbits // 8), generator=g, dtype=torch.uint8)
    scale = torch.rand(rows, D // gs, generator=g).to(torch.float16)
    zero = torch.randn(rows, D // gs, generator=g).to(torch.float16)
    for t, vals in ((scale, (float("inf"), 0.0, 6e-8)), (zero, (float("nan"), float("-inf"), -0.0))):
        flat = t.view(-1)
        for i, v in enumerate(vals):
            flat[(7 * i + 3) % flat.numel()] = v
    return packed, scale, zero


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("nbits", [2, 4])
@pytest.mark.parametrize("gs", [16, 32, 64, 128])
@pytest.mark.parametrize("rows", [1, 63, 130])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16, torch.float64])
def test_dequantize_matches_the_oracle_bitwise(D, nbits, gs, rows, dtype):
    if gs > D:
        pytest.skip("group larger than head_dim")
    from tritonkv_amd.quantize import QuantizedTensor, dequantize_groupwise

    packed, scale, zero = _cache(rows, D, nbits, gs, D + nbits + gs + rows)
    ref = oq.dequantize_groupwise(oq.QuantNP(packed.numpy(), scale.numpy(), zero.numpy(), nbits, gs, D))
    want = torch.from_numpy(ref).to(dtype)
    qt = QuantizedTensor(packed.to(DEV), scale.to(DEV), zero.to(DEV), nbits, gs, D)
    got = dequantize_groupwise(qt, dtype).cpu()
    assert got.dtype == dtype and got.shape == want.shape
    nan = want.isnan()
    assert torch.equal(got.isnan(), nan)
    ints = {2: torch.int16, 4: torch.int32, 8: torch.int64}[want.element_size()]
    assert torch.equal(got[~nan].view(ints), want[~nan].view(ints))


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("nbits", [2, 4])
@pytest.mark.parametrize("rows", [1, 63, 130])
def test_unpack_codes_matches_the_oracle(D, nbits, rows):
    from tritonkv_amd.quantize import unpack_codes

    packed, _, _ = _cache(rows, D, nbits, 16, rows)
    got = unpack_codes(packed.to(DEV), nbits, D).cpu().numpy()
    assert np.array_equal(got, oq.unpack_codes(packed.numpy(), nbits, D))
