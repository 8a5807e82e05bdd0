"""A prompt into a per-channel cache: layouts, lengths and storage alignment, bit for bit.

``extend`` reads K and V in the layout they have.  Every form is compared with
the same tokens quantized through the two quantizers (each bit-exact with the
oracle) from contiguous copies.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import channel as och

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _kv(B, HKV, N, D, layout, seed):
    g = torch.Generator().manual_seed(seed)
    out = []
    for _ in range(2):
        x = (torch.randn(B, HKV, N, D, generator=g) * 2).to(torch.float16)
        x[..., 3] *= 9
        x[0, 0, N // 2, 5] = float("inf")
        x = x.to(DEV)
        if layout == "tokens":          # (B, N, HKV, D) in memory
            x = x.transpose(1, 2).contiguous().transpose(1, 2)
        elif layout == "slice":         # a slice of a longer prompt
            x = torch.cat([x[:, :, :1], x, x], 2)[:, :, 1:N + 1]
        elif layout == "heads":         # one head's rows, expanded
            x = x[:, :1].expand(B, HKV, N, D)
        elif layout == "unaligned":     # rows that start 2 bytes off
            buf = torch.empty(B, HKV, N, D + 1, dtype=x.dtype, device=DEV)
            buf[..., 1:] = x
            x = buf[..., 1:]
        elif layout == "strided":       # channels not adjacent
            x = x.repeat_interleave(2, -1)[..., ::2]
        out.append(x)
    return out


def _tensors(c):
    return {"kp": c.keys.packed, "ks": c.keys.scale, "kz": c.keys.zero, "vp": c.values.packed,
            "vs": c.values.scale, "vz": c.values.zero, "kr": c.k_res, "vr": c.v_res}


@pytest.mark.parametrize("layout", ["heads_major", "tokens", "slice", "heads", "unaligned", "strided"])
@pytest.mark.parametrize("N", [1, 31, 32, 33, 197])
@pytest.mark.parametrize("D,kb,vb,gs", [(128, 2, 2, 32), (128, 4, 2, 16), (64, 2, 4, 32), (64, 4, 4, 64)])
def test_extend_matches_the_quantizers_bitwise(layout, N, D, kb, vb, gs):
    from tritonkv_amd.channel import ChannelKVCache, append_keys_per_channel
    from tritonkv_amd.quantize import append_kv

    B, HKV = 3, 2
    k, v = _kv(B, HKV, N, D, layout, N + D)
    got = ChannelKVCache(B, HKV, 320, D, kb, vb, gs, device=DEV)
    want = ChannelKVCache(B, HKV, 320, D, kb, vb, gs, device=DEV)
    got.extend(k, v)
    whole = N // 32 * 32
    if whole:
        append_keys_per_channel(want.keys, k[:, :, :whole].contiguous())
        append_kv(want.values, v[:, :, :whole].contiguous())
    want.k_res[:, :, :N - whole] = k[:, :, whole:]
    want.v_res[:, :, :N - whole] = v[:, :, whole:]
    for name, t in _tensors(want).items():
        assert torch.equal(_tensors(got)[name].view(torch.uint8), t.view(torch.uint8)), name
    assert len(got) == N and (got.quantized, got.window) == (whole, N - whole)
    assert got._qlens.tolist() == [whole] * B and got._rlens.tolist() == [N - whole] * B
    # a second prompt into the open window, then past it, equals one prompt of both
    k2, v2 = _kv(B, HKV, 70, D, layout, 1000 + N)
    got.extend(k2, v2)
    both = ChannelKVCache(B, HKV, 320, D, kb, vb, gs, device=DEV)
    both.extend(torch.cat([k, k2], 2), torch.cat([v, v2], 2))
    n = both.quantized
    for name, t in _tensors(both).items():
        rows = {"kr": both.window, "vr": both.window, "ks": n // 32, "kz": n // 32}.get(name, n)
        a, b = (x[:, :, :rows].contiguous().view(torch.uint8) for x in (_tensors(got)[name], t))
        assert torch.equal(a, b), name
    assert got._qlens.tolist() == both._qlens.tolist() and got._rlens.tolist() == both._rlens.tolist()


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("nbits", [2, 4])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_key_quantizer_from_unaligned_storage_matches_the_oracle(D, nbits, dtype):
    """Pairs of channels not loadable as one aligned word; an odd number of blocks."""
    from tritonkv_amd.channel import quantize_keys_per_channel

    g = torch.Generator().manual_seed(D + nbits)
    k = (torch.randn(1, 3, 5 * 32, D, generator=g) * 2).to(dtype)
    k[..., 7] = torch.round(k[..., 7] * 4) / 4  # ties
    k[..., 8] *= 1e-6                           # a subnormal scale
    buf = torch.empty(k.numel() + 1, dtype=dtype, device=DEV)
    x = buf[1:].view(k.shape)
    x.copy_(k)
    ck = quantize_keys_per_channel(x, nbits)
    ref = och.quantize_keys_per_channel(k.numpy(), nbits)
    assert np.array_equal(ck.packed.cpu().numpy(), ref.packed)
    assert np.array_equal(ck.scale.cpu().numpy().view(np.uint16), ref.scale.view(np.uint16))
    assert np.array_equal(ck.zero.cpu().numpy().view(np.uint16), ref.zero.view(np.uint16))
