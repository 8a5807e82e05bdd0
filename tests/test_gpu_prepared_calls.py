"""Repeated decode calls through a workspace: every form that must not reuse the
checked call, on the paged and per-channel entry points and with tensors that
change behind an unchanged address; results against calls without a workspace."""

from __future__ import annotations

import pytest
import torch

from tests.helpers import make_case

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _paged(B=3, HQ=8, HKV=2, page=32, pages=4):
    from tritonkv_amd.paged import empty_paged_pool, paged_append

    g = torch.Generator().manual_seed(5)
    table = torch.randperm(B * pages, generator=g).to(torch.int32).view(B, pages).to(DEV)
    pools = []
    for _ in range(2):
        pool = empty_paged_pool(B * pages, HKV, page, 128, 4, 32, DEV)
        x = torch.randn(B, HKV, page * pages, 128, generator=g).to(torch.float16).to(DEV)
        pools.append(paged_append(pool, x, table, torch.zeros(B, dtype=torch.int32, device=DEV)))
    lens = torch.tensor([5, 77, 128], dtype=torch.int32, device=DEV)
    q = torch.randn(B, HQ, 128, generator=g).to(torch.float16).to(DEV)
    return q, pools, table, lens


def test_paged_calls_reuse_only_the_checked_form():
    from tritonkv_amd.paged import paged_decode_attention

    q, (kp, vp), table, lens = _paged()
    ws, out = {}, torch.empty(3, 8, 128, device=DEV)

    def both(q, table, lens, **kw):
        got = paged_decode_attention(q, kp, vp, table, lens, out=kw.pop("out", out), _workspace=ws, **kw)
        return torch.equal(got, paged_decode_attention(q, kp, vp, table, lens, **kw))

    assert both(q, table, lens) and "call" in ws
    prep = ws["call"]
    assert both(q * 2, table, lens) and both(q, table, lens, out=None) and ws["call"] is prep
    lens.fill_(9)  # lengths change in place on the device
    assert both(q, table, lens) and ws["call"] is prep
    assert both(q.float(), table, lens) and ws["call"] is not prep
    assert both(q, table.clone(), lens) and both(q, table, lens.clone()) and both(q, table, None)
    assert both(q, table.t().contiguous().t(), lens)              # a strided table
    assert both(q, table, torch.stack([lens, lens], 1)[:, 0])     # strided lengths
    assert both(q, table, lens, num_splits=2) and both(q, table, lens, sm_scale=0.2)
    wide = torch.randn(3, 8, 256, device=DEV).to(torch.float16)
    assert both(wide[..., :128], table, lens)                     # a strided q
    with pytest.raises(ValueError):
        paged_decode_attention(q, kp, vp, table, lens.long(), out=out, _workspace=ws)


def test_strided_new_tokens_are_not_read_as_contiguous():
    from tritonkv_amd.kernels import fused_decode_attention

    q, _, _, kq, vq = make_case(2, 8, 2, 128, 96, 4, 32, seed=3)
    lens = torch.tensor([40, 96], dtype=torch.int32, device=DEV)
    new = torch.randn(2, 2, 2, 128, device=DEV).to(torch.float16)
    ws = {}
    for step in range(3):
        kn, vn = new[:, :, 0], new[:, :, 1]  # rows of one projection, not contiguous
        got = fused_decode_attention(q, kq, vq, seq_lens=lens, k_new=kn, v_new=vn, _workspace=ws)
        want = fused_decode_attention(q, kq, vq, seq_lens=lens, k_new=kn.contiguous(),
                                      v_new=vn.contiguous())
        assert torch.equal(got, want), step
        new = new * 0.5


def test_a_workspace_shared_by_two_entry_points_keeps_its_buffers():
    """The second entry point replaces the workspace's partials; the first call's
    argument block still points into its own."""
    from tritonkv_amd.kernels import fp16_decode_attention, fused_decode_attention

    q, k, v, kq, vq = make_case(1, 8, 2, 128, 3000, 4, 32, seed=4)
    ws = {}
    want = fused_decode_attention(q, kq, vq, num_splits=4)
    assert torch.equal(fused_decode_attention(q, kq, vq, num_splits=4, _workspace=ws), want)
    prep = ws["call"]
    want16 = fp16_decode_attention(q, k, v, num_splits=9)
    assert torch.equal(fp16_decode_attention(q, k, v, num_splits=9, _workspace=ws), want16)
    junk = [torch.full((1 << 16,), float("nan"), device=DEV) for _ in range(4)]
    ws["call"] = prep  # as a caller's copy of the workspace would hold it
    assert torch.equal(fused_decode_attention(q, kq, vq, num_splits=4, _workspace=ws), want)
    assert all(bool(t.isnan().all()) for t in junk)


def test_channel_attend_follows_lengths_and_tensors():
    from tritonkv_amd.channel import ChannelKVCache, channel_decode_attention

    g = torch.Generator().manual_seed(6)
    cache = ChannelKVCache(2, 2, 256, 128, device=DEV)
    out = torch.empty(2, 8, 128, device=DEV)
    for n in (70, 1, 40):
        k, v = (torch.randn(2, 2, n, 128, generator=g).to(torch.float16).to(DEV) for _ in range(2))
        cache.extend(k, v)
        for dtype in (torch.float16, torch.float32, torch.float16):
            q = torch.randn(2, 8, 128, generator=g).to(dtype).to(DEV)
            for o in (out, None):
                got = cache.attend(q, out=o)
                want = channel_decode_attention(q, cache.keys, cache.values, cache.k_res, cache.v_res,
                                                cache._qlens, cache._rlens, equal_lengths=True)
                assert torch.equal(got, want)


def test_another_stream_and_a_side_thread():
    import threading

    from tritonkv_amd.kernels import fused_decode_attention

    q, _, _, kq, vq = make_case(1, 8, 2, 128, 600, 4, 32, seed=7)
    want, ws, got = fused_decode_attention(q, kq, vq), {}, []
    fused_decode_attention(q, kq, vq, _workspace=ws)
    torch.cuda.synchronize()

    def work():
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            got.append(fused_decode_attention(q, kq, vq, _workspace=ws))
        s.synchronize()

    t = threading.Thread(target=work)
    t.start(), t.join()
    assert torch.equal(got[0], want)


def test_everything_runs_without_the_native_module(monkeypatch):
    """The C ABI is all the kernels need; calls are then checked in full each time."""
    import sys

    from tritonkv_amd import _lib
    from tritonkv_amd.kernels import fused_decode_attention
    from tritonkv_amd.quantize import dequantize_groupwise, quantize_groupwise

    q, k, _, kq, vq = make_case(1, 8, 2, 128, 600, 4, 32, seed=8)
    want = fused_decode_attention(q, kq, vq), dequantize_groupwise(kq)
    monkeypatch.setattr(_lib, "_HOST", None)
    monkeypatch.setattr(_lib, "_HOST_SOUGHT", False)
    monkeypatch.delattr("tritonkv_amd._hostcall", raising=False)
    monkeypatch.setitem(sys.modules, "tritonkv_amd._hostcall", None)
    monkeypatch.setattr(_lib, "_LIB", None)
    ws = {}
    with pytest.warns(RuntimeWarning, match="_hostcall"):
        again = quantize_groupwise(k, 4, 32)
    for _ in range(2):
        assert torch.equal(fused_decode_attention(q, again, vq, _workspace=ws), want[0])
    assert "call" not in ws and torch.equal(dequantize_groupwise(again), want[1])
