"""What a user of this framework has it do, as cases to time.

Every case goes through the package's Python entry points as a serving program
calls them: the decode step over quantized caches (contiguous, ragged with the
append fused in, paged), the fp16 control, per-channel keys with an fp16
window, and the two directions of the codec that surround decoding: quantizing
a prompt's K and V, and dequantizing a cache.

A case is a dict with ``kind`` and the sizes of that kind; ``listed`` are the
shapes of the repository's benchmark, tests and ``transformers`` cache, and
generic sizes beside them; ``draw`` gives others of the same ranges.  K and V
are N(0, 1) with four channels per KV head scaled by 8 (fixed outlier channels,
as the benchmark's); every tensor is drawn on the GPU from the seed, one
generator per batch row, so ``exact`` can redraw one row at a time.
"""

from __future__ import annotations

import math

import torch

from tritonkv_amd.channel import ChannelKVCache
from tritonkv_amd.kernels import fp16_decode_attention, fused_decode_attention
from tritonkv_amd.paged import empty_paged_pool, paged_append, paged_decode_attention
from tritonkv_amd.quantize import (QuantizedTensor, append_kv, dequantize_groupwise, empty_cache,
                                   quantize_kv)

DEV = "cuda"
OUTLIERS, OUTLIER_SCALE = 4, 8.0
KEY_BLOCK = 32  # tokens of one per-channel key group
DTYPES = {"float16": torch.float16, "bfloat16": torch.bfloat16, "float32": torch.float32}


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------


def _decode(name, B, HQ, HKV, D, S, k_bits, v_bits, gs, lengths="full", append=False,
            q="float16"):
    return dict(name=name, kind="decode", B=B, HQ=HQ, HKV=HKV, D=D, S=S, k_bits=k_bits,
                v_bits=v_bits, gs=gs, lengths=lengths, append=append, q=q)


def listed():
    return [
        # The smallest call: one sequence of the Qwen2.5-1.5B shape, a short chat.
        _decode("decode_b1_short", 1, 12, 2, 128, 512, 4, 4, 32),
        # One sequence far into a long context, the step of a transformers
        # cache: length on the device, the new token appended by the call.
        _decode("decode_b1_long", 1, 12, 2, 128, 16001, 4, 4, 32, "equal", True),
        # A small batch of a model with head dim 64, odd length, fp32 q.
        _decode("decode_d64", 8, 32, 8, 64, 2999, 4, 4, 64, q="float32"),
        # The benchmark's headline: Llama-3-8B attention, 32 sequences at 32k.
        _decode("decode_8b_4bit", 32, 32, 8, 128, 32768, 4, 4, 32),
        # The same model at 2 bits and an odd length.
        _decode("decode_8b_2bit", 32, 32, 8, 128, 24571, 2, 2, 32),
        # A 70B-style continuous batch: 4-bit K, 2-bit V, lengths from 1k to
        # 64k, every sequence's new token appended by the call.
        _decode("decode_70b_ragged", 32, 64, 8, 128, 65536, 4, 2, 32, "ragged", True),
        # A serving engine's step: shuffled 64-token pages, ragged, fused append.
        dict(name="paged_decode", kind="paged", B=16, HQ=32, HKV=8, D=128, S=8192, page=64,
             k_bits=4, v_bits=4, gs=32, q="float16"),
        # The fp16 cache of the same engine (the unquantized control).
        dict(name="fp16_decode", kind="fp16", B=16, HQ=12, HKV=2, D=128, S=8192, q="float16"),
        # 2-bit per-channel keys: attention over history and window.
        dict(name="channel_attend", kind="channel_attend", B=16, HQ=32, HKV=8, D=128, S=16403,
             k_bits=2, v_bits=2, gs=32, q="float16"),
        # A prompt going into such a cache, as the projections leave K and V
        # (token-major, viewed as (B, HKV, N, D)), its length no multiple of 32.
        dict(name="channel_prefill", kind="channel_prefill", B=4, HKV=8, D=128, S=8213, k_bits=2,
             v_bits=2, gs=32, x="float16"),
        # A prompt's K and V quantized per token.
        dict(name="quantize", kind="quantize", B=4, HKV=8, D=128, S=16384, bits=4, gs=32,
             x="float16"),
        # A cache turned back into fp16, as a prefix handed to dense attention.
        dict(name="dequantize", kind="dequantize", B=2, HKV=8, D=128, S=8191, bits=4, gs=32,
             out="float16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "paged", "fp16", "channel_attend",
                       "channel_prefill", "quantize", "dequantize"])
    D = rng.choice([128, 128, 128, 64])
    HKV = rng.choice([1, 2, 4, 8])
    G = rng.choice([1, 2, 4, 6, 7, 8, 12, 16])
    bits, gs = rng.choice([2, 4]), rng.choice([g for g in (16, 32, 32, 64, 128) if g <= D])
    q = rng.choice(["float16", "float16", "float32"])
    x = rng.choice(["float16", "float16", "float32"])
    if kind == "decode":
        B = _log(rng, 1, 64)
        lengths = rng.choice(["full", "equal", "ragged"])
        S = _log(rng, 100, min(65536 if lengths == "ragged" else 32768, 4_000_000 // (B * HKV)))
        k_bits, v_bits = rng.choice([(4, 4), (2, 2), (4, 2)])
        c = _decode("", B, HKV * G, HKV, D, S, k_bits, v_bits, gs, lengths,
                    lengths != "full" and rng.random() < 0.7, q)
        del c["name"]
        return c
    if kind == "paged":
        B, page = _log(rng, 1, 64), rng.choice([32, 64, 128, 256])
        S = -(-_log(rng, 200, min(32768, 2_000_000 // (B * HKV))) // page) * page
        return dict(kind=kind, B=B, HQ=HKV * G, HKV=HKV, D=D, S=S, page=page, k_bits=bits,
                    v_bits=bits, gs=gs, q=q)
    if kind == "fp16":
        B = _log(rng, 1, 64)
        S = _log(rng, 100, min(32768, 1_000_000 // (B * HKV)))
        return dict(kind=kind, B=B, HQ=HKV * G, HKV=HKV, D=D, S=S, q=q)
    if kind in ("channel_attend", "channel_prefill"):
        B = _log(rng, 1, 32)
        S = _log(rng, 100, min(32768, 2_000_000 // (B * HKV)))
        c = dict(kind=kind, B=B, HKV=HKV, D=D, S=S, k_bits=rng.choice([2, 4]),
                 v_bits=rng.choice([2, 4]), gs=rng.choice([16, 32]))
        return dict(c, HQ=HKV * G, q=q) if kind == "channel_attend" else dict(c, x=x)
    B = _log(rng, 1, 16)
    if kind == "quantize":
        S = _log(rng, 20, min(32768, 1_000_000 // (B * HKV)))
        return dict(kind=kind, B=B, HKV=HKV, D=D, S=S, bits=bits, gs=gs, x=x)
    S = _log(rng, 100, min(32768, 1_000_000 // (B * HKV)))
    return dict(kind=kind, B=B, HKV=HKV, D=D, S=S, bits=bits, gs=gs,
                out=rng.choice(["float16", "bfloat16", "float32"]))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------


def _gen(seed, row):
    return torch.Generator(device=DEV).manual_seed(seed * 1_000_003 + 7919 * (row + 2))


def _multipliers(c, seed):
    """(HKV, D): 8 at four channels of each KV head, else 1."""
    g = _gen(seed, -2)
    m = torch.ones(c["HKV"], c["D"], device=DEV)
    for h in range(c["HKV"]):
        m[h, torch.randperm(c["D"], device=DEV, generator=g)[:OUTLIERS]] = OUTLIER_SCALE
    return m


def _row_kv(c, seed, b, L, mult, dtype=torch.float16):
    """K and V of batch row b: (HKV, L, D) each."""
    g = _gen(seed, b)
    return [torch.randn(c["HKV"], L, c["D"], device=DEV, generator=g, dtype=dtype)
            .mul_(mult[:, None].to(dtype)) for _ in range(2)]


def _q_and_new(c, seed):
    g = _gen(seed, -1)
    q = torch.randn(c["B"], c["HQ"], c["D"], device=DEV, generator=g).to(DTYPES[c["q"]])
    new = [torch.randn(c["B"], c["HKV"], c["D"], device=DEV, generator=g, dtype=torch.float16)
           for _ in range(2)]
    return q, new


def _lengths(c, seed):
    """Tokens of each batch row, as host numbers."""
    if c["kind"] != "paged" and c.get("lengths") != "ragged":
        return [c["S"]] * c["B"]
    lo = max(1, c["S"] // 64) if c["kind"] == "decode" else max(1, c["S"] // 16)
    g = torch.Generator().manual_seed(seed)
    return [int(n) for n in torch.randint(lo, c["S"] + 1, (c["B"],), generator=g)]


def _capacity(c):
    """Room for growth where the lengths live on the device, as a serving loop keeps."""
    return c["S"] if c["lengths"] != "equal" else -(-(c["S"] + 1) // 512) * 512


def _zeroed(cache):
    for t in (cache.packed, cache.scale, cache.zero):
        t.zero_()
    return cache


def _int32(values):
    return torch.tensor(values, dtype=torch.int32, device=DEV)


def _prepare_decode(c, seed):
    B, HKV, D = c["B"], c["HKV"], c["D"]
    lens, mult = _lengths(c, seed), _multipliers(c, seed)
    cap = _capacity(c)
    kc = _zeroed(empty_cache(B, HKV, cap, D, c["k_bits"], c["gs"], DEV))
    vc = _zeroed(empty_cache(B, HKV, cap, D, c["v_bits"], c["gs"], DEV))
    for b in range(B):
        for cache, x in zip((kc, vc), _row_kv(c, seed, b, lens[b], mult)):
            append_kv(QuantizedTensor(cache.packed[b:b + 1], cache.scale[b:b + 1],
                                      cache.zero[b:b + 1], cache.nbits, c["gs"], D), x[None])
    q, (k_new, v_new) = _q_and_new(c, seed)
    kw = dict(out=torch.empty(B, c["HQ"], D, device=DEV), _workspace={},
              allow_mixed_bits=c["k_bits"] != c["v_bits"])
    if c["lengths"] != "full":
        kw.update(seq_lens=_int32(lens), equal_lengths=c["lengths"] == "equal")
    if c["append"]:
        kw.update(k_new=k_new, v_new=v_new)
    return dict(case=c, q=q, kc=kc, vc=vc, kw=kw)


def _prepare_paged(c, seed):
    B, HKV, D, page = c["B"], c["HKV"], c["D"], c["page"]
    lens, mult, per_row = _lengths(c, seed), _multipliers(c, seed), c["S"] // c["page"]
    table = torch.randperm(B * per_row, device=DEV, generator=_gen(seed, -3))
    table = table.to(torch.int32).view(B, per_row)
    kp = _zeroed(empty_paged_pool(B * per_row, HKV, page, D, c["k_bits"], c["gs"], DEV))
    vp = _zeroed(empty_paged_pool(B * per_row, HKV, page, D, c["v_bits"], c["gs"], DEV))
    start = _int32([0])
    for b in range(B):
        for pool, x in zip((kp, vp), _row_kv(c, seed, b, lens[b], mult)):
            paged_append(pool, x[None], table[b:b + 1], start)
    q, (k_new, v_new) = _q_and_new(c, seed)
    kw = dict(out=torch.empty(B, c["HQ"], D, device=DEV), _workspace={}, k_new=k_new, v_new=v_new)
    return dict(case=c, q=q, kc=kp, vc=vp, table=table, lens=_int32(lens), kw=kw)


def _batch_kv(c, seed, dtype=torch.float16, token_major=False):
    """K and V of the whole batch, (B, HKV, S, D); token_major: laid out (B, S, HKV, D)."""
    B, HKV, S, D = c["B"], c["HKV"], c["S"], c["D"]
    shape = (B, S, HKV, D) if token_major else (B, HKV, S, D)
    full = [torch.empty(shape, device=DEV, dtype=dtype) for _ in range(2)]
    full = [t.transpose(1, 2) if token_major else t for t in full]
    mult = _multipliers(c, seed)
    for b in range(B):
        for t, x in zip(full, _row_kv(c, seed, b, S, mult, dtype)):
            t[b].copy_(x)
    return full


def prepare(case, seed):
    c = case
    kind = c["kind"]
    if kind == "decode":
        return _prepare_decode(c, seed)
    if kind == "paged":
        return _prepare_paged(c, seed)
    if kind == "fp16":
        k, v = _batch_kv(c, seed)
        kw = dict(out=torch.empty(c["B"], c["HQ"], c["D"], device=DEV), _workspace={})
        return dict(case=c, q=_q_and_new(c, seed)[0], k=k, v=v, kw=kw)
    if kind in ("channel_attend", "channel_prefill"):
        cache = ChannelKVCache(c["B"], c["HKV"], c["S"] + 64, c["D"], k_nbits=c["k_bits"],
                               v_nbits=c["v_bits"], group_size=c["gs"], device=DEV)
        if kind == "channel_prefill":
            k, v = _batch_kv(c, seed, DTYPES[c["x"]], token_major=True)
            return dict(case=c, cache=cache, k=k, v=v)
        cache.extend(*_batch_kv(c, seed))
        return dict(case=c, cache=cache, q=_q_and_new(c, seed)[0],
                    out=torch.empty(c["B"], c["HQ"], c["D"], device=DEV))
    if kind == "quantize":
        k, v = _batch_kv(c, seed, DTYPES[c["x"]])
        return dict(case=c, k=k, v=v)
    kq, vq = quantize_kv(*_batch_kv(c, seed), c["bits"], c["gs"])
    return dict(case=c, kq=kq, vq=vq)


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------


def _cache_tensors(kc, vc):
    return {"k": [kc.packed, kc.scale, kc.zero], "v": [vc.packed, vc.scale, vc.zero]}


def run(state):
    c = state["case"]
    kind = c["kind"]
    if kind == "decode":
        out = fused_decode_attention(state["q"], state["kc"], state["vc"], **state["kw"])
        return dict(_cache_tensors(state["kc"], state["vc"]), out=out) if c["append"] else {"out": out}
    if kind == "paged":
        out = paged_decode_attention(state["q"], state["kc"], state["vc"], state["table"],
                                     state["lens"], **state["kw"])
        return dict(_cache_tensors(state["kc"], state["vc"]), out=out)
    if kind == "fp16":
        return {"out": fp16_decode_attention(state["q"], state["k"], state["v"], **state["kw"])}
    if kind == "channel_attend":
        return {"out": state["cache"].attend(state["q"], out=state["out"])}
    if kind == "channel_prefill":
        cache = state["cache"]
        cache.reset()
        cache.extend(state["k"], state["v"])
        return dict(_cache_tensors(cache.keys, cache.values), window=[cache.k_res, cache.v_res])
    if kind == "quantize":
        return _cache_tensors(*quantize_kv(state["k"], state["v"], c["bits"], c["gs"]))
    dtype = DTYPES[c["out"]]
    return [dequantize_groupwise(t, dtype) for t in (state["kq"], state["vq"])]


# ---------------------------------------------------------------------------
# the work a pass cannot do without, and how exact its outputs are
# ---------------------------------------------------------------------------


def _row_bytes(D, bits, gs):
    return D * bits // 8 + 4 * (D // gs)


def work(case):
    c = case
    kind, B, HKV, D, S = c["kind"], c["B"], c["HKV"], c["D"], c["S"]
    size = {"float16": 2, "bfloat16": 2, "float32": 4}
    if kind == "quantize":
        rows = 2 * B * HKV * S
        return {"bytes": rows * (D * size[c["x"]] + _row_bytes(D, c["bits"], c["gs"])),
                "flops": rows * D * 6}
    if kind == "dequantize":
        rows = 2 * B * HKV * S
        return {"bytes": rows * (D * size[c["out"]] + _row_bytes(D, c["bits"], c["gs"])),
                "flops": rows * D * 2}
    if kind == "channel_prefill":
        whole = S // KEY_BLOCK * KEY_BLOCK
        rows, rest = B * HKV * whole, B * HKV * (S - whole)
        kv = _row_bytes(D, c["k_bits"], KEY_BLOCK) + _row_bytes(D, c["v_bits"], c["gs"])
        return {"bytes": rows * (2 * D * size[c["x"]] + kv) + rest * 2 * D * (size[c["x"]] + 2),
                "flops": 2 * rows * D * 6}
    # decoding: the caches once, q once, the output once
    HQ = c["HQ"]
    if c.get("lengths") == "ragged":
        tokens = B * (max(1, S // 64) + S) // 2
    elif kind == "paged":
        tokens = B * (max(1, S // 16) + S) // 2
    else:
        tokens = B * S
    if kind == "fp16":
        row = 4 * D
    elif kind == "channel_attend":
        row = _row_bytes(D, c["k_bits"], KEY_BLOCK) + _row_bytes(D, c["v_bits"], c["gs"])
    else:
        row = _row_bytes(D, c["k_bits"], c["gs"]) + _row_bytes(D, c["v_bits"], c["gs"])
    return {"bytes": tokens * HKV * row + B * HQ * D * (size[c["q"]] + 4),
            "flops": 4 * tokens * HQ * D}


def tolerance(case):
    # Codes, fp16 scales and zeros, and dequantized values are defined to the bit.
    if case["kind"] in ("quantize", "dequantize", "channel_prefill"):
        return "exact"
    # fp16 probabilities in the PV products, fp32 sums: three to six times the
    # distance from 64 bits seen over the listed and drawn cases (the fp16 cache
    # up to 7e-5, the quantized ones, whose scaled probabilities are rounded to
    # fp16 once more, up to 8e-4), and ten times that for a single value.
    rel = 4e-4 if case["kind"] == "fp16" else 2.5e-3
    return {"rel": rel, "max": 10 * rel}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------


def _groupwise(x, bits, dim):
    """(scale, zero, dequantized) in 64 bits of groups along `dim`: scale and
    zero rounded to fp16 before the codes are taken, as the format has it."""
    x, qmax = x.float(), 2 ** bits - 1
    mn, mx = x.amin(dim, keepdim=True), x.amax(dim, keepdim=True)
    sc = (mx - mn) / qmax
    sc = torch.where(sc > 0, sc, torch.ones_like(sc))
    s16, z16 = sc.half().float(), mn.half().float()
    codes = torch.round((x - z16) / s16).clamp_(0, qmax)
    return sc.double(), mn.double(), codes.double() * s16.double() + z16.double()


def _per_token(x, bits, gs):
    """x (..., D), groups of gs dims: scale and zero (..., D / gs), values (..., D)."""
    sc, zr, y = _groupwise(x.unflatten(-1, (-1, gs)), bits, -1)
    return sc.squeeze(-1), zr.squeeze(-1), y.flatten(-2)


def _per_channel(x, bits):
    """x (HKV, n * 32, D), one group per (32 tokens, channel)."""
    sc, zr, y = _groupwise(x.unflatten(1, (-1, KEY_BLOCK)), bits, 2)
    return sc.squeeze(2), zr.squeeze(2), y.flatten(1, 2)


def _attend(q, k, v, D):
    """q (HQ, D), k and v (HKV, L, D), all float64."""
    HKV = k.shape[0]
    s = torch.bmm(q.view(HKV, -1, D), k.transpose(1, 2).contiguous()) / math.sqrt(D)
    return torch.bmm(torch.softmax(s, -1), v.contiguous()).reshape(-1, D)


def _exact_row(c, seed, b, L, mult, new):
    """K and V of batch row b as the decode step sees them, float64 (HKV, L, D)."""
    k, v = _row_kv(c, seed, b, L, mult)
    if c["kind"] == "fp16":
        return k.double(), v.double()
    if c["kind"] == "channel_attend":
        n = L // KEY_BLOCK * KEY_BLOCK
        v64 = _per_token(v[:, :n], c["v_bits"], c["gs"])[2]
        k64 = _per_channel(k[:, :n], c["k_bits"])[2] if n else k[:, :0].double()
        return torch.cat([k64, k[:, n:].double()], 1), torch.cat([v64, v[:, n:].double()], 1)
    if c["kind"] == "paged" or c["append"]:
        k[:, L - 1], v[:, L - 1] = new[0][b], new[1][b]
    return _per_token(k, c["k_bits"], c["gs"])[2], _per_token(v, c["v_bits"], c["gs"])[2]


def _exact_prefill(c, seed, mult):
    """Scales, zeros and windows of a prefilled per-channel cache (zeros where nothing is written)."""
    B, HKV, D, S = c["B"], c["HKV"], c["D"], c["S"]
    n, cap = S // KEY_BLOCK * KEY_BLOCK, -(-(S + 64) // KEY_BLOCK) * KEY_BLOCK
    k = [torch.zeros(B, HKV, cap // KEY_BLOCK, D, device=DEV, dtype=torch.float64) for _ in range(2)]
    v = [torch.zeros(B, HKV, cap, D // c["gs"], device=DEV, dtype=torch.float64) for _ in range(2)]
    w = [torch.zeros(B, HKV, KEY_BLOCK, D, device=DEV, dtype=torch.float64) for _ in range(2)]
    for b in range(B):
        x = [t.half() for t in _row_kv(c, seed, b, S, mult, DTYPES[c["x"]])]  # the cache takes fp16
        for t, y in zip(w, x):
            t[b, :, :S - n] = y[:, n:].double()
        if n:
            for i, (kk, vv) in enumerate(zip(_per_channel(x[0][:, :n], c["k_bits"])[:2],
                                             _per_token(x[1][:, :n], c["v_bits"], c["gs"])[:2])):
                k[i][b, :, :n // KEY_BLOCK], v[i][b, :, :n] = kk, vv
    return {"k": [None] + k, "v": [None] + v, "window": w}


def exact(case, seed):
    c = case
    kind, D = c["kind"], c["D"]
    mult = _multipliers(c, seed)
    if kind in ("quantize", "dequantize"):
        outs = []
        for which in range(2):
            rows = []
            for b in range(c["B"]):
                x = _row_kv(c, seed, b, c["S"], mult, DTYPES[c.get("x", "float16")])[which]
                rows.append(_per_token(x, c["bits"], c["gs"]))
            outs.append([torch.stack([r[i] for r in rows]) for i in range(3)])
        if kind == "dequantize":
            return [o[2] for o in outs]
        return {"k": [None, outs[0][0], outs[0][1]], "v": [None, outs[1][0], outs[1][1]]}
    if kind == "channel_prefill":
        return _exact_prefill(c, seed, mult)
    q, new = _q_and_new(c, seed)
    q = q.half().double()  # the decode step takes q in fp16
    out = []
    for b, L in enumerate(_lengths(c, seed)):
        k, v = _exact_row(c, seed, b, L, mult, new)
        out.append(_attend(q[b], k, v, D))
    res = {"out": torch.stack(out)}
    if kind == "paged" or c.get("append"):
        res.update(k=[None] * 3, v=[None] * 3)
    return res
