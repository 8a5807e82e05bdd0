// GPU quantize/pack (decode-step append and whole-cache setup), split-P pack
// of given codes, and the unpack/dequant export used to prove bit-exactness.
//
// Reference behaviour being reproduced bit for bit:
//   quantize_groupwise  quantize.py:186-236   (fp32 min/max per group,
//       scale = range/qmax or 1 for a degenerate group, scale and zero rounded
//       to fp16 first, code = rint((x - zero)/scale) clamped to [0, qmax])
//   pack_codes          quantize.py:149-169
//   unpack_codes        quantize.py:172-183
//   dequantize_groupwise quantize.py:239-246 (fp32 code*scale + zero; the
//       product is exact since code <= 15 and scale has 11 significant bits,
//       so fmaf gives the same bits as the reference's mul-then-add)
//
// The arithmetic relies on IEEE binary32 division (hipcc's default correctly
// rounded fp32 divide -- this file must not be built with fast-math) and on
// rintf rounding half to even like torch.round.
#include <stdint.h>
#include <type_traits>

#include "tkv_codec.h"
#include "tkv_quant.h"
#include "../../include/tkv.h"

namespace tkv {

// Destination of appended rows in a paged cache (page_size > 0): logical token
// t of batch row b goes to pool page block_table[b * stride + t / page_size],
// slot t % page_size; pools are laid out (num_pages, HKV, page_size, ...).
struct PageMap {
  const int32_t* block_table;
  int stride, page_size, num_pages;
};

// Rows to quantize: value d of token t of (b, kv head) is element
// b * sb + kv * sh + t * st + d of x.
struct TokenSource {
  const void* x;
  int64_t sb, sh, st;
};

// One wave per cache row (token x kv head), quantized by quantize_row: lane j
// owns packed byte j of the row.  Used when the input or the codes are not
// aligned for the wide kernel below.
template <int D, int NB, int GS, bool F32>
__global__ void __launch_bounds__(256)
quantize_pack_kernel(const void* __restrict__ x, int64_t row0, int64_t rows, int HKV, int N,
                     const int32_t* __restrict__ positions, int S_cap, PageMap pm,
                     uint8_t* __restrict__ packed, uint16_t* __restrict__ scale,
                     uint16_t* __restrict__ zero) {
  using R = RowQuant<D, NB, GS>;
  constexpr int P = R::P, DP = R::DP, NG = R::NG;

  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int64_t rr = row0 + (int64_t)blockIdx.x * 4 + w;
  if (rr >= rows) return;  // whole wave
  float xv[P];
  load_row_for_quant<D, NB>(static_cast<const uint8_t*>(x) + rr * D * (F32 ? 4 : 2), F32, lane, xv);
  const int64_t bh = rr / N;
  const int t = (int)(rr - bh * N);
  const int b = (int)(bh / HKV), kv = (int)(bh - (int64_t)b * HKV);
  const int64_t dst_t = (int64_t)(positions ? positions[b] : 0) + t;
  bool in_range = dst_t >= 0 && dst_t < S_cap;
  int64_t dst_row = bh * S_cap + dst_t;
  if (pm.page_size > 0 && in_range) {  // S_cap == stride * page_size
    const int e = pm.block_table[(int64_t)b * pm.stride + dst_t / pm.page_size];
    in_range = e >= 0 && e < pm.num_pages;  // rows mapped outside the pool are not written
    dst_row = ((int64_t)e * HKV + kv) * pm.page_size + dst_t % pm.page_size;
  }
  const R q = quantize_row<D, NB, GS>(xv, lane);
  if (!in_range) return;
  if (lane < DP) packed[dst_row * DP + lane] = (uint8_t)q.byte;
  if (lane < NG) {
    scale[dst_row * NG + lane] = (uint16_t)(q.meta & 0xFFFFu);
    zero[dst_row * NG + lane] = (uint16_t)(q.meta >> 16);
  }
}

// The same quantization spread over lanes eight bytes at a time (the same
// arithmetic, so the same bits).  A lane (slot r = l / LPR, column c = l % LPR)
// owns the E = 8 packed bytes [8c, 8c + 8) of its row, i.e. the 8P codes of
// dims 8c + e + p*DP: P runs of 8 consecutive values (16-byte loads) in, one
// 8-byte store of codes out.
template <int D, int NB, int GS, bool F32>
struct WideRow {
  static constexpr int P = 8 / NB, DP = D / P, NG = D / GS, QMAX = (1 << NB) - 1, E = 8;
  static constexpr int LPR = DP / E, RPS = 64 / LPR;  // lanes per row, rows per wave and step
  static constexpr int NV = F32 ? 2 : 1;              // 16-byte loads per run of E values
  // Rows are read once, but where several of a wave's load instructions take
  // pieces of the same cache line, a non-temporal line is gone before the last of
  // them (524288 rows, plain -> non-temporal loads, us: D = 64 2-bit fp16 15.6 ->
  // 21.5, fp32 26.7 -> 40.6, 4-bit fp16 17.4 -> 18.6; D = 128 2-bit fp32 54.2 -> 54.7).
  // fp16 rows of 128 dims gain: 4-bit 31.8 -> 31.3, 2-bit 31.3 -> 30.3.
  static constexpr bool kNonTemporal = D == 128 && !F32;
  static_assert(DP % E == 0 && LPR >= 2 && LPR <= 16, "row shape");
  static_assert(GS > DP ? GS % DP == 0 : GS % E == 0, "group shape");

  // Whether this lane holds the first byte of a group of slice p, and which group.
  __device__ static bool first_byte(int c, int p) {
    if constexpr (GS <= DP) return (c * E) % GS == 0;
    else return c == 0 && p % (GS / DP) == 0;
  }
  __device__ static constexpr int group_of(int c, int p) { return (p * DP + c * E) / GS; }

  __device__ static void load(const void* x, int64_t off, int c, u4 (&raw)[P][NV]) {
#pragma unroll
    for (int p = 0; p < P; ++p)
#pragma unroll
      for (int k = 0; k < NV; ++k) {
        const int64_t e = off + p * DP + c * E;
        const u4* v = F32 ? reinterpret_cast<const u4*>(static_cast<const float*>(x) + e)
                          : reinterpret_cast<const u4*>(static_cast<const _Float16*>(x) + e);
        if constexpr (kNonTemporal) raw[p][k] = __builtin_nontemporal_load(v + k);
        else raw[p][k] = v[k];
      }
  }

  // Value e of a run.  fp32: whole-vector casts (this compiler folds a min/max
  // over floats cast one by one from an integer vector's elements to the first).
  __device__ static float value(const u4 (&raw)[NV], int e) {
    if constexpr (F32) return __builtin_bit_cast(f4, raw[e / 4])[e % 4];
    else return (float)__builtin_bit_cast(h8, raw[0])[e];
  }

  // The lane's 8 code bytes, and each slice's fp16 scale (low half) and zero.
  __device__ static void quantize(const u4 (&raw)[P][NV], u2& codes, uint32_t (&sz)[P]) {
    float mn[P], mx[P];
    if constexpr (F32) {
#pragma unroll
      for (int p = 0; p < P; ++p) {
        mn[p] = mx[p] = value(raw[p], 0);
#pragma unroll
        for (int e = 1; e < E; ++e) {
          mn[p] = nan_min(mn[p], value(raw[p], e));
          mx[p] = nan_max(mx[p], value(raw[p], e));
        }
      }
      if constexpr (GS <= DP) {
#pragma unroll
        for (int p = 0; p < P; ++p) minmax_lanes<GS / E>(mn[p], mx[p]);
      } else {
        constexpr int SPG = GS / DP;
#pragma unroll
        for (int p = 0; p < P; p += SPG) {
#pragma unroll
          for (int e = 1; e < SPG; ++e) {
            mn[p] = nan_min(mn[p], mn[p + e]);
            mx[p] = nan_max(mx[p], mx[p + e]);
          }
          minmax_lanes<LPR>(mn[p], mx[p]);
#pragma unroll
          for (int e = 1; e < SPG; ++e) mn[p + e] = mn[p], mx[p + e] = mx[p];
        }
      }
    } else {
      // fp16 values are their own min and max: packed v_pk_minimum3 / maximum3
      // fold the run, then (min, -max) travels as one fp16 pair.
      h2 mm[P];
#pragma unroll
      for (int p = 0; p < P; ++p) mm[p] = run_minmax(raw[p][0]);
      if constexpr (GS <= DP) {
#pragma unroll
        for (int p = 0; p < P; ++p) mm[p] = pair_min_lanes<GS / E>(mm[p]);
      } else {
        constexpr int SPG = GS / DP;
#pragma unroll
        for (int p = 0; p < P; p += SPG) {
#pragma unroll
          for (int e = 1; e < SPG; ++e) mm[p] = __builtin_elementwise_minimum(mm[p], mm[p + e]);
          mm[p] = pair_min_lanes<LPR>(mm[p]);
#pragma unroll
          for (int e = 1; e < SPG; ++e) mm[p + e] = mm[p];
        }
      }
#pragma unroll
      for (int p = 0; p < P; ++p) {
        mn[p] = (float)mm[p][0];
        mx[p] = -(float)mm[p][1];
      }
    }
    float sf[P], zf[P], special = 0.0f;
    uint32_t w[2] = {code_bias<P, NB>(), code_bias<P, NB>()};
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const GroupScale g = group_scale<QMAX>(mn[p], mx[p]);
      sz[p] = g.bits;
      sf[p] = g.s;
      zf[p] = g.z;
      const float rs = __builtin_amdgcn_rcpf(g.s);
      special += group_special(g.s, g.z, rs);
#pragma unroll
      for (int e = 0; e < E; ++e)
        w[e / 4] += code_term<QMAX>(value_less(raw[p], e, g.z), g.s, rs) << (8 * (e % 4) + p * NB);
    }
    if (__builtin_expect(special != 0.0f, 0)) {  // NaN: redo the lane's codes by division
      w[0] = w[1] = 0;
#pragma unroll
      for (int p = 0; p < P; ++p)
#pragma unroll
        for (int e = 0; e < E; ++e)
          w[e / 4] |= code_by_division<QMAX>(value(raw[p], e) - zf[p], sf[p]) << (8 * (e % 4) + p * NB);
    }
    codes = u2{w[0], w[1]};
  }

 private:
  // Value e of a run less z; fp16 as one v_fma_mix (the opaque 1.0 keeps the
  // conversion inside the multiply-add: one rounding, that of the difference).
  __device__ static float value_less(const u4 (&raw)[NV], int e, float z) {
    if constexpr (F32) return value(raw, e) - z;
    else return half_less(raw[0][e / 2], e & 1, z);
  }
};

// A few rows, and paged caches: each wave finds its rows' batch row, head and
// destination by division.  BULK takes several steps of rows, all their loads
// issued before any arithmetic.  Requires x 16-byte and packed 8-byte aligned,
// rows < 2^31.
template <int D, int NB, int GS, bool F32, bool BULK>
__global__ void __launch_bounds__(256)
quantize_pack_wide_kernel(const void* __restrict__ x, int rows, int HKV, int N,
                          const int32_t* __restrict__ positions, int S_cap, PageMap pm,
                          uint8_t* __restrict__ packed, uint16_t* __restrict__ scale,
                          uint16_t* __restrict__ zero) {
  using W = WideRow<D, NB, GS, F32>;
  constexpr int P = W::P, DP = W::DP, NG = W::NG, RPS = W::RPS;
  constexpr int STEPS = BULK && 8 / (P * W::NV) > 0 ? 8 / (P * W::NV) : 1;  // ~128 B per lane

  const int lane = threadIdx.x & 63, slot = lane / W::LPR, c = lane % W::LPR;
  const int first = ((int)blockIdx.x * 4 + (int)(threadIdx.x >> 6)) * STEPS * RPS;
  u4 raw[STEPS][P][W::NV];
#pragma unroll
  for (int s = 0; s < STEPS; ++s)
    W::load(x, (int64_t)min(first + s * RPS + slot, rows - 1) * D, c, raw[s]);
#pragma unroll
  for (int s = 0; s < STEPS; ++s) {
    const int rr = first + s * RPS + slot;
    u2 codes;
    uint32_t sz[P];
    W::quantize(raw[s], codes, sz);
    if (rr >= rows) continue;  // after the cross-lane steps, which need every lane
    const int bh = rr / N, t = rr - bh * N;
    const int b = bh / HKV, kv = bh - b * HKV;
    const int64_t dst_t = (int64_t)(positions ? positions[b] : 0) + t;
    bool in_range = dst_t >= 0 && dst_t < S_cap;
    int64_t dst_row = (int64_t)bh * S_cap + dst_t;
    if (pm.page_size > 0 && in_range) {  // S_cap == stride * page_size
      const int e = pm.block_table[(int64_t)b * pm.stride + dst_t / pm.page_size];
      in_range = e >= 0 && e < pm.num_pages;  // rows mapped outside the pool are not written
      dst_row = ((int64_t)e * HKV + kv) * pm.page_size + dst_t % pm.page_size;
    }
    if (!in_range) continue;
    *reinterpret_cast<u2*>(packed + dst_row * DP + c * W::E) = codes;
    // Group g's scale and zero are written by the lane holding its first byte.
#pragma unroll
    for (int p = 0; p < P; ++p)
      if (W::first_byte(c, p)) {
        scale[dst_row * NG + W::group_of(c, p)] = (uint16_t)sz[p];
        zero[dst_row * NG + W::group_of(c, p)] = (uint16_t)(sz[p] >> 16);
      }
  }
}

// A prompt's rows (many tokens per head) into a contiguous cache: HBM-bound
// with VALU close behind, so a workgroup's tokens all belong to one (b, kv
// head), whose addresses are scalar, and the metadata of a wave's rows meets
// in LDS and leaves as whole dwords (64 lanes store 256 consecutive bytes,
// where each group's first lane used to store its own 2 bytes).  524288 rows of
// D = 128 fp16, groups of 32: 4-bit 53 -> 31.5 us (5.6 TB/s), 2-bit 54 -> 30.4
// us (5.2 TB/s); the gain is VALU: 1.1k -> 0.8k instructions per 32 rows from
// the exact quotient that needs no fallback for ties, packed fp16 min/max and
// no integer divisions.
// Workgroup x takes tile x / HKV of head x % HKV when the source is
// token-major (tile % tiles of head x / tiles otherwise), so that workgroups
// running together read neighbouring memory; y is the batch row.
// Requires x 16-byte, its strides 16-byte multiples, packed 8-byte and
// scale / zero 4-byte aligned.
template <int D, int NB, int GS, int STEPS>
__global__ void __launch_bounds__(256)
quantize_tokens_kernel(TokenSource src, int HKV, int N, int tiles,
                       const int32_t* __restrict__ positions, int start, int S_cap,
                       uint8_t* __restrict__ packed, uint16_t* __restrict__ scale,
                       uint16_t* __restrict__ zero) {
  using W = WideRow<D, NB, GS, false>;
  constexpr int P = W::P, DP = W::DP, NG = W::NG, RPS = W::RPS, ROWS = STEPS * RPS;
  __shared__ __attribute__((aligned(16))) uint32_t meta_lds[4][ROWS * NG];

  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int slot = lane / W::LPR, c = lane % W::LPR;
  const bool heads_first = src.st != D;
  const int q = (int)blockIdx.x / (heads_first ? HKV : tiles);
  const int m = (int)blockIdx.x - q * (heads_first ? HKV : tiles);
  const int kv = heads_first ? m : q, tile = heads_first ? q : m, b = blockIdx.y;
  const int t0 = (tile * 4 + w) * ROWS;
  if (t0 >= N) return;  // whole wave
  const int64_t base = b * src.sb + kv * src.sh + t0 * src.st;
  u4 raw[STEPS][P][W::NV];
#pragma unroll
  for (int s = 0; s < STEPS; ++s)
    W::load(src.x, base + (int64_t)min(s * RPS + slot, N - 1 - t0) * src.st, c, raw[s]);

  // Token t0 + i of the wave goes to row dst0 + i of the (b, kv head) block; rows
  // i in [lo, hi) exist and fit the capacity.
  const int64_t dst0 = (int64_t)(positions ? positions[b] : start) + t0;
  const int64_t left = max((int64_t)S_cap - dst0, (int64_t)0);
  const int lo = (int)min(max(-dst0, (int64_t)0), (int64_t)ROWS);
  const int hi = (int)min((int64_t)min(ROWS, N - t0), left);
  const int64_t row0 = ((int64_t)b * HKV + kv) * S_cap + dst0;
  uint32_t* const meta = meta_lds[w];
#pragma unroll
  for (int s = 0; s < STEPS; ++s) {
    u2 codes;
    uint32_t sz[P];
    W::quantize(raw[s], codes, sz);
    const int i = s * RPS + slot;
    if (i >= lo && i < hi) *reinterpret_cast<u2*>(packed + (row0 + i) * DP + c * W::E) = codes;
#pragma unroll
    for (int p = 0; p < P; ++p)
      if (W::first_byte(c, p)) meta[i * NG + W::group_of(c, p)] = sz[p];
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  if constexpr (NG >= 2) {
#pragma unroll
    for (int k = lane; k < ROWS * NG / 2; k += 64) {  // dword k: groups 2k, 2k + 1 of the wave's rows
      const int i = 2 * k / NG;
      const u2 two = *reinterpret_cast<const u2*>(meta + 2 * k);
      if (i >= lo && i < hi) {
        reinterpret_cast<uint32_t*>(scale + row0 * NG)[k] = perm(two[1], two[0], 0x05040100u);
        reinterpret_cast<uint32_t*>(zero + row0 * NG)[k] = perm(two[1], two[0], 0x07060302u);
      }
    }
  } else {
#pragma unroll
    for (int i = lane; i < ROWS; i += 64)
      if (i >= lo && i < hi) {
        scale[row0 + i] = (uint16_t)meta[i];
        zero[row0 + i] = (uint16_t)(meta[i] >> 16);
      }
  }
}

// Per-channel (KIVI-style) keys.  A block of 32 tokens of one (b, kv head) is
// quantized by D / 2 lanes of a wave: every channel of the block is one group of
// 32 values (min/max, fp16 scale and zero, codes), the group-wise arithmetic
// of quantize_row applied along the token axis.  Lane j of the block owns
// channels 2j and 2j + 1, so a token's row is one contiguous load (256 bytes at
// D = 128 fp16), the min/max need no cross-lane step, and scale and zero leave
// as whole dwords.  A byte column's P channels sit in P lanes LS = DP / 2
// apart: each lane packs its codes of two tokens into a dword at its slice's
// bits, an OR-reduction over those lanes by lane swaps leaves every lane
// 16 / P of the dwords, and two exchanges with neighbouring lanes turn them into
// 8-byte pieces of packed rows.
// Bound by HBM: 4 x 8 heads of 8192 tokens, D = 128, fp16 to 2-bit, from a
// token-major source: 18.1 us (4.4 TB/s); byte columns per lane (2-byte loads,
// byte stores) took 35.9 us after a 36.4 us copy to contiguous keys.
template <int D, int NB, bool F32>
struct KeyBlock {
  static constexpr int P = 8 / NB, DP = D / P, QMAX = (1 << NB) - 1, T = 32;
  static constexpr int LB = D / 2;          // lanes of a block
  static constexpr int BPW = 64 / LB;       // blocks per wave
  static constexpr int LS = DP / 2;         // lanes of a slice
  static constexpr int NW = T / 2;          // dwords of codes per lane: two tokens each
  static constexpr int NR = NW / P;         // ... after the reduction over the slices

  // x: the first row of the block, rows st elements apart (wide: pairs of
  // channels may be read as one aligned load); packed: the block's first row;
  // scale / zero: its D values; ok: whether this lane's block is stored.
  __device__ static void quantize(const void* __restrict__ x, int64_t st, bool wide, int lane,
                                  bool ok, uint8_t* __restrict__ packed,
                                  uint16_t* __restrict__ scale, uint16_t* __restrict__ zero) {
    const int j = lane % LB;
    uint32_t raw[T][F32 ? 2 : 1];
    if (wide) {
#pragma unroll
      for (int t = 0; t < T; ++t) {
        if constexpr (F32) {
          const u2 v = __builtin_nontemporal_load(
              reinterpret_cast<const u2*>(static_cast<const float*>(x) + t * st + 2 * j));
          raw[t][0] = v[0];
          raw[t][1] = v[1];
        } else {
          raw[t][0] = __builtin_nontemporal_load(
              reinterpret_cast<const uint32_t*>(static_cast<const uint16_t*>(x) + t * st + 2 * j));
        }
      }
    } else {
#pragma unroll
      for (int t = 0; t < T; ++t) {
        if constexpr (F32) {
          const uint32_t* v = static_cast<const uint32_t*>(x) + t * st + 2 * j;
          raw[t][0] = v[0];
          raw[t][1] = v[1];
        } else {
          const uint16_t* v = static_cast<const uint16_t*>(x) + t * st + 2 * j;
          raw[t][0] = (uint32_t)v[0] | ((uint32_t)v[1] << 16);
        }
      }
    }
    float mn[2], mx[2];
    if constexpr (F32) {
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        mn[c] = mx[c] = as_float(raw[0][c]);
#pragma unroll
        for (int t = 1; t < T; ++t) {
          mn[c] = nan_min(mn[c], as_float(raw[t][c]));
          mx[c] = nan_max(mx[c], as_float(raw[t][c]));
        }
      }
    } else {
      h2 lo = __builtin_bit_cast(h2, raw[0][0]), hi = lo;
#pragma unroll
      for (int t = 1; t < T; ++t) {
        lo = __builtin_elementwise_minimum(lo, __builtin_bit_cast(h2, raw[t][0]));
        hi = __builtin_elementwise_maximum(hi, __builtin_bit_cast(h2, raw[t][0]));
      }
#pragma unroll
      for (int c = 0; c < 2; ++c) mn[c] = (float)lo[c], mx[c] = (float)hi[c];
    }
    uint32_t w[NW], bits[2];
    float sf[2], zf[2], special = 0.0f;
#pragma unroll
    for (int k = 0; k < NW; ++k) w[k] = code_bias<1, NB>();
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const GroupScale g = group_scale<QMAX>(mn[c], mx[c]);
      bits[c] = g.bits;
      sf[c] = g.s;
      zf[c] = g.z;
      const float rs = __builtin_amdgcn_rcpf(g.s);
      special += group_special(g.s, g.z, rs);
#pragma unroll
      for (int t = 0; t < T; ++t)
        w[t / 2] += code_term<QMAX>(less(raw[t], c, g.z), g.s, rs) << (16 * (t & 1) + 8 * c);
    }
    if (__builtin_expect(special != 0.0f, 0)) {  // NaN: redo the lane's codes by division
#pragma unroll
      for (int k = 0; k < NW; ++k) w[k] = 0;
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int t = 0; t < T; ++t)
          w[t / 2] |= code_by_division<QMAX>(less(raw[t], c, zf[c]), sf[c]) << (16 * (t & 1) + 8 * c);
    }
    // Dword k of lane j: tokens 2k, 2k + 1 (low, high half) at slice j / LS's bits.
    const int shift = (j / LS) * NB;
#pragma unroll
    for (int k = 0; k < NW; ++k) w[k] <<= shift;
    // OR over the lanes of a byte column; each step leaves a lane half of its
    // dwords, the upper half where the lane's bit is set.
    int k0 = 0;  // index of dword 0
    if constexpr (D == 128) {
      or_scatter<32, NW>(w, lane, k0);
      if constexpr (P == 4) or_scatter<16, NW / 2>(w, lane, k0);
    } else {
      or_scatter<16, NW>(w, lane, k0);
      if constexpr (P == 4) or_scatter<8, NW / 2>(w, lane, k0);
    }
    if (ok) {
      if (!(((uintptr_t)scale | (uintptr_t)zero) & 3)) {
        reinterpret_cast<uint32_t*>(scale)[j] = perm(bits[1], bits[0], 0x05040100u);
        reinterpret_cast<uint32_t*>(zero)[j] = perm(bits[1], bits[0], 0x07060302u);
      } else {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          scale[2 * j + c] = (uint16_t)bits[c];
          zero[2 * j + c] = (uint16_t)(bits[c] >> 16);
        }
      }
    }
    // Lanes j, j ^ 1 hold adjacent byte pairs of two tokens each: the even lane
    // takes the four bytes of token 2k, the odd one those of 2k + 1.
    const bool odd = lane & 1, upper = lane & 2;
    const uint32_t sel = odd ? 0x03020706u : 0x05040100u;
#pragma unroll
    for (int k = 0; k < NR; ++k) w[k] = perm(dpp<0xB1>(w[k]), w[k], sel);
    // Lanes j, j ^ 2 then hold adjacent dwords: the lower takes 8 bytes of even
    // dwords' tokens, the upper of odd ones'.
    const int col = 8 * ((j % LS) >> 2);
#pragma unroll
    for (int i = 0; i < NR / 2; ++i) {
      const uint32_t got = dpp<0x4E>(upper ? w[2 * i] : w[2 * i + 1]);
      const u2 v = upper ? u2{got, w[2 * i + 1]} : u2{w[2 * i], got};
      const int t = 2 * (k0 + 2 * i + (upper ? 1 : 0)) + (odd ? 1 : 0);
      if (!ok) continue;
      uint8_t* dst = packed + t * DP + col;
      if (!((uintptr_t)packed & 7)) {
        *reinterpret_cast<u2*>(dst) = v;
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) dst[e] = (uint8_t)(v[e / 4] >> (8 * (e % 4)));
      }
    }
  }

 private:
  __device__ static float as_float(uint32_t v) { return __builtin_bit_cast(float, v); }
  __device__ static float less(const uint32_t (&raw)[F32 ? 2 : 1], int c, float z) {
    if constexpr (F32) return as_float(raw[c]) - z;
    else return half_less(raw[0], c, z);
  }
  template <int CTRL>
  __device__ static uint32_t dpp(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, CTRL, 0xF, 0xF, true);
  }
  // w[0 .. N/2) = the OR over lanes l and l ^ X of w[k] (bit X of l clear) or
  // w[k + N/2] (set).
  template <int X, int N>
  __device__ static void or_scatter(uint32_t (&w)[NW], int lane, int& k0) {
    const bool set = lane & X;
#pragma unroll
    for (int k = 0; k < N / 2; ++k) {
      if constexpr (X == 8) {
        const uint32_t keep = set ? w[k + N / 2] : w[k], send = set ? w[k] : w[k + N / 2];
        w[k] = keep | dpp<0x128>(send);
      } else {
        // the swap leaves (own, partner's) halves of w[k] in the clear lanes
        // and of w[k + N/2] in the set ones
        const auto s = X == 32 ? __builtin_amdgcn_permlane32_swap(w[k], w[k + N / 2], false, false)
                               : __builtin_amdgcn_permlane16_swap(w[k], w[k + N / 2], false, false);
        w[k] = opaque(s[0]) | opaque(s[1]);
      }
    }
    if (set) k0 += N / 2;
  }
};

// Workgroup wg's four waves of the key blocks of batch row b.  A block whose
// destination does not start on a 32-token boundary, or does not fit
// [0, S_cap), is not written.  Blocks are dealt to waves heads first for a
// token-major source (neighbouring waves then read neighbouring memory), tokens
// first otherwise.
template <int D, int NB, bool F32>
__device__ __forceinline__ void quantize_key_blocks(const TokenSource& src, bool wide, int wg, int b,
                                                    int HKV, int NBLK, int64_t start, int S_cap,
                                                    uint8_t* __restrict__ packed,
                                                    uint16_t* __restrict__ scale,
                                                    uint16_t* __restrict__ zero) {
  using K = KeyBlock<D, NB, F32>;
  constexpr int T = K::T;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int first = (wg * 4 + w) * K::BPW, blocks = HKV * NBLK;
  if (first >= blocks) return;  // whole wave
  const int i = first + (K::BPW > 1 ? lane / K::LB : 0);
  const int ii = min(i, blocks - 1);
  const bool heads_first = src.st != D;
  const int q = ii / (heads_first ? HKV : NBLK), m = ii - q * (heads_first ? HKV : NBLK);
  const int kv = heads_first ? m : q, tb = heads_first ? q : m;
  const int64_t off = b * src.sb + kv * src.sh + (int64_t)tb * T * src.st;
  const int64_t dst_t = start + (int64_t)tb * T;
  const bool ok = i < blocks && dst_t >= 0 && dst_t % T == 0 && dst_t + T <= S_cap;
  const int64_t bh = (int64_t)b * HKV + kv;
  const int64_t meta = ok ? (bh * (S_cap / T) + dst_t / T) * D : 0;
  K::quantize(F32 ? (const void*)(static_cast<const float*>(src.x) + off)
                  : (const void*)(static_cast<const uint16_t*>(src.x) + off),
              src.st, wide, lane, ok, packed + (ok ? (bh * S_cap + dst_t) * K::DP : 0), scale + meta,
              zero + meta);
}

template <int D, int NB, bool F32>
__global__ void __launch_bounds__(256)
quantize_keys_channel_kernel(TokenSource src, bool wide, int B, int HKV, int NBLK,
                             const int32_t* __restrict__ positions, int S_cap,
                             uint8_t* __restrict__ packed, uint16_t* __restrict__ scale,
                             uint16_t* __restrict__ zero) {
  for (int b = blockIdx.y; b < B; b += gridDim.y)
    quantize_key_blocks<D, NB, F32>(src, wide, blockIdx.x, b, HKV, NBLK, positions ? positions[b] : 0,
                                    S_cap, packed, scale, zero);
}

// A prompt's keys and what lies past its last whole block, in one launch:
// workgroups x < key_wgs quantize key blocks to token `start` on; workgroup
// key_wgs + kv copies the last `rest` tokens of kv head kv into rows
// [0, rest) of the windows (their own launch took 3-5 us behind the values'),
// and the first of them sets the batch row's lengths.
template <int D, int NB>
__global__ void __launch_bounds__(256)
channel_extend_kernel(TokenSource ks, TokenSource vs, int key_wgs, int HKV, int NBLK, int start,
                      int S_cap, uint8_t* __restrict__ packed, uint16_t* __restrict__ scale,
                      uint16_t* __restrict__ zero, int rest, uint16_t* __restrict__ k_res,
                      uint16_t* __restrict__ v_res, int32_t* __restrict__ q_lens,
                      int32_t* __restrict__ res_lens) {
  constexpr int T = 32;
  const int b = blockIdx.y;
  if ((int)blockIdx.x < key_wgs) {
    quantize_key_blocks<D, NB, false>(ks, true, blockIdx.x, b, HKV, NBLK, start, S_cap, packed, scale, zero);
    return;
  }
  const int kv = blockIdx.x - key_wgs, n = rest * D / 8;  // 16-byte vectors per tensor
  for (int i = threadIdx.x; i < 2 * n; i += blockDim.x) {
    const TokenSource& s = i < n ? ks : vs;
    const int e = (i < n ? i : i - n) * 8, t = e / D, d = e % D;
    const uint16_t* from =
        static_cast<const uint16_t*>(s.x) + b * s.sb + kv * s.sh + (int64_t)(NBLK * T + t) * s.st + d;
    uint16_t* to = (i < n ? k_res : v_res) + (((int64_t)b * HKV + kv) * T + t) * D + d;
    *reinterpret_cast<u4*>(to) = *reinterpret_cast<const u4*>(from);
  }
  if (kv == 0 && threadIdx.x == 0) {
    q_lens[b] = start + NBLK * T;
    res_lens[b] = rest;
  }
}

// The fp16 window of per-channel keys: K and V windows (B, HKV, 32, D), row b
// holding res_lens[b] tokens after q_lens[b] quantized ones.
//
// Append: one workgroup per batch row writes the new token of every kv head
// at window row res_lens[b] (if it is below 32) and then advances res_lens[b].
__global__ void __launch_bounds__(256)
channel_window_append_kernel(const uint16_t* __restrict__ k_new, const uint16_t* __restrict__ v_new,
                             int HKV, int D, uint16_t* __restrict__ k_res,
                             uint16_t* __restrict__ v_res, int32_t* __restrict__ res_lens) {
  constexpr int T = 32;
  const int b = blockIdx.x;
  const int r = res_lens[b];
  if (r < 0 || r >= T) return;  // whole workgroup: a full window must be flushed first
  const int n = HKV * D / 8;    // 16-byte vectors per token and tensor
  for (int i = threadIdx.x; i < 2 * n; i += blockDim.x) {
    const int which = i / n, e = (i % n) * 8, kv = e / D, d = e % D;
    const uint16_t* src = (which ? v_new : k_new) + (int64_t)b * HKV * D + e;
    uint16_t* dst = (which ? v_res : k_res) + (((int64_t)b * HKV + kv) * T + r) * D + d;
    *reinterpret_cast<u4*>(dst) = *reinterpret_cast<const u4*>(src);
  }
  __syncthreads();
  if (threadIdx.x == 0) res_lens[b] = r + 1;
}

// Flush: one workgroup per batch row; if its window holds 32 tokens, wave w
// quantizes the blocks of kv heads w, w + 4, ...: keys per channel (KeyBlock;
// lanes past the block's repeat it), values per token (quantize_row, as the append kernel)
// into the history at q_lens[b]; then q_lens[b] += 32 and res_lens[b] = 0.
// A window that does not fit the history ([q, q + 32) outside [0, S_cap)) is
// not written and the lengths do not move: res_lens[b] becomes 33, the
// overflow mark, which the append kernel treats as full (nothing more is
// appended) and the decode clamps to the 32 tokens the window holds.
template <int D, int KNB, int VNB, int GS>
__global__ void __launch_bounds__(256)
channel_window_flush_kernel(const uint16_t* __restrict__ k_res, const uint16_t* __restrict__ v_res,
                            int HKV, int S_cap, int32_t* __restrict__ q_lens,
                            int32_t* __restrict__ res_lens, uint8_t* __restrict__ kp,
                            uint16_t* __restrict__ ks, uint16_t* __restrict__ kz,
                            uint8_t* __restrict__ vp, uint16_t* __restrict__ vs,
                            uint16_t* __restrict__ vz) {
  using R = RowQuant<D, VNB, GS>;
  constexpr int T = 32, VDP = R::DP, VNG = R::NG;
  const int b = blockIdx.x;
  if (res_lens[b] != T) return;  // whole workgroup
  const int q = q_lens[b];
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (!(q >= 0 && q % T == 0 && q + T <= S_cap)) {  // uniform over the workgroup
    if (threadIdx.x == 0) res_lens[b] = T + 1;
    return;
  }
  using K = KeyBlock<D, KNB, false>;
  const bool wide = !((uintptr_t)k_res & 3);
  for (int kv = w; kv < HKV; kv += 4) {
    const int64_t bh = (int64_t)b * HKV + kv, meta = (bh * (S_cap / T) + q / T) * D;
    K::quantize(k_res + bh * T * D, D, wide, lane, lane < K::LB, kp + (bh * S_cap + q) * K::DP,
                ks + meta, kz + meta);
    for (int t = 0; t < T; ++t) {
      float x[R::P];
      load_row_for_quant<D, VNB>(v_res + (bh * T + t) * D, false, lane, x);
      const R r = quantize_row<D, VNB, GS>(x, lane);
      const int64_t row = bh * S_cap + q + t;
      if (lane < VDP) vp[row * VDP + lane] = (uint8_t)r.byte;
      if (lane < VNG) {
        vs[row * VNG + lane] = (uint16_t)(r.meta & 0xFFFFu);
        vz[row * VNG + lane] = (uint16_t)(r.meta >> 16);
      }
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    q_lens[b] = q + T;
    res_lens[b] = 0;
  }
}

// One thread per packed dword (grid-stride: the grid is capped at 2^20 workgroups).
__global__ void __launch_bounds__(256)
pack_codes_kernel(const uint8_t* __restrict__ codes, int64_t rows, int D, int NB,
                  uint8_t* __restrict__ packed) {
  const int P = 8 / NB, DP = D / P, DW = DP / 4;
  const int64_t n = rows * DW, step = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += step) {
    const int64_t row = i / DW;
    const int q = (int)(i % DW);
    const uint8_t* c = codes + row * D;
    uint32_t word = 0;
    for (int k = 0; k < 4; ++k) {
      const int jb = 4 * q + k;
      uint32_t byte = 0;
      for (int p = 0; p < P; ++p) byte |= (uint32_t)(c[jb + p * DP] & ((1 << NB) - 1)) << (p * NB);
      word |= byte << (8 * k);
    }
    reinterpret_cast<uint32_t*>(packed + row * DP)[q] = word;
  }
}

__device__ __forceinline__ void emit(uint8_t* codes_out, float* values_out,
                                     const uint16_t* scale, const uint16_t* zero, int64_t row,
                                     int D, int GS, int d, uint32_t code) {
  if (codes_out) codes_out[row * D + d] = (uint8_t)code;
  if (values_out) {
    const int NG = D / GS;
    const float s = (float)__builtin_bit_cast(_Float16, scale[row * NG + d / GS]);
    const float z = (float)__builtin_bit_cast(_Float16, zero[row * NG + d / GS]);
    values_out[row * D + d] = fmaf((float)code, s, z);
  }
}

// Path 0: the K-operand extraction of the decode kernel.  One wave per 16 rows;
// lane (r = l%16, j = l/16) plays the MFMA A-operand role for row r.
template <int D, int NB, int GS>
__global__ void __launch_bounds__(64)
unpack_k_kernel(const uint8_t* __restrict__ packed, const uint16_t* __restrict__ scale,
                const uint16_t* __restrict__ zero, int64_t rows, uint8_t* codes_out,
                float* values_out) {
  using KL = KLayout<D, NB, GS>;
  const int lane = threadIdx.x, r = lane & 15, j = lane >> 4;
  const int64_t row = (int64_t)blockIdx.x * 16 + r;
  const int64_t lr = row < rows ? row : rows - 1;
  typename std::conditional<KL::CB == 8, u2, uint32_t>::type kx[KL::NLOAD];
#pragma unroll
  for (int Lh = 0; Lh < KL::NLOAD; ++Lh) {
    const uint8_t* src = packed + lr * KL::DP + KL::load_offset(Lh, j);
    if constexpr (KL::CB == 8) kx[Lh] = ld_u2(src);
    else kx[Lh] = ld_u32(src);
  }
  if (row >= rows) return;
#pragma unroll
  for (int m = 0; m < KL::NKM; ++m) {
    const int p = KL::slice_of(m, j);
    const uint32_t mask = slice_mask<NB>(p);
    uint32_t wv[4] = {0, 0, 0, 0};
    if constexpr (KL::CB == 8) {
      const u4 a = k_extract8(kx[KL::load_of_step(m)], mask);
      wv[0] = a[0]; wv[1] = a[1]; wv[2] = a[2]; wv[3] = a[3];
    } else {
      const u2 a = k_extract4(kx[KL::load_of_step(m)], mask);
      wv[0] = a[0]; wv[1] = a[1];
    }
#pragma unroll
    for (int s = 0; s < KL::CB; ++s) {
      const uint32_t half = (s & 1) ? (wv[s / 2] >> 16) : wv[s / 2];
      emit(codes_out, values_out, scale, zero, row, D, GS, KL::dim_of(m, j, s),
           code_of_half(half, p * NB));
    }
  }
}

// Path 1: the transposed V-operand extraction.  One wave per 32 tokens; lane
// (r, j) gathers tokens slot_token(j, 0..7) for A-operand row r.
template <int D, int NB, int GS>
__global__ void __launch_bounds__(64)
unpack_v_kernel(const uint8_t* __restrict__ packed, const uint16_t* __restrict__ scale,
                const uint16_t* __restrict__ zero, int64_t rows, uint8_t* codes_out,
                float* values_out) {
  using VL = VLayout<D, NB, GS>;
  const int lane = threadIdx.x, r = lane & 15, j = lane >> 4;
  const int64_t base = (int64_t)blockIdx.x * 32;
  uint32_t vx[8][VL::NWIN];
  int64_t tok[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    tok[i] = base + (i < 4 ? 0 : 12) + 4 * j + i;
    const int64_t lr = tok[i] < rows ? tok[i] : rows - 1;
#pragma unroll
    for (int wi = 0; wi < VL::NWIN; ++wi)
      vx[i][wi] = ld_u32(packed + lr * VL::DP + VL::dword_offset(wi, r));
  }
#pragma unroll
  for (int wi = 0; wi < VL::NWIN; ++wi) {
#pragma unroll
    for (int e = 0; e < VL::NE; ++e) {
      const uint32_t sel = VL::perm_sel(VL::byte_in_dword(e, r));
#pragma unroll
      for (int p = 0; p < VL::P; ++p) {
        const int mv = VL::mfma_index(p, wi, e);
        const int d = VL::dim_of(mv, r);
        const uint32_t mask = slice_mask<NB>(p);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const uint32_t pr = v_extract(vx[2 * i + 1][wi], vx[2 * i][wi], sel, mask);
          if (tok[2 * i] < rows)
            emit(codes_out, values_out, scale, zero, tok[2 * i], D, GS, d,
                 code_of_half(pr, p * NB));
          if (tok[2 * i + 1] < rows)
            emit(codes_out, values_out, scale, zero, tok[2 * i + 1], D, GS, d,
                 code_of_half(pr >> 16, p * NB));
        }
      }
    }
  }
}

// Rows from which a wave takes several steps of rows: fewer rows run one step
// per wave, at most eight waves for each of the chip's 1024 SIMDs.
constexpr int64_t kBulkRows = 65536;

// Steps of rows per wave: ~128 bytes of input per lane when there are many.
template <int NB>
static constexpr int quantize_steps(bool f32, bool bulk) {
  const int per = (8 / NB) * (f32 ? 2 : 1);  // 16-byte loads per lane and step
  return bulk && 8 / per > 0 ? 8 / per : 1;
}

// fp16 tokens a workgroup of quantize_tokens_kernel takes.
template <int D, int NB, int GS>
static constexpr int tokens_per_wg(bool bulk) {
  return 4 * WideRow<D, NB, GS, false>::RPS * quantize_steps<NB>(false, bulk);
}

// Whether N tokens a head fill such workgroups well enough.  All tokens of one
// belong to one head, so a head's last workgroup is partly empty, where
// quantize_pack_wide_kernel runs the rows of all heads together (8192 heads, 128
// tokens a workgroup, 4-bit, us, all heads together -> by head: N = 33 21.7 -> 29.5,
// 64 34.8 -> 32.5, 80 41.4 -> 41.5, 96 48.6 -> 44.8, 100 50.4 -> 51.5, 128 63.4 -> 57.2,
// 129 64.0 -> 88.9, 200 97.3 -> 99.2, 257 127.9 -> 139.6, 300 149 -> 159): seven eighths
// full, or one workgroup a head at least half full of whole waves.  4-bit rows of
// 128 dims whose input the last-level cache holds (256 MB; a quarter of it where a
// head has one workgroup) gain earlier (2048 heads: N = 65 13.8 -> 12.4, 80 14.6 -> 13.2,
// 100 18.0 -> 16.0, 129 21.4 -> 27.0, 160 24.7 -> 27.7, 200 29.3 -> 28.8, 257 34.9 -> 34.1, 300
// 39.5 -> 37.2; 256 heads, 257 9.0 -> 7.9; 8192 heads, 65 35.2 -> 40.0), 2-bit ones do
// not (100 15.2 -> 16.0, 300 36.6 -> 37.8).
template <int D, int NB, int GS>
static bool tokens_fill_wgs(int64_t rows, int N, bool bulk) {
  const int per_wg = tokens_per_wg<D, NB, GS>(bulk);
  constexpr bool early = D == 128 && NB == 4;
  if (N < per_wg) return 2 * N >= per_wg && ((early && rows <= 1 << 18) || N % (per_wg / 4) == 0);
  const int64_t room = ((int64_t)N + per_wg - 1) / per_wg * per_wg;
  return early && rows <= 1 << 20 ? 3 * (int64_t)N >= 2 * room : 8 * (int64_t)N >= 7 * room;
}

// quantize_tokens_kernel for what it takes; false (nothing launched) otherwise.
template <int D, int NB, int GS>
static bool launch_tokens(const TokenSource& src, bool bulk, int B, int HKV, int N,
                          const int32_t* pos, int start, int S_cap, uint8_t* pk, uint16_t* sc,
                          uint16_t* zr, hipStream_t st) {
  const uintptr_t align = (uintptr_t)src.x | (uintptr_t)(src.sb * 2) | (uintptr_t)(src.sh * 2) |
                          (uintptr_t)(src.st * 2);
  if ((align & 15) || ((uintptr_t)pk & 7) || (((uintptr_t)sc | (uintptr_t)zr) & 3)) return false;
  const int per_wg = tokens_per_wg<D, NB, GS>(bulk);
  const int64_t tiles = ((int64_t)N + per_wg - 1) / per_wg;
  if (B > 65535 || tiles * HKV > INT32_MAX / 256) return false;
  const dim3 grid((unsigned)(tiles * HKV), (unsigned)B);
  if (bulk)
    quantize_tokens_kernel<D, NB, GS, quantize_steps<NB>(false, true)><<<grid, 256, 0, st>>>(
        src, HKV, N, (int)tiles, pos, start, S_cap, pk, sc, zr);
  else
    quantize_tokens_kernel<D, NB, GS, quantize_steps<NB>(false, false)><<<grid, 256, 0, st>>>(
        src, HKV, N, (int)tiles, pos, start, S_cap, pk, sc, zr);
  return true;
}

template <int D, int NB, int GS>
static void launch_quantize(const TokenSource& src, bool f32, int B, int HKV, int N,
                            const int32_t* pos, int S_cap, PageMap pm, uint8_t* pk, uint16_t* sc,
                            uint16_t* zr, hipStream_t st) {
  // fp32 rows gain nothing from it (524288 rows of 128, 4-bit 56.1 -> 56.2 us, 2-bit 53.5 -> 54.2)
  const int64_t rows = (int64_t)B * HKV * N;
  const bool bulk = rows >= kBulkRows;
  if (!f32 && pm.page_size == 0 && tokens_fill_wgs<D, NB, GS>(rows, N, bulk) &&
      launch_tokens<D, NB, GS>(src, bulk, B, HKV, N, pos, 0, S_cap, pk, sc, zr, st))
    return;
  const bool wide = !((uintptr_t)src.x & 15) && !((uintptr_t)pk & 7);
  if (wide && rows <= INT32_MAX) {
    const int per_wg = 4 * WideRow<D, NB, GS, false>::RPS * quantize_steps<NB>(f32, bulk);
    const dim3 grid((unsigned)((rows + per_wg - 1) / per_wg));
    const int r = (int)rows;
#define TKV_WIDE(F, BK) \
  quantize_pack_wide_kernel<D, NB, GS, F, BK><<<grid, 256, 0, st>>>(src.x, r, HKV, N, pos, S_cap, pm, pk, sc, zr)
    if (f32) {
      if (bulk) TKV_WIDE(true, true); else TKV_WIDE(true, false);
    } else {
      if (bulk) TKV_WIDE(false, true); else TKV_WIDE(false, false);
    }
#undef TKV_WIDE
  } else {
    // One wave per row, four per workgroup; launched in pieces so that no grid
    // exceeds 2^32 work-items.
    constexpr int64_t kMaxBlocks = (1 << 24) - 1;
    for (int64_t row0 = 0; row0 < rows; row0 += 4 * kMaxBlocks) {
      const int64_t n = rows - row0 < 4 * kMaxBlocks ? rows - row0 : 4 * kMaxBlocks;
      const dim3 grid((unsigned)((n + 3) / 4));
      if (f32)
        quantize_pack_kernel<D, NB, GS, true><<<grid, 256, 0, st>>>(src.x, row0, rows, HKV, N, pos, S_cap, pm, pk, sc, zr);
      else
        quantize_pack_kernel<D, NB, GS, false><<<grid, 256, 0, st>>>(src.x, row0, rows, HKV, N, pos, S_cap, pm, pk, sc, zr);
    }
  }
}

// Workgroups of four waves for the nblk key blocks of HKV heads.
template <int D>
static unsigned key_workgroups(int HKV, int nblk) {
  constexpr int per_wg = 4 * KeyBlock<D, 4, false>::BPW;
  return (unsigned)(((int64_t)HKV * nblk + per_wg - 1) / per_wg);
}

template <int D, int NB>
static void launch_key_blocks(const void* x, bool f32, int B, int HKV, int nblk, const int32_t* pos,
                              int S_cap, uint8_t* pk, uint16_t* sc, uint16_t* zr, hipStream_t st) {
  const TokenSource src{x, (int64_t)HKV * nblk * 32 * D, (int64_t)nblk * 32 * D, D};
  const bool wide = !((uintptr_t)x & (f32 ? 7 : 3));  // a lane's two channels in one load
  const dim3 grid(key_workgroups<D>(HKV, nblk), (unsigned)(B < 65535 ? B : 65535));
  if (f32)
    quantize_keys_channel_kernel<D, NB, true><<<grid, 256, 0, st>>>(src, wide, B, HKV, nblk, pos, S_cap, pk, sc, zr);
  else
    quantize_keys_channel_kernel<D, NB, false><<<grid, 256, 0, st>>>(src, wide, B, HKV, nblk, pos, S_cap, pk, sc, zr);
}

template <int D, int NB>
static void launch_channel_extend(const TokenSource& ks, const TokenSource& vs, int B, int HKV, int N,
                                  int start, int S_cap, uint8_t* pk, uint16_t* sc, uint16_t* zr,
                                  uint16_t* kr, uint16_t* vr, int32_t* ql, int32_t* rl, hipStream_t st) {
  const int nblk = N / 32;
  const unsigned wgs = key_workgroups<D>(HKV, nblk);
  channel_extend_kernel<D, NB><<<dim3(wgs + HKV, (unsigned)B), 256, 0, st>>>(
      ks, vs, (int)wgs, HKV, nblk, start, S_cap, pk, sc, zr, N % 32, kr, vr, ql, rl);
}

template <int D, int NB, int GS>
static void launch_unpack(const uint8_t* pk, const uint16_t* sc, const uint16_t* zr, int64_t rows,
                          int path, uint8_t* co, float* vo, hipStream_t st) {
  if (path == 0)
    unpack_k_kernel<D, NB, GS><<<dim3((unsigned)((rows + 15) / 16)), 64, 0, st>>>(pk, sc, zr, rows, co, vo);
  else
    unpack_v_kernel<D, NB, GS><<<dim3((unsigned)((rows + 31) / 32)), 64, 0, st>>>(pk, sc, zr, rows, co, vo);
}

// Calls F<D, NB, GS>::run(args...) for the compiled (D, nbits, group size) set.
#define TKV_DISPATCH_DNG(D_, NB_, GS_, CALL)                                          \
  do {                                                                               \
    if ((D_) == 128) {                                                               \
      if ((NB_) == 4) {                                                              \
        if ((GS_) == 16) { CALL(128, 4, 16); }                                       \
        else if ((GS_) == 32) { CALL(128, 4, 32); }                                  \
        else if ((GS_) == 64) { CALL(128, 4, 64); }                                  \
        else if ((GS_) == 128) { CALL(128, 4, 128); }                                \
        else return TKV_EUNSUPPORTED;                                                \
      } else {                                                                       \
        if ((GS_) == 16) { CALL(128, 2, 16); }                                       \
        else if ((GS_) == 32) { CALL(128, 2, 32); }                                  \
        else if ((GS_) == 64) { CALL(128, 2, 64); }                                  \
        else if ((GS_) == 128) { CALL(128, 2, 128); }                                \
        else return TKV_EUNSUPPORTED;                                                \
      }                                                                              \
    } else if ((D_) == 64) {                                                         \
      if ((NB_) == 4) {                                                              \
        if ((GS_) == 16) { CALL(64, 4, 16); }                                        \
        else if ((GS_) == 32) { CALL(64, 4, 32); }                                   \
        else if ((GS_) == 64) { CALL(64, 4, 64); }                                   \
        else return TKV_EUNSUPPORTED;                                                \
      } else {                                                                       \
        if ((GS_) == 16) { CALL(64, 2, 16); }                                        \
        else if ((GS_) == 32) { CALL(64, 2, 32); }                                   \
        else if ((GS_) == 64) { CALL(64, 2, 64); }                                   \
        else return TKV_EUNSUPPORTED;                                                \
      }                                                                              \
    } else {                                                                         \
      return TKV_EUNSUPPORTED;                                                       \
    }                                                                                \
  } while (0)

}  // namespace tkv

extern "C" int tkv_quantize_pack(const void* x, int32_t x_is_fp32, int32_t B, int32_t HKV,
                                 int32_t N, int32_t D, int32_t nbits, int32_t group_size,
                                 const int32_t* positions, int32_t S_cap, uint8_t* packed,
                                 uint16_t* scale, uint16_t* zero, tkv_stream_t stream) {
  using namespace tkv;
  if (!x || !packed || !scale || !zero) return TKV_EINVAL;
  if (B <= 0 || HKV <= 0 || N <= 0 || D <= 0 || S_cap <= 0) return TKV_EINVAL;
  if (nbits != 2 && nbits != 4) return TKV_EINVAL;
  if (group_size <= 0 || D % group_size) return TKV_EINVAL;
  if (!positions && N > S_cap) return TKV_EINVAL;
  if (((uintptr_t)packed & 3) || ((uintptr_t)scale & 1) || ((uintptr_t)zero & 1)) return TKV_EINVAL;
  if ((uintptr_t)x & (x_is_fp32 ? 3 : 1)) return TKV_EINVAL;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const PageMap pm{nullptr, 0, 0, 0};
  const TokenSource src{x, (int64_t)HKV * N * D, (int64_t)N * D, D};
  (void)hipGetLastError();
#define TKV_Q(Dv, NBv, GSv) \
  launch_quantize<Dv, NBv, GSv>(src, x_is_fp32 != 0, B, HKV, N, positions, S_cap, pm, packed, scale, zero, st)
  TKV_DISPATCH_DNG(D, nbits, group_size, TKV_Q);
#undef TKV_Q
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? TKV_OK : (int)e;
}

extern "C" int tkv_paged_quantize_pack(const void* x, int32_t x_is_fp32, int32_t B, int32_t HKV,
                                       int32_t N, int32_t D, int32_t nbits, int32_t group_size,
                                       const int32_t* positions, const int32_t* block_table,
                                       int32_t block_table_stride, int32_t page_size,
                                       int32_t num_pages, uint8_t* packed, uint16_t* scale,
                                       uint16_t* zero, tkv_stream_t stream) {
  using namespace tkv;
  if (!x || !packed || !scale || !zero || !positions || !block_table) return TKV_EINVAL;
  if (B <= 0 || HKV <= 0 || N <= 0 || D <= 0) return TKV_EINVAL;
  if (block_table_stride <= 0 || page_size <= 0 || page_size % 32 || num_pages <= 0)
    return TKV_EINVAL;
  if ((int64_t)block_table_stride * page_size > INT32_MAX) return TKV_EINVAL;
  if (nbits != 2 && nbits != 4) return TKV_EINVAL;
  if (group_size <= 0 || D % group_size) return TKV_EINVAL;
  if (((uintptr_t)packed & 3) || ((uintptr_t)scale & 1) || ((uintptr_t)zero & 1)) return TKV_EINVAL;
  if ((uintptr_t)x & (x_is_fp32 ? 3 : 1)) return TKV_EINVAL;
  const int S_cap = block_table_stride * page_size;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const TokenSource src{x, (int64_t)HKV * N * D, (int64_t)N * D, D};
  const PageMap pm{block_table, block_table_stride, page_size, num_pages};
  (void)hipGetLastError();
#define TKV_Q(Dv, NBv, GSv) \
  launch_quantize<Dv, NBv, GSv>(src, x_is_fp32 != 0, B, HKV, N, positions, S_cap, pm, packed, scale, zero, st)
  TKV_DISPATCH_DNG(D, nbits, group_size, TKV_Q);
#undef TKV_Q
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? TKV_OK : (int)e;
}

extern "C" int tkv_quantize_keys_channel(const void* x, int32_t x_is_fp32, int32_t B, int32_t HKV,
                                         int32_t N, int32_t D, int32_t nbits,
                                         const int32_t* positions, int32_t S_cap, uint8_t* packed,
                                         uint16_t* scale, uint16_t* zero, tkv_stream_t stream) {
  using namespace tkv;
  constexpr int T = 32;
  if (!x || !packed || !scale || !zero) return TKV_EINVAL;
  if (B <= 0 || HKV <= 0 || N <= 0 || D <= 0 || S_cap <= 0) return TKV_EINVAL;
  if (N % T || S_cap % T) return TKV_EINVAL;
  if (!positions && N > S_cap) return TKV_EINVAL;
  if (nbits != 2 && nbits != 4) return TKV_EINVAL;
  if (((uintptr_t)scale & 1) || ((uintptr_t)zero & 1)) return TKV_EINVAL;
  if ((uintptr_t)x & (x_is_fp32 ? 3 : 1)) return TKV_EINVAL;
  if ((int64_t)HKV * (N / T) > INT32_MAX) return TKV_EINVAL;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  (void)hipGetLastError();
#define TKV_KC(Dv, NBv) \
  launch_key_blocks<Dv, NBv>(x, x_is_fp32 != 0, B, HKV, N / T, positions, S_cap, packed, scale, zero, st)
  if (D == 128) {
    if (nbits == 4) TKV_KC(128, 4); else TKV_KC(128, 2);
  } else if (D == 64) {
    if (nbits == 4) TKV_KC(64, 4); else TKV_KC(64, 2);
  } else {
    return TKV_EUNSUPPORTED;
  }
#undef TKV_KC
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? TKV_OK : (int)e;
}

extern "C" int tkv_channel_extend(const void* k, const int64_t* k_strides, const void* v,
                                  const int64_t* v_strides, int32_t B, int32_t HKV, int32_t N,
                                  int32_t D, int32_t k_nbits, int32_t v_nbits, int32_t group_size,
                                  int32_t start, void* k_res, void* v_res, int32_t res_cap,
                                  int32_t* q_lens, int32_t* res_lens, int32_t S_cap,
                                  uint8_t* k_packed, uint16_t* k_scale, uint16_t* k_zero,
                                  uint8_t* v_packed, uint16_t* v_scale, uint16_t* v_zero,
                                  tkv_stream_t stream) {
  using namespace tkv;
  constexpr int T = 32;
  if (!k || !v || !k_strides || !v_strides || !k_res || !v_res || !q_lens || !res_lens || !k_packed ||
      !k_scale || !k_zero || !v_packed || !v_scale || !v_zero)
    return TKV_EINVAL;
  if (B <= 0 || HKV <= 0 || N <= 0 || S_cap <= 0 || S_cap % T || res_cap != T) return TKV_EINVAL;
  if (start < 0 || start % T || (int64_t)start + N > S_cap) return TKV_EINVAL;
  if ((k_nbits != 2 && k_nbits != 4) || (v_nbits != 2 && v_nbits != 4)) return TKV_EINVAL;
  if (D != 64 && D != 128) return TKV_EUNSUPPORTED;
  if (group_size != 16 && group_size != 32 && group_size != 64 && group_size != D) return TKV_EUNSUPPORTED;
  const TokenSource ks{k, k_strides[0], k_strides[1], k_strides[2]};
  const TokenSource vs{v, v_strides[0], v_strides[1], v_strides[2]};
  uintptr_t align = (uintptr_t)k | (uintptr_t)v | (uintptr_t)k_res | (uintptr_t)v_res;
  for (int i = 0; i < 3; ++i) align |= (uintptr_t)(2 * k_strides[i]) | (uintptr_t)(2 * v_strides[i]);
  if ((align & 15) || (((uintptr_t)k_packed | (uintptr_t)v_packed) & 7) ||
      (((uintptr_t)k_scale | (uintptr_t)k_zero | (uintptr_t)v_scale | (uintptr_t)v_zero) & 3))
    return TKV_EINVAL;
  const int whole = N / T * T;
  if ((int64_t)HKV * (whole / T) > INT32_MAX / 256) return TKV_EINVAL;
  constexpr int kMaxB = 65535;  // a grid's y limit: more batch rows go in pieces
  for (int b0 = 0; B > kMaxB && b0 < B; b0 += kMaxB) {
    const int64_t r = (int64_t)b0 * HKV;
    const int rc = tkv_channel_extend(
        static_cast<const uint16_t*>(k) + b0 * k_strides[0], k_strides,
        static_cast<const uint16_t*>(v) + b0 * v_strides[0], v_strides, B - b0 < kMaxB ? B - b0 : kMaxB,
        HKV, N, D, k_nbits, v_nbits, group_size, start, static_cast<uint16_t*>(k_res) + r * T * D,
        static_cast<uint16_t*>(v_res) + r * T * D, res_cap, q_lens + b0, res_lens + b0, S_cap,
        k_packed + r * S_cap * (D * k_nbits / 8), k_scale + r * (S_cap / T) * D,
        k_zero + r * (S_cap / T) * D, v_packed + r * S_cap * (D * v_nbits / 8),
        v_scale + r * S_cap * (D / group_size), v_zero + r * S_cap * (D / group_size), stream);
    if (rc || b0 + kMaxB >= B) return rc;
  }
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  (void)hipGetLastError();
#define TKV_CE(Dv, NBv)                                                                       \
  launch_channel_extend<Dv, NBv>(ks, vs, B, HKV, N, start, S_cap, k_packed, k_scale, k_zero,  \
                                 static_cast<uint16_t*>(k_res), static_cast<uint16_t*>(v_res), \
                                 q_lens, res_lens, st)
  if (D == 128) {
    if (k_nbits == 4) TKV_CE(128, 4); else TKV_CE(128, 2);
  } else {
    if (k_nbits == 4) TKV_CE(64, 4); else TKV_CE(64, 2);
  }
#undef TKV_CE
  if (whole) {
    bool done = false;
#define TKV_VT(Dv, NBv, GSv) \
  done = launch_tokens<Dv, NBv, GSv>(vs, (int64_t)B * HKV * whole >= kBulkRows, B, HKV, whole, nullptr, start, S_cap, v_packed, v_scale, v_zero, st)
    TKV_DISPATCH_DNG(D, v_nbits, group_size, TKV_VT);
#undef TKV_VT
    if (!done) return TKV_EINVAL;
  }
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? TKV_OK : (int)e;
}

extern "C" int tkv_channel_window_append(const void* k_new, const void* v_new, int32_t B,
                                         int32_t HKV, int32_t D, void* k_res, void* v_res,
                                         int32_t res_cap, int32_t* res_lens, tkv_stream_t stream) {
  using namespace tkv;
  if (!k_new || !v_new || !k_res || !v_res || !res_lens) return TKV_EINVAL;
  if (B <= 0 || HKV <= 0 || (D != 64 && D != 128)) return TKV_EINVAL;
  if (res_cap != 32) return TKV_EINVAL;
  if (((uintptr_t)k_new | (uintptr_t)v_new | (uintptr_t)k_res | (uintptr_t)v_res) & 15)
    return TKV_EINVAL;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  (void)hipGetLastError();
  channel_window_append_kernel<<<dim3((unsigned)B), 256, 0, st>>>(
      static_cast<const uint16_t*>(k_new), static_cast<const uint16_t*>(v_new), HKV, D,
      static_cast<uint16_t*>(k_res), static_cast<uint16_t*>(v_res), res_lens);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? TKV_OK : (int)e;
}

extern "C" int tkv_channel_window_flush(const void* k_res, const void* v_res, int32_t B,
                                        int32_t HKV, int32_t D, int32_t k_nbits, int32_t v_nbits,
                                        int32_t group_size, int32_t res_cap, int32_t* q_lens,
                                        int32_t* res_lens, int32_t S_cap, uint8_t* k_packed,
                                        uint16_t* k_scale, uint16_t* k_zero, uint8_t* v_packed,
                                        uint16_t* v_scale, uint16_t* v_zero, tkv_stream_t stream) {
  using namespace tkv;
  if (!k_res || !v_res || !q_lens || !res_lens || !k_packed || !k_scale || !k_zero || !v_packed ||
      !v_scale || !v_zero)
    return TKV_EINVAL;
  if (B <= 0 || HKV <= 0 || S_cap <= 0 || S_cap % 32 || res_cap != 32) return TKV_EINVAL;
  if ((k_nbits != 2 && k_nbits != 4) || (v_nbits != 2 && v_nbits != 4)) return TKV_EINVAL;
  if (((uintptr_t)k_res | (uintptr_t)v_res) & 1) return TKV_EINVAL;
  if ((((uintptr_t)k_scale | (uintptr_t)k_zero | (uintptr_t)v_scale | (uintptr_t)v_zero) & 1))
    return TKV_EINVAL;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)B);
  const uint16_t* kr = static_cast<const uint16_t*>(k_res);
  const uint16_t* vr = static_cast<const uint16_t*>(v_res);
  (void)hipGetLastError();
#define TKV_FL(Dv, KB, VB, GSv)                                                                  \
  channel_window_flush_kernel<Dv, KB, VB, GSv><<<grid, 256, 0, st>>>(                            \
      kr, vr, HKV, S_cap, q_lens, res_lens, k_packed, k_scale, k_zero, v_packed, v_scale, v_zero)
#define TKV_FL_GS(Dv, KB, VB)                                                                    \
  do {                                                                                           \
    if (group_size == 16) TKV_FL(Dv, KB, VB, 16);                                                \
    else if (group_size == 32) TKV_FL(Dv, KB, VB, 32);                                           \
    else return TKV_EUNSUPPORTED;                                                                \
  } while (0)
#define TKV_FL_V(Dv, KB)                                                                         \
  do {                                                                                           \
    if (v_nbits == 4) TKV_FL_GS(Dv, KB, 4); else TKV_FL_GS(Dv, KB, 2);                          \
  } while (0)
  if (D == 128) {
    if (k_nbits == 4) TKV_FL_V(128, 4); else TKV_FL_V(128, 2);
  } else if (D == 64) {
    if (k_nbits == 4) TKV_FL_V(64, 4); else TKV_FL_V(64, 2);
  } else {
    return TKV_EUNSUPPORTED;
  }
#undef TKV_FL_V
#undef TKV_FL_GS
#undef TKV_FL
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? TKV_OK : (int)e;
}

extern "C" int tkv_pack_codes(const uint8_t* codes, int64_t rows, int32_t D, int32_t nbits,
                              uint8_t* packed, tkv_stream_t stream) {
  using namespace tkv;
  if (!codes || !packed || rows <= 0 || D <= 0) return TKV_EINVAL;
  if (nbits != 2 && nbits != 4) return TKV_EINVAL;
  const int P = 8 / nbits;
  if (D % (4 * P)) return TKV_EUNSUPPORTED;  // whole packed dwords per row
  if ((uintptr_t)packed & 3) return TKV_EINVAL;
  const int64_t n = rows * (D / P / 4);
  (void)hipGetLastError();
  const int64_t blocks = (n + 255) / 256 < (1 << 20) ? (n + 255) / 256 : (1 << 20);  // grid-stride beyond
  pack_codes_kernel<<<dim3((unsigned)blocks), 256, 0,
                      reinterpret_cast<hipStream_t>(stream)>>>(codes, rows, D, nbits, packed);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? TKV_OK : (int)e;
}

extern "C" int tkv_unpack_dequant(const uint8_t* packed, const uint16_t* scale,
                                  const uint16_t* zero, int64_t rows, int32_t D, int32_t nbits,
                                  int32_t group_size, int32_t path, uint8_t* codes_out,
                                  float* values_out, tkv_stream_t stream) {
  using namespace tkv;
  if (!packed || rows <= 0 || D <= 0) return TKV_EINVAL;
  if (nbits != 2 && nbits != 4) return TKV_EINVAL;
  if (group_size <= 0 || D % group_size) return TKV_EINVAL;
  if (path != 0 && path != 1) return TKV_EINVAL;
  if (values_out && (!scale || !zero)) return TKV_EINVAL;
  if ((uintptr_t)packed & 7) return TKV_EINVAL;  // dwordx2 loads of the K unpack path
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  (void)hipGetLastError();
#define TKV_U(Dv, NBv, GSv) \
  launch_unpack<Dv, NBv, GSv>(packed, scale, zero, rows, path, codes_out, values_out, st)
  TKV_DISPATCH_DNG(D, nbits, group_size, TKV_U);
#undef TKV_U
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? TKV_OK : (int)e;
}
