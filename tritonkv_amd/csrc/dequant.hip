// Whole-cache dequantization and unpacking: packed split-P codes back to
// values (fp32, fp16 or bf16) or to uint8 codes.
//
// Reference behaviour being reproduced:
//   unpack_codes         quantize.py:172-183
//   dequantize_groupwise quantize.py:239-246 (fp32 code * scale + zero, then
//       the caller's dtype; the product is exact, so fmaf gives the same bits
//       as the reference's mul-then-add)
//
// Bound by HBM: a row's codes and metadata are read once and its values
// written once, in the caller's dtype (no fp32 intermediate).  A lane takes E
// consecutive packed bytes of a row, whose P slices are P runs of E
// consecutive dims, and stores each run as one 16-byte vector (E = 8 fp16 /
// bf16 values, 4 fp32 ones; 8 bytes of codes), so every store instruction
// covers whole 64- or 128-byte pieces of rows.  Each lane loads the codes and
// metadata of two rows before it uses either.  Measured at 131056 rows of
// D = 128, 4-bit, groups of 32, to fp16: 8.0 us a launch (5.5 TB/s of codes,
// metadata and values), against 47.8 us for the decode kernel's unpack order
// (one 4-byte store per value) and 14.8 us for a conversion pass after it.
#include "../../include/tkv.h"
#include "tkv_device.h"

namespace tkv {

typedef __bf16 bf8 __attribute__((ext_vector_type(8)));

enum { kOutFp32 = 0, kOutFp16 = 1, kOutBf16 = 2, kOutCodes = 3 };

// fp32 -> bf16, ties to even; a NaN becomes torch's canonical 0x7FC0.
__device__ __forceinline__ __bf16 to_bf16(float v) {
  return v != v ? __builtin_bit_cast(__bf16, (uint16_t)0x7FC0u) : (__bf16)v;
}

template <int D, int NB, int GS, int OUT>
__global__ void __launch_bounds__(256)
dequant_kernel(const uint8_t* __restrict__ packed, const uint16_t* __restrict__ scale,
               const uint16_t* __restrict__ zero, int64_t rows, void* __restrict__ out) {
  constexpr int P = 8 / NB, DP = D / P, NG = D / GS;
  constexpr int E = OUT == kOutFp32 ? 4 : 8;  // packed bytes, and values of a run, per lane
  constexpr int LPR = DP / E, RPS = 64 / LPR, STEPS = 2;
  constexpr bool VALUES = OUT != kOutCodes;
  static_assert(DP % E == 0 && LPR <= 64 && GS % E == 0, "row shape");
  const int lane = threadIdx.x & 63, slot = lane / LPR, c = lane % LPR;
  const int64_t stride = (int64_t)gridDim.x * 4 * STEPS * RPS;
  for (int64_t first = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * STEPS * RPS; first < rows;
       first += stride) {
    uint32_t w[STEPS][E / 4];
    uint16_t sb[STEPS][P], zb[STEPS][P];
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
      int64_t row = first + s * RPS + slot;
      if (row >= rows) row = rows - 1;
      const uint8_t* src = packed + row * DP + c * E;
      if constexpr (E == 8) {
        const u2 v = ld_u2(src);
        w[s][0] = v[0];
        w[s][1] = v[1];
      } else {
        w[s][0] = ld_u32(src);
      }
      if constexpr (VALUES) {
#pragma unroll
        for (int p = 0; p < P; ++p) {
          const int64_t g = row * NG + (p * DP + c * E) / GS;
          sb[s][p] = scale[g];
          zb[s][p] = zero[g];
        }
      }
    }
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
      const int64_t row = first + s * RPS + slot;
      if (row >= rows) continue;
      const int64_t dst = row * D + c * E;
#pragma unroll
      for (int p = 0; p < P; ++p) {
        uint32_t k[E / 4];  // slice p's codes, one per byte
#pragma unroll
        for (int i = 0; i < E / 4; ++i) k[i] = (w[s][i] >> (p * NB)) & (((1u << NB) - 1u) * 0x01010101u);
        if constexpr (VALUES) {
          const float sf = (float)__builtin_bit_cast(_Float16, sb[s][p]);
          const float zf = (float)__builtin_bit_cast(_Float16, zb[s][p]);
          float v[E];
#pragma unroll
          for (int e = 0; e < E; ++e) v[e] = fmaf((float)((k[e / 4] >> (8 * (e % 4))) & 0xFFu), sf, zf);
          if constexpr (OUT == kOutFp32) {
            *reinterpret_cast<f4*>(static_cast<float*>(out) + dst + p * DP) = f4{v[0], v[1], v[2], v[3]};
          } else if constexpr (OUT == kOutFp16) {
            h8 o;
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] = (_Float16)v[e];
            *reinterpret_cast<h8*>(static_cast<_Float16*>(out) + dst + p * DP) = o;
          } else {
            bf8 o;
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] = to_bf16(v[e]);
            *reinterpret_cast<bf8*>(static_cast<__bf16*>(out) + dst + p * DP) = o;
          }
        } else {
          *reinterpret_cast<u2*>(static_cast<uint8_t*>(out) + dst + p * DP) = u2{k[0], k[1]};
        }
      }
    }
  }
}

template <int D, int NB, int GS, int OUT>
static void launch_dequant(const uint8_t* packed, const uint16_t* scale, const uint16_t* zero,
                           int64_t rows, void* out, hipStream_t st) {
  constexpr int DP = D * NB / 8, E = OUT == kOutFp32 ? 4 : 8;
  constexpr int64_t per_wg = 4 * 2 * (64 / (DP / E));  // waves x steps x rows a step
  const int64_t wgs = (rows + per_wg - 1) / per_wg, most = 1 << 22;  // grid-stride beyond
  dequant_kernel<D, NB, GS, OUT><<<dim3((unsigned)(wgs < most ? wgs : most)), 256, 0, st>>>(
      packed, scale, zero, rows, out);
}

template <int D, int NB, int GS>
static int dispatch_out(const uint8_t* packed, const uint16_t* scale, const uint16_t* zero,
                        int64_t rows, int out_type, void* out, hipStream_t st) {
  switch (out_type) {
    case kOutFp32: launch_dequant<D, NB, GS, kOutFp32>(packed, scale, zero, rows, out, st); break;
    case kOutFp16: launch_dequant<D, NB, GS, kOutFp16>(packed, scale, zero, rows, out, st); break;
    default: launch_dequant<D, NB, GS, kOutBf16>(packed, scale, zero, rows, out, st); break;
  }
  return TKV_OK;
}

template <int D, int NB>
static int dispatch_group(const uint8_t* packed, const uint16_t* scale, const uint16_t* zero,
                          int64_t rows, int gs, int out_type, void* out, hipStream_t st) {
  if (out_type == kOutCodes) {  // codes do not depend on the group size
    launch_dequant<D, NB, D, kOutCodes>(packed, scale, zero, rows, out, st);
    return TKV_OK;
  }
  switch (gs) {
    case 16: return dispatch_out<D, NB, 16>(packed, scale, zero, rows, out_type, out, st);
    case 32: return dispatch_out<D, NB, 32>(packed, scale, zero, rows, out_type, out, st);
    case 64: return dispatch_out<D, NB, 64>(packed, scale, zero, rows, out_type, out, st);
    case 128:
      if constexpr (D >= 128) return dispatch_out<D, NB, 128>(packed, scale, zero, rows, out_type, out, st);
      return TKV_EUNSUPPORTED;
    default: return TKV_EUNSUPPORTED;
  }
}

}  // namespace tkv

extern "C" int tkv_dequantize(const uint8_t* packed, const uint16_t* scale, const uint16_t* zero,
                              int64_t rows, int32_t D, int32_t nbits, int32_t group_size,
                              int32_t out_type, void* out, tkv_stream_t stream) {
  using namespace tkv;
  if (!packed || !out || rows <= 0 || D <= 0) return TKV_EINVAL;
  if (nbits != 2 && nbits != 4) return TKV_EINVAL;
  if (group_size <= 0 || D % group_size) return TKV_EINVAL;
  if (out_type < kOutFp32 || out_type > kOutCodes) return TKV_EINVAL;
  if (out_type != kOutCodes && (!scale || !zero)) return TKV_EINVAL;
  if (((uintptr_t)packed & 7) || ((uintptr_t)scale & 1) || ((uintptr_t)zero & 1)) return TKV_EINVAL;
  if ((uintptr_t)out & (out_type == kOutCodes ? 7 : 15)) return TKV_EINVAL;
  if (D != 64 && D != 128) return TKV_EUNSUPPORTED;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  (void)hipGetLastError();
  int rc;
  if (D == 128)
    rc = nbits == 4 ? dispatch_group<128, 4>(packed, scale, zero, rows, group_size, out_type, out, st)
                    : dispatch_group<128, 2>(packed, scale, zero, rows, group_size, out_type, out, st);
  else
    rc = nbits == 4 ? dispatch_group<64, 4>(packed, scale, zero, rows, group_size, out_type, out, st)
                    : dispatch_group<64, 2>(packed, scale, zero, rows, group_size, out_type, out, st);
  if (rc) return rc;
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? TKV_OK : (int)e;
}
