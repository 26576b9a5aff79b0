// Device-side building blocks shared by the Q4 kernels that feed MFMA.
#pragma once

#include "q4d_device.h"

namespace q4d {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));

// ---- int4 -> fp16 -----------------------------------------------------------------------
// A 32-bit word holds columns 0..7, low nibble first, as two's complement int4.  A nibble
// moved to bits 6..9 of an fp16 with its top bit flipped is the denormal u 2^-18, u = q + 8,
// exactly linear in u; one packed fma per pair then gives
//     (u 2^-18) (s 2^18) - 8 s = q s
// rounded once, the same value as the fp16 product of q and s.  s 2^18 (the Q2.14 code times
// 16) is a finite fp16 up to code 4094; larger codes (scale 0.25 and more) go through the
// integers (codes_wide).  Shift + bit operation + fma per pair: 12 VALU instructions per
// word in pair order, 16 in column order, against 20 through 0x6400 | u, subtract, multiply.
constexpr uint32_t kScaleFastMax = 4094;

struct W16Scale {
  h2 mul, add;  // s 2^18 and -8 s, s = the fp16 scale
  h2 s;
};
__device__ __forceinline__ W16Scale w16_scale(uint32_t code) {
  const _Float16 m = (_Float16)((float)code * 16.0f), b = (_Float16)((float)code * (-8.0f / 16384.0f));
  const _Float16 s = (_Float16)((float)code * (1.0f / 16384.0f));
  return {make_h2(m, m), make_h2(b, b), make_h2(s, s)};
}
// Nibbles at bits 6..9 and 22..25, top bits flipped.
__device__ __forceinline__ uint32_t nib_pair(uint32_t x) { return (x & 0x03C003C0u) ^ 0x02000200u; }

// Whether any lane of the wave holds a scale code past the fast form's range.
__device__ __forceinline__ bool scale_wide(uint32_t code) { return __builtin_amdgcn_ballot_w64(code > kScaleFastMax); }

// fp16 integers of a word in pair order (word p = columns p, p + 4): (0x6400 | u) - 1032.
__device__ __forceinline__ u32x4 codes_wide(uint32_t w) {
  const h2 bias = make_h2((_Float16)1032.0f, (_Float16)1032.0f);
  const uint32_t v = w ^ 0x88888888u;
  u32x4 out;
#pragma unroll
  for (int p = 0; p < 4; ++p)
    out[p] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2, ((v >> (4 * p)) & 0x000F000Fu) | 0x64006400u) - bias);
  return out;
}

// q x scale in pair order: word p = columns p, p + 4 (an MFMA does not depend on the order of
// the eight k values of a lane, as long as both operands share it).
template <bool WIDE>
__device__ __forceinline__ u32x4 dequant8_pairs(uint32_t w, const W16Scale& f) {
  u32x4 out;
  if constexpr (WIDE) {
    const u32x4 q = codes_wide(w);
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const uint32_t qp = q[p];
      out[p] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2, qp) * f.s);
    }
  } else {
    const uint32_t x[4] = {w << 6, w << 2, w >> 2, w >> 6};
#pragma unroll
    for (int p = 0; p < 4; ++p)
      out[p] = __builtin_bit_cast(
          uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(h2, nib_pair(x[p])), f.mul, f.add));
  }
  return out;
}

// q / 8 exactly, in pair order.
__device__ __forceinline__ u32x4 codes8_pairs(uint32_t w) {
  const h2 mul = make_h2((_Float16)32768.0f, (_Float16)32768.0f), add = make_h2((_Float16)-1.0f, (_Float16)-1.0f);
  const uint32_t x[4] = {w << 6, w << 2, w >> 2, w >> 6};
  u32x4 out;
#pragma unroll
  for (int p = 0; p < 4; ++p)
    out[p] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(h2, nib_pair(x[p])), mul, add));
  return out;
}

// q x scale in column order: word p = columns 2p, 2p + 1.
template <bool WIDE>
__device__ __forceinline__ u32x4 dequant8(uint32_t w, const W16Scale& f) {
  u32x4 out;
  if constexpr (WIDE) {
    const h2 bias = make_h2((_Float16)1032.0f, (_Float16)1032.0f);
    const uint32_t v = w ^ 0x88888888u;
    const uint32_t lo = v & 0x0F0F0F0Fu;         // nibbles 0, 2, 4, 6 in bytes 0..3
    const uint32_t hi = (v >> 4) & 0x0F0F0F0Fu;  // nibbles 1, 3, 5, 7
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      // fp16 pair (nibble 2p, nibble 2p+1): low byte of each half from lo / hi byte p
      const uint32_t sel = (uint32_t)(p) | (0x0Cu << 8) | ((uint32_t)(4 + p) << 16) | (0x0Cu << 24);
      const uint32_t pr = __builtin_amdgcn_perm(hi, lo, sel) | 0x64006400u;
      out[p] = __builtin_bit_cast(uint32_t, (__builtin_bit_cast(h2, pr) - bias) * f.s);
    }
  } else {
    const uint32_t a = w << 6, b = w << 2, c = w >> 2, d = w >> 6;
    const uint32_t x[4] = {__builtin_amdgcn_perm(b, a, 0x05040100u), __builtin_amdgcn_perm(d, c, 0x05040100u),
                           __builtin_amdgcn_perm(b, a, 0x07060302u), __builtin_amdgcn_perm(d, c, 0x07060302u)};
#pragma unroll
    for (int p = 0; p < 4; ++p)
      out[p] = __builtin_bit_cast(
          uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(h2, nib_pair(x[p])), f.mul, f.add));
  }
  return out;
}

// Eight fp16 values (column order) into pair order.
__device__ __forceinline__ u32x4 to_pairs(const u32x4 v) {
  return u32x4{__builtin_amdgcn_perm(v[2], v[0], 0x05040100u), __builtin_amdgcn_perm(v[2], v[0], 0x07060302u),
               __builtin_amdgcn_perm(v[3], v[1], 0x05040100u), __builtin_amdgcn_perm(v[3], v[1], 0x07060302u)};
}

// Word s of lane row group G becomes word G of row group s (lane l % 16 kept).
// v_permlane32_swap(A, B) returns (A.lo | B.lo, A.hi | B.hi) over lanes 0-31 | 32-63;
// v_permlane16_swap(A, B) returns (A.r0 | B.r0 | A.r2 | B.r2, A.r1 | B.r1 | A.r3 | B.r3)
// over the 16-lane rows r0..r3.
__device__ __forceinline__ void rows_transpose4(uint32_t (&d)[4]) {
  // the off-diagonal 2 x 2 blocks: rows 0-1 words 2-3 <-> rows 2-3 words 0-1
  const auto a = __builtin_amdgcn_permlane32_swap(d[0], d[2], false, false);
  const auto b = __builtin_amdgcn_permlane32_swap(d[1], d[3], false, false);
  const uint32_t e0 = a[0], e2 = a[1], e1 = b[0], e3 = b[1];
  // inside each 2 x 2 block: the even rows' odd words <-> the odd rows' even words
  const auto c = __builtin_amdgcn_permlane16_swap(e0, e1, false, false);
  const auto f = __builtin_amdgcn_permlane16_swap(e2, e3, false, false);
  d[0] = c[0];
  d[1] = c[1];
  d[2] = f[0];
  d[3] = f[1];
}

// ---- arithmetic the prefill GEMM epilogues share ------------------------------------
// A prompt in chunks gives the same bits as one call whichever kernel a chunk's size picks,
// so the roundings are spelt out: sums as explicit fused multiply-adds, and a product that
// goes to fp16 either rounded once (mul_f16) or pinned in fp32 first.  Left to itself the
// compiler may choose differently in each kernel.
__device__ __forceinline__ float pin_f32(float v) {
  asm volatile("" : "+v"(v));
  return v;
}
// a * b rounded once to fp16.
__device__ __forceinline__ _Float16 mul_f16(float a, float b) {
  uint32_t d;
  asm("v_fma_mixlo_f16 %0, %1, %2, 0" : "=v"(d) : "v"(a), "v"(b));
  return __builtin_bit_cast(_Float16, (uint16_t)d);
}

__device__ __forceinline__ _Float16 swiglu(float g, float u) { return mul_f16(g / (1.0f + expf(-g)), u); }

// One head's row in the hands of two 16-lane rows: lane cl of half wn holds x[j] = dims
// 32 wn + 16 j + cl and x[j + 2] = their rotate-half partners + 64 (j = 0, 1).
// This half's part of the sum of squares (the same in its 16 lanes):
__device__ __forceinline__ float rope_half_ss(float x0, float x1, float x2, float x3) {
  return row16_sum(fmaf(x3, x3, fmaf(x2, x2, fmaf(x1, x1, x0 * x0))));
}
__device__ __forceinline__ float rope_inv(float ss, float eps) { return 1.0f / sqrtf(fmaf(ss, 1.0f / 128.0f, eps)); }
// RMSNorm scale, gamma and rotation of dim d (a) and d + 64 (b), in place:
__device__ __forceinline__ void rope_pair(float& a, float& b, float inv, float ga, float gb, float c, float s) {
  const float n0 = (a * inv) * ga, n1 = (b * inv) * gb;
  a = fmaf(n0, c, -pin_f32(n1 * s));
  b = fmaf(n0, s, pin_f32(n1 * c));
}
// q leaves with the softmax scale folded in: dim d rounded once, dim d + 64 after an fp32
// product.
__device__ __forceinline__ _Float16 rope_q_lo(float v, float qscale) { return mul_f16(v, qscale); }
__device__ __forceinline__ _Float16 rope_q_hi(float v, float qscale) { return (_Float16)pin_f32(v * qscale); }

}  // namespace q4d
