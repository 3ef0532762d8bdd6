// Device-side pieces shared by the convolution kernels: MFMA register layout helpers, the
// saturating pack, the 64-bit-constant requantisation of a row block, the fused EltwiseAdd on 16
// requantised channels, and buffer-descriptor loads.
#pragma once

#include "common.hpp"

#include <type_traits>
#include <utility>

namespace tpuhip {}
using namespace tpuhip;

// f(integral_constant<int, 0>) ... f(integral_constant<int, N - 1>), in order: a loop whose index is a
// compile-time constant in every trip
template <typename F, int... I>
__device__ __forceinline__ void static_for_impl(F &&f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F &&f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef unsigned int v4u __attribute__((ext_vector_type(4)));

// tile-local weight row (as the MFMA sees it) -> tile-local output channel
__host__ __device__ inline int mfma_row_to_oc(int row, int tm) {
  const int wave_rows = tm * 32;
  const int wrow = row % wave_rows, wbase = row - wrow;
  const int i = wrow / 32, ri = wrow % 32;
  const int fk = (ri >> 2) & 1;
  const int r = (ri >> 3) * 4 + (ri & 3);
  return wbase + fk * 16 * tm + i * 16 + r;
}

typedef short v2s __attribute__((ext_vector_type(2)));
typedef unsigned short v2us __attribute__((ext_vector_type(2)));

// four int32 -> four saturated int8 in one dword; lo is -128 or 0 (fused ReLU)
__device__ __forceinline__ uint32_t pack_sat4(int32_t a, int32_t b, int32_t c, int32_t d, int lo) {
  v2s p0 = __builtin_amdgcn_cvt_pk_i16(a, b);
  v2s p1 = __builtin_amdgcn_cvt_pk_i16(c, d);
  const v2s vlo = {(short)lo, (short)lo}, vhi = {127, 127};
  p0 = __builtin_elementwise_min(__builtin_elementwise_max(p0, vlo), vhi);
  p1 = __builtin_elementwise_min(__builtin_elementwise_max(p1, vlo), vhi);
  return __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, p1), __builtin_bit_cast(uint32_t, p0),
                               0x06040200u);
}

// 16-byte load through a buffer descriptor: an offset at or beyond the
// descriptor's size yields zeros, which is how padding taps, pixels past the end
// of the tensor and K steps past the end of the filter are fed to the MFMAs
// without a branch.
__device__ __forceinline__ v4i buffer_load16(__amdgpu_buffer_rsrc_t rsrc, uint32_t offset) {
  return (v4i)__builtin_amdgcn_raw_buffer_load_b128(rsrc, offset, 0, 0);
}
constexpr uint32_t kOobOffset = 0x7fffffffu;

// Requantisation of accumulators that started at zero, for layers whose overflow-free form the
// host has proved: the bias rides in the addend of the 64-bit multiply-add,
//   (acc + b) * m + 2^30 == acc * m + c,   c = b * m + 2^30   (pc64: (low, high) pairs per channel).
// RELU (the layer clamps at 0 after saturation): pc64 holds c + 2^(r-1) * 2^31, pshift r - 1, and the
// result is hi32(acc * m + c') >> (r - 1); otherwise x = (acc * m + c) >> 31 and the rounding shift
// (x + 2^(r-1) - (x < 0)) >> r with pshift = r, phpot = 2^(r-1).
template <int TN, bool RELU>
__device__ __forceinline__ void requant_rows_c64(const v16i (&acc)[TN], int lo, const int32_t *pc64,
                                                 const int32_t *pmult, const int32_t *pshift,
                                                 const int32_t *phpot, uint32_t (&outw)[TN][4]) {
#pragma unroll
  for (int qd = 0; qd < 4; ++qd) {
    const v4i c01 = *reinterpret_cast<const v4i *>(pc64 + qd * 8);
    const v4i c23 = *reinterpret_cast<const v4i *>(pc64 + qd * 8 + 4);
    const v4i m4 = *reinterpret_cast<const v4i *>(pmult + qd * 4);
    const v4i r4 = *reinterpret_cast<const v4i *>(pshift + qd * 4);
    v4i h4 = {0, 0, 0, 0};
    if (!RELU) h4 = *reinterpret_cast<const v4i *>(phpot + qd * 4);
    const int64_t c[4] = {(int64_t)(((uint64_t)(uint32_t)c01[1] << 32) | (uint32_t)c01[0]),
                          (int64_t)(((uint64_t)(uint32_t)c01[3] << 32) | (uint32_t)c01[2]),
                          (int64_t)(((uint64_t)(uint32_t)c23[1] << 32) | (uint32_t)c23[0]),
                          (int64_t)(((uint64_t)(uint32_t)c23[3] << 32) | (uint32_t)c23[2])};
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      int32_t y[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int64_t p = (int64_t)acc[j][qd * 4 + e] * (int64_t)m4[e] + c[e];
        if (RELU) {
          y[e] = (int32_t)(p >> 32) >> r4[e];
        } else {
          const int32_t x = (int32_t)(p >> 31);
          y[e] = (x + h4[e] + (x >> 31)) >> r4[e];
        }
      }
      outw[j][qd] = pack_sat4(y[0], y[1], y[2], y[3], lo);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

// The same requantisation with the saturation and the last shift left to packed int16 instructions, for layers whose constants
// allow it (narrow_requant()): with p' = (acc + b) * m / 2^f + ..., exact because 2^f divides m, the high word of p' holds the
// result times 2^s, s = r - 1 - f <= 8.  v_cvt_pk_i16_i32 saturates it to 16 bits, a saturating packed multiply by 2^(8-s) makes
// it the result times 256, and its high byte is the saturated result.
//   RELU: the rounding term is in pc64 and one multiply-add gives p'.
//   otherwise x = floor(p / 2^31) is rounded by x + 2^(r-1) - (x < 0): where p' < 0, one unit of x (2^(31-f), punit holds its
//   negative) is subtracted by a second multiply-add; 2^(r-1) is 128 in the packed scale, added with the multiply.
// 2.75 and 4.25 instructions per output, where the forms above take 3.75 and 6.75.  1x1 64 -> 256 on 32 x 56 x 56 16.5 -> 14.5 us,
// 3x3 128 -> 256 on 8 x 76 x 76 28.3 -> 26.2 (a leaky ReLU behind it included), 3x3 32 -> 64 on 8 x 304 x 304 49.4 -> 46.0;
// kernels that wait for memory (depthwise, 1x1 at 14 x 14) stay where they were.
// pscale: at an even channel 2^(8-s) of it and of the next one as two int16.
__device__ __forceinline__ int32_t pack_sat16(int32_t a, int32_t b) {
  return __builtin_bit_cast(int32_t, __builtin_amdgcn_cvt_pk_i16(a, b));
}
// the last steps for four channels under a ReLU: y the high words, s01 and s23 the pairs of scales
__device__ __forceinline__ uint32_t pack_narrow_relu(const int32_t (&y)[4], int32_t s01, int32_t s23) {
  int32_t a, b;
  asm("v_pk_mad_i16 %0, %1, %2, 0 clamp" : "=v"(a) : "v"(pack_sat16(y[0], y[1])), "v"(s01));
  asm("v_pk_mad_i16 %0, %1, %2, 0 clamp" : "=v"(b) : "v"(pack_sat16(y[2], y[3])), "v"(s23));
  const v2s zero = {0, 0};
  const v2s ra = __builtin_elementwise_max(__builtin_bit_cast(v2s, a), zero), rb = __builtin_elementwise_max(__builtin_bit_cast(v2s, b), zero);
  return __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, rb), __builtin_bit_cast(uint32_t, ra), 0x07050301u);
}
template <int TN, bool RELU>
__device__ __forceinline__ void requant_rows_narrow(const v16i (&acc)[TN], const int32_t *pc64, const int32_t *pmult,
                                                    const int32_t *pscale, const int32_t *punit, uint32_t (&outw)[TN][4]) {
  int32_t half = 0x00800080;
  asm("" : "+s"(half));
#pragma unroll
  for (int qd = 0; qd < 4; ++qd) {
    const v4i c01 = *reinterpret_cast<const v4i *>(pc64 + qd * 8);
    const v4i c23 = *reinterpret_cast<const v4i *>(pc64 + qd * 8 + 4);
    const v4i m4 = *reinterpret_cast<const v4i *>(pmult + qd * 4);
    const v4i s4 = *reinterpret_cast<const v4i *>(pscale + qd * 4);
    v4i u4 = {0, 0, 0, 0};
    if (!RELU) u4 = *reinterpret_cast<const v4i *>(punit + qd * 4);
    const int64_t c[4] = {(int64_t)(((uint64_t)(uint32_t)c01[1] << 32) | (uint32_t)c01[0]),
                          (int64_t)(((uint64_t)(uint32_t)c01[3] << 32) | (uint32_t)c01[2]),
                          (int64_t)(((uint64_t)(uint32_t)c23[1] << 32) | (uint32_t)c23[0]),
                          (int64_t)(((uint64_t)(uint32_t)c23[3] << 32) | (uint32_t)c23[2])};
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      int32_t y[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        int64_t p = (int64_t)acc[j][qd * 4 + e] * (int64_t)m4[e] + c[e];
        if (!RELU) {
          int32_t neg = (int32_t)((uint64_t)p >> 63);
          asm("" : "+v"(neg));   // a number to multiply by, not a condition to select with
          p = (int64_t)neg * (int64_t)u4[e] + p;
        }
        y[e] = (int32_t)(p >> 32);
      }
      if (RELU) {
        outw[j][qd] = pack_narrow_relu(y, s4[0], s4[2]);
      } else {
        int32_t a, b;
        asm("v_pk_mad_i16 %0, %1, %2, %3 clamp" : "=v"(a) : "v"(pack_sat16(y[0], y[1])), "v"(s4[0]), "s"(half));
        asm("v_pk_mad_i16 %0, %1, %2, %3 clamp" : "=v"(b) : "v"(pack_sat16(y[2], y[3])), "v"(s4[2]), "s"(half));
        outw[j][qd] = __builtin_amdgcn_perm((uint32_t)b, (uint32_t)a, 0x07050301u);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

__host__ __device__ inline bool allows_narrow(int32_t mult, int32_t rshift) {
  const int f = rshift > 9 ? rshift - 9 : 0;
  return rshift >= 2 && rshift <= 31 && !(mult & (int32_t)((1u << f) - 1u));
}
// One channel's constants for requant_rows_narrow; false: they do not allow it (a right shift of 1 or less, or a multiplier
// without the trailing zeros: one that was stored as a float has at least 7 below 2^31, which covers right shifts to 16).
// relu: c holds the rounding term of the short form.
__host__ __device__ inline bool narrow_requant(int64_t c, int32_t mult, int32_t rshift, int64_t *cn, int32_t *mn, int32_t *scale, int32_t *unit) {
  const int f = rshift > 9 ? rshift - 9 : 0, s = rshift - 1 - f;
  if (!allows_narrow(mult, rshift)) return false;
  *cn = c >> f;
  *mn = mult >> f;
  *scale = 1 << (8 - s);
  *unit = (int32_t)(0u - (1u << (31 - f)));
  return true;
}

// the form a layer's planes hold
template <int TN, bool NARROW>
__device__ __forceinline__ void requant_rows_planes(const v16i (&acc)[TN], bool relu, int lo, const int32_t *pc64,
                                                    const int32_t *pmult, const int32_t *pshift, const int32_t *phpot,
                                                    uint32_t (&outw)[TN][4]) {
  if constexpr (NARROW) {
    if (relu) requant_rows_narrow<TN, true>(acc, pc64, pmult, pshift, phpot, outw);
    else requant_rows_narrow<TN, false>(acc, pc64, pmult, pshift, phpot, outw);
  } else {
    if (relu) requant_rows_c64<TN, true>(acc, 0, pc64, pmult, pshift, phpot, outw);
    else requant_rows_c64<TN, false>(acc, lo, pc64, pmult, pshift, phpot, outw);
  }
}

// A leaky ReLU on four int8: max(y, (y * m + 2^(r-1)) >> r) with 0 < m <= 2^r, r >= 1 and 128 * m + 2^(r-1) < 2^15, on packed
// int16 (even and odd bytes apart): 2.5 instructions per output.  Zero stays zero, so pad channels do.
__device__ __forceinline__ uint32_t leaky_word(uint32_t w, int m, int r) {
  const v2us ueight = {8, 8};
  const v2s eight = {8, 8}, m2 = {(short)m, (short)m}, r2 = {(short)r, (short)r};
  const short half = (short)(1 << (r - 1));
  const v2s h2 = {half, half};
  const v2s lo = __builtin_bit_cast(v2s, __builtin_bit_cast(v2us, w) << ueight) >> eight, hi = __builtin_bit_cast(v2s, w) >> eight;
  const v2s zl = __builtin_elementwise_max(lo, (lo * m2 + h2) >> r2);
  const v2s zh = __builtin_elementwise_max(hi, (hi * m2 + h2) >> r2);
  return __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, zh), __builtin_bit_cast(uint32_t, zl), 0x06020400u);
}
__device__ __forceinline__ v4i leaky_chunk(const v4i &o, int m, int r) {
  v4i z;
#pragma unroll
  for (int q = 0; q < 4; ++q) z[q] = (int)leaky_word((uint32_t)o[q], m, r);
  return z;
}

// EltwiseAdd (core/eltwise.cpp:52-85, integer form) of 16 freshly requantised channels o with
// the other operand's 16 bytes sv:  sat8(floor(relu?(sv * m_src + o * m_conv) / 2^rshift + 0.5)).
// pk: |multipliers| <= 127 and rshift <= 8, so the sum fits packed int16 arithmetic.
__device__ __forceinline__ v4i fused_add_chunk(const v4i &o, const v4i &sv, int m_src, int m_conv, int rshift,
                                               int relu, int pk) {
  v4i z;
  if (pk) {
    // two outputs per instruction: the bytes of both operands widen to packed int16 (even and
    // odd bytes apart), src * m_src + y * m_conv + 2^(r-1) stays inside int16, and ReLU / lower
    // saturation (a floor before the shift), shift and upper saturation are packed ops too
    const int r = rshift;
    const short rnd = (short)(r > 0 ? (1 << (r - 1)) : 0);
    const short fl = (short)(relu ? 0 : -(128 << r));
    const v2s msrc = {(short)m_src, (short)m_src}, mconv = {(short)m_conv, (short)m_conv};
    const v2s rnd2 = {rnd, rnd}, fl2 = {fl, fl}, top = {127, 127}, sh = {(short)r, (short)r}, eight = {8, 8};
    const v2us ueight = {8, 8};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int32_t ow = o[q], sw_ = sv[q];   // plain copies: a vector element is no object to bit_cast
      const v2s o16 = __builtin_bit_cast(v2s, ow), s16 = __builtin_bit_cast(v2s, sw_);
      // even bytes: up by 8 as unsigned halves (a signed shift may be assumed not to overflow), down arithmetically
      const v2s olo = __builtin_bit_cast(v2s, __builtin_bit_cast(v2us, ow) << ueight) >> eight, ohi = o16 >> eight;
      const v2s slo = __builtin_bit_cast(v2s, __builtin_bit_cast(v2us, sw_) << ueight) >> eight, shi = s16 >> eight;
      v2s tlo = olo * mconv + (slo * msrc + rnd2);
      v2s thi = ohi * mconv + (shi * msrc + rnd2);
      tlo = __builtin_elementwise_min(__builtin_elementwise_max(tlo, fl2) >> sh, top);
      thi = __builtin_elementwise_min(__builtin_elementwise_max(thi, fl2) >> sh, top);
      z[q] = (int)__builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, thi), __builtin_bit_cast(uint32_t, tlo),
                                        0x06020400u);
    }
    return z;
  }
  // sum = src * m_src + y * m_conv as one 4 x int8 dot product per output (the two unused byte
  // lanes are zero), with the rounding term as its addend: adding 2^(r-1) before the ReLU gives
  // the same quotient as after it.
  int32_t rnd = rshift > 0 ? (1 << (rshift - 1)) : 0;
  int32_t mpair = (m_src & 0xff) | ((m_conv & 0xff) << 8);
  int32_t floor_ = relu ? 0 : (int32_t)0x80000000;
  // one scalar and one vector copy of the uniform operands, made once
  asm volatile("" : "+s"(rnd), "+v"(mpair), "+s"(floor_));
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    int32_t t[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const uint32_t pair = __builtin_amdgcn_perm((uint32_t)o[q], (uint32_t)sv[q],
                                                  0x0c0c0000u | ((4u + b) << 8) | (uint32_t)b);
      int32_t sum;   // the three-operand form: no copy of the addend into the result first
      asm("v_dot4_i32_i8 %0, %1, %2, %3" : "=v"(sum) : "v"(pair), "v"(mpair), "s"(rnd));
      t[b] = max(sum, floor_) >> rshift;
    }
    z[q] = (int)pack_sat4(t[0], t[1], t[2], t[3], -128);
  }
  return z;
}
