// Matrix-core helpers shared by the mean scorer (score_mfma.hip) and the
// max-over-offsets scorer (score_max.hip).
#pragma once

#include "score_internal.h"

namespace kvc {

constexpr int kMfmaMaxQpk = 8;                // make_shape admits qpk <= 8
constexpr int kStageStride = kScoreTile + 4;  // floats per staged query-head row

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Two floats -> packed bf16 pair, round to nearest even (one v_cvt_pk_bf16_f32).
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
}
// Two floats -> packed fp16 pair, round to nearest even (one v_cvt_pk_f16_f32).
__device__ __forceinline__ uint32_t pack_f16(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, f16x2));
}

// The 16-bit element type of a cache: A/B operand vector, the MFMA, the
// unpacking and hi/lo packing of |k|.
template <bool F16>
struct MfmaElem;
template <>
struct MfmaElem<false> {
  typedef bf16x8 vec;
  static constexpr float kMagScale = 1.0f;
  static constexpr float kLowScale = 1.0f;
  static constexpr uint32_t kLeadMask = 0xffffu;
  __device__ __forceinline__ static f32x4 mfma(vec a, vec b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
  __device__ __forceinline__ static float lo(uint32_t w) { return bf16_lo(w); }
  __device__ __forceinline__ static float hi(uint32_t w) { return bf16_hi(w); }
  __device__ __forceinline__ static uint32_t pack(float a, float b) { return pack_bf16(a, b); }
  // Sum of both halves' squares.  The dot instruction rounds a little less well
  // than a product and a multiply-add (root mean square error 0.112 against 0.103
  // x 2^-24), far below the 2^-16 that two bf16 words of the root keep.
  __device__ __forceinline__ static float square_sum(uint32_t w) {
    const bf16x2 v = __builtin_bit_cast(bf16x2, w);
    return __builtin_amdgcn_fdot2_f32_bf16(v, v, 0.0f, false);
  }
};
template <>
struct MfmaElem<true> {
  typedef f16x8 vec;
  static constexpr float kMagScale = 0.25f;  // |k| of fp16 keys reaches 2^16.5
  // Of three words the first keeps eight significant bits, as bf16 does: its
  // products then leave the matrix core's sum the bits that full fp16 products
  // would use up.  Each further word is held times 2^8 (at most 2^15), so that
  // fp16's subnormals cut a weight at 2^-54 of its column's largest and |k| at
  // 2^-40; the products are scaled back.
  static constexpr float kLowScale = 1.0f / 256.0f;
  static constexpr uint32_t kLeadMask = 0xfff8u;
  __device__ __forceinline__ static f32x4 mfma(vec a, vec b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
  __device__ __forceinline__ static float lo(uint32_t w) { return fp16_lo(w); }
  __device__ __forceinline__ static float hi(uint32_t w) { return fp16_hi(w); }
  __device__ __forceinline__ static uint32_t pack(float a, float b) { return pack_f16(a, b); }
  // Two fp16 words keep 2^-22 of the root, where the dot instruction's rounding
  // (0.31 against 0.29 x 2^-24) showed: scores of 20000 tokens of 128 dims were
  // 8.246e-8 from float64 with it, 8.214e-8 without.
  __device__ __forceinline__ static float square_sum(uint32_t w) {
    const float re = lo(w), im = hi(w);
    return fmaf(im, im, re * re);
  }
};

// K is read once per scoring layer, with plain loads: non-temporal ones
// (meant to keep K from evicting the weight fragments in L2) measured 0.85 ms
// against 0.72 ms on the Qwen2.5-14B shape.
__device__ __forceinline__ u32x4 load_k(KVC_GLOBAL const u32x4* p) {
  return *p;
}

// Round-to-nearest-even float32 -> bf16 bits (finite inputs).
__device__ __forceinline__ uint32_t bf16_bits(float x) {
  const uint32_t u = __float_as_uint(x);
  return (u + 0x7FFFu + ((u >> 16) & 1u)) >> 16;
}
__device__ __forceinline__ float bf16_value(uint32_t bits) { return __uint_as_float(bits << 16); }

// |k| of the eight frequencies of magnitude K step q held by this lane, as
// TERMS 16-bit A operands, each the rounding of what the ones before it leave
// (two: |k| * kMagScale to ~2^-16; three: to float32, each divided by kLowScale
// more than the one before).  Two frequencies per output word: half style pairs word w of linear steps q
// (real parts) and q + NF (imaginary parts); interleaved takes words 2w, 2w+1
// of step 2q (w < 2) or 2q + 1, each word one (real, imaginary) pair.
template <bool F16, bool IL, int NK, int NF, int TERMS>
__device__ __forceinline__ void magnitude_words(const u32x4 (&ka)[NK], int q, typename MfmaElem<F16>::vec (&out)[TERMS]) {
  typedef MfmaElem<F16> E;
  typedef typename E::vec vec_t;
  u32x4 words[TERMS];
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    uint32_t re_w, im_w;
    if (IL) {
      const uint32_t w0 = ka[2 * q + (w >> 1)][(2 * w) & 3], w1 = ka[2 * q + (w >> 1)][(2 * w + 1) & 3];
      // (re0, re1) = (lo of w0, lo of w1), (im0, im1) = (hi of w0, hi of w1)
      re_w = (w0 & 0xffffu) | (w1 << 16);
      im_w = (w0 >> 16) | (w1 & 0xffff0000u);
    } else {
      re_w = ka[q][w];
      im_w = ka[q + NF][w];
    }
    float m0, m1;
    if constexpr (TERMS == 2) {
      // Sums of squares of (real, imaginary) words.
      const uint32_t p0 = IL ? ka[2 * q + (w >> 1)][(2 * w) & 3] : __builtin_amdgcn_perm(im_w, re_w, 0x05040100);
      const uint32_t p1 = IL ? ka[2 * q + (w >> 1)][(2 * w + 1) & 3] : __builtin_amdgcn_perm(im_w, re_w, 0x07060302);
      m0 = __builtin_amdgcn_sqrtf(E::square_sum(p0)) * E::kMagScale;
      m1 = __builtin_amdgcn_sqrtf(E::square_sum(p1)) * E::kMagScale;
    } else {
      const float re0 = E::lo(re_w), re1 = E::hi(re_w);
      const float im0 = E::lo(im_w), im1 = E::hi(im_w);
      m0 = __builtin_amdgcn_sqrtf(fmaf(im0, im0, re0 * re0)) * E::kMagScale;
      m1 = __builtin_amdgcn_sqrtf(fmaf(im1, im1, re1 * re1)) * E::kMagScale;
    }
#pragma unroll
    for (int k = 0; k < TERMS; ++k) {
      uint32_t word = E::pack(m0, m1);
      if (F16 && TERMS == 3 && k == 0) word &= E::kLeadMask * 0x10001u;
      words[k][w] = word;
      m0 -= E::lo(word);
      m1 -= E::hi(word);
      if (TERMS == 3 && k < 2) {
        m0 *= 1.0f / E::kLowScale;
        m1 *= 1.0f / E::kLowScale;
      }
    }
  }
#pragma unroll
  for (int k = 0; k < TERMS; ++k) out[k] = __builtin_bit_cast(vec_t, words[k]);
}

}  // namespace kvc
