/* SPDX-License-Identifier: Apache-2.0 */
/**
 * @file   q6k_device.h
 * @brief  Q6_K weights times their scales as two int8 planes, for the matrix-core kernels (gemm_q6k.hip, gemm_rows_q6k.hip).
 */
#ifndef HIPQ_Q6K_DEVICE_H
#define HIPQ_Q6K_DEVICE_H

#include "gemv_device.h"

typedef uint16_t hipq_v2us __attribute__((ext_vector_type(2)));

/* a * b + c in both 16-bit lanes: one v_pk_mad_u16, as an expression, so that the compiler knows of its hazards with matrix
 * instructions under way (as inline assembly it was given registers that a matrix step had still to write). */
__device__ __forceinline__ uint32_t hipq_pk_mad(uint32_t a, uint32_t b, uint32_t c) {
  return __builtin_bit_cast(uint32_t, __builtin_bit_cast(hipq_v2us, a) * __builtin_bit_cast(hipq_v2us, b) +
                                        __builtin_bit_cast(hipq_v2us, c));
}

struct hipq_q6k_planes { /* weights 0 2 4 6 | 8 10 12 14 | 1 3 5 7 | 9 11 13 15 of a step */
  uint32_t l[4], h[4];
};

/* Four 6-bit weights u, one per byte of x, times the step's scale s. In 16-bit lanes
 *     t = u * 4s + (128 - 128 s) = 4 (u - 32) s + 128,     |4 (u - 32) s| <= 16256,
 * so that 4 (u - 32) s = 256 * hi(t) + (lo(t) - 128) with hi the signed high byte of t and
 * lo(t) - 128 = lo(t) ^ 0x80 a signed byte: both operand bytes come out of t by byte
 * selection, no shifts or masks. The two planes then hold four times the product; the
 * factor leaves with the column scale. */
__device__ __forceinline__ void hipq_scale_split(uint32_t x, uint32_t s2, uint32_t c2, uint32_t &l, uint32_t &h) {
  const uint32_t ta = hipq_pk_mad(__builtin_amdgcn_perm(x, x, 0x0c020c00u), s2, c2); /* bytes 0 and 2 */
  const uint32_t tb = hipq_pk_mad(__builtin_amdgcn_perm(x, x, 0x0c030c01u), s2, c2); /* bytes 1 and 3 */
  l = __builtin_amdgcn_perm(tb, ta, 0x06020400u) ^ 0x80808080u; /* low bytes: a0 b0 a1 b1 */
  h = __builtin_amdgcn_perm(tb, ta, 0x07030501u);               /* high bytes */
}

/* A step of sixteen weights: x0, x1 their low nibbles, hb their high bits, in the order of the tile copy (hipq_internal.h),
 * sc the step's scale. */
__device__ __forceinline__ hipq_q6k_planes hipq_q6k_expand(uint32_t x0, uint32_t x1, uint32_t hb, int sc) {
  /* four times the scale, sign-extended, in both 16-bit lanes; c2 = 128 - 128 * scale */
  const int s = sc << 2;
  const uint32_t s2 = __builtin_amdgcn_perm((uint32_t)s, (uint32_t)s, 0x05040100u);
  uint32_t c2 = hipq_pk_mad(s2, 0xffe0ffe0u, 0x00800080u);
  asm("" : "+v"(c2)); /* no instruction: u * s2 + c2 is not taken apart into (u - 32) * s2 + 128, a subtraction more */
  /* 6-bit weights, one per byte: the even ones (0, 2 .. 14), then the odd ones */
  const uint32_t e0 = (x0 & HIPQ_M4) | ((hb << 4) & 0x30303030u), e1 = (x1 & HIPQ_M4) | ((hb << 2) & 0x30303030u);
  const uint32_t o0 = ((x0 >> 4) & HIPQ_M4) | (hb & 0x30303030u), o1 = ((x1 >> 4) & HIPQ_M4) | ((hb >> 2) & 0x30303030u);
  hipq_q6k_planes p;
  hipq_scale_split(e0, s2, c2, p.l[0], p.h[0]);
  hipq_scale_split(e1, s2, c2, p.l[1], p.h[1]);
  hipq_scale_split(o0, s2, c2, p.l[2], p.h[2]);
  hipq_scale_split(o1, s2, c2, p.l[3], p.h[3]);
  return p;
}

#endif
