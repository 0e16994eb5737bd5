// SPDX-License-Identifier: Apache-2.0
/**
 * @file   quantize_device.h
 * @brief  The Q8_K activation quantizer of one wavefront (one 256-value
 *         super-block) and the Q8_0 quantizer of eight lanes (one 32-value
 *         block), shared by the quantizer kernels and by kernels that quantize
 *         rows as part of another launch.
 *
 * Bit-exact with the reference CPU quantizers in an x86 AVX2 GCC build
 * (IMPL = nntrainer/tensor/cpu_backend/ggml_interface/nntr_ggml_impl):
 *   Q8_0 IMPL/nntr_ggml_impl_quant.cpp:613-701 and the per-row content of
 *        IMPL/nntr_ggml_impl.cpp:7879-7980
 *   ROW  IMPL/nntr_ggml_impl_quant.cpp:1334-1374, where the compiler fuses
 *        iscale*x + 1.5*2^23 into a single rounding
 *   MAT  IMPL/nntr_ggml_impl.cpp:7504-7737 (product rounded to fp32, then to
 *        the nearest-even integer; scale negative iff some x == +amax)
 */
#ifndef HIPQ_QUANTIZE_DEVICE_H
#define HIPQ_QUANTIZE_DEVICE_H
#include "hipq_internal.h"

static constexpr float kRoundMagic = 12582912.f; /* 1.5 * 2^23 */

__device__ __forceinline__ int magic_to_int(float biased) {
  return (int)(__float_as_uint(biased) & 0x007fffffu) - 0x00400000;
}

__device__ __forceinline__ int pack4(int a, int b, int c, int d) {
  return (a & 0xff) | ((b & 0xff) << 8) | ((c & 0xff) << 16) | ((d & 0xff) << 24);
}

/* The 16-byte matrix operand of a 16-value group, from the four lanes of a quad that
 * hold its values 4i .. 4i+3 each (q[0..3] of lane i): the 8 even values first, then
 * the 8 odd ones. Every lane of the quad returns the whole operand. */
__device__ __forceinline__ uint4 hipq_quad_operand(const int (&q)[4]) {
  const int mine = (q[0] & 0xff) | ((q[2] & 0xff) << 8) | ((q[1] & 0xff) << 16) | ((q[3] & 0xff) << 24);
  const uint32_t d0 = (uint32_t)hipq_dpp_i<0x00>(mine), d1 = (uint32_t)hipq_dpp_i<0x55>(mine);
  const uint32_t d2 = (uint32_t)hipq_dpp_i<0xAA>(mine), d3 = (uint32_t)hipq_dpp_i<0xFF>(mine);
  return make_uint4((d0 & 0xffffu) | (d1 << 16), (d2 & 0xffffu) | (d3 << 16), (d0 >> 16) | (d1 & 0xffff0000u),
                    (d2 >> 16) | (d3 & 0xffff0000u));
}

/* Q8_0: the calling lane holds four consecutive values of a 32-value block, the
 * eight lanes of the block are consecutive. Returns the lane's four int8 values
 * packed; dh = the block's fp16 scale. */
__device__ __forceinline__ int hipq_quantize_q8_0_lane(const float4 &x, uint16_t &dh, int &qsum) {
  float amax = fmaxf(fmaxf(fabsf(x.x), fabsf(x.y)), fmaxf(fabsf(x.z), fabsf(x.w)));
  amax = hipq_group_max<8>(amax);
  const float d = __fdiv_rn(amax, 127.f);
  const float id = (amax != 0.0f) ? __fdiv_rn(127.f, amax) : 0.0f;
  const int q0 = (int)rintf(__fmul_rn(x.x, id));
  const int q1 = (int)rintf(__fmul_rn(x.y, id));
  const int q2 = (int)rintf(__fmul_rn(x.z, id));
  const int q3 = (int)rintf(__fmul_rn(x.w, id));
  dh = hipq_f2h(d);
  qsum = q0 + q1 + q2 + q3;
  return pack4(q0, q1, q2, q3);
}

/* The same with V (4, 8 or 16) consecutive values of the block in the calling lane, the 32 / V lanes of the block
 * consecutive: the bytes packed in q, the block's scale and sum. For one row quantized by a few wavefronts that wait
 * for it: what is per block (the reductions, the two divisions) is done by fewer lanes, and
 * no value depends on another's. Rounding by the add of 1.5 * 2^23 leaves the byte in the low bits, which two
 * permutes a dword gather. */
template <int V>
__device__ __forceinline__ void hipq_quantize_q8_0_values(const float4 (&x)[V / 4], uint32_t (&q)[V / 4], uint16_t &dh,
                                                          int &bsum) {
  float amax = 0.f;
#pragma unroll
  for (int i = 0; i < V / 4; ++i)
    amax = fmaxf(fmaxf(fmaxf(fabsf(x[i].x), fabsf(x[i].y)), fmaxf(fabsf(x[i].z), fabsf(x[i].w))), amax);
  amax = hipq_group_max<32 / V>(amax);
  const float id = amax != 0.0f ? __fdiv_rn(127.f, amax) : 0.0f;
  auto biased = [&](float v) { return __float_as_uint(__fadd_rn(__fmul_rn(v, id), kRoundMagic)); };
  int sum = 0;
#pragma unroll
  for (int i = 0; i < V / 4; ++i) {
    q[i] = __builtin_amdgcn_perm(biased(x[i].y), biased(x[i].x), 0x0c0c0400u) |
           __builtin_amdgcn_perm(biased(x[i].w), biased(x[i].z), 0x04000c0cu);
    sum = hipq_dot4((int)q[i], 0x01010101, sum);
  }
  bsum = hipq_group_sum_i<32 / V>(sum);
  uint32_t h = hipq_f2h(__fdiv_rn(amax, 127.f));
  asm volatile("" : "+v"(h)); /* here, beside the rest, and not behind the condition that stores it */
  dh = (uint16_t)h;
}

/* output forms of the Q8_K quantizer */
enum {
  Q8K_PLANES = 0,
  Q8K_CANONICAL = 1,
  Q8K_ROWMMA = 3,
  Q8K_DIGITS = 4, /* of the planes only what the Q4_K GEMV reads: ql, qh, bsum, d */
  Q8K_BYTES = 5   /* of the planes only what the Q6_K GEMV reads: q, d */
};

/* Super-block sb = (row m, block b) by the calling wavefront (all 64 lanes), lane l
 * holding its values 4l .. 4l+3 in xv. Rows below mat_rows take the 4-row
 * quantizer's semantics, the others the row quantizer's. d_stride: distance of
 * consecutive super-blocks' scales in d_out (the row form only). */
template <int MODE>
__device__ __forceinline__ void hipq_quantize_q8_K_values(
  const float4 &xv, int64_t m, int b, int64_t sb, int nsb, int64_t mat_rows, int8_t *__restrict__ q_out,
  float *__restrict__ d_out, int16_t *__restrict__ bsum_out, uint8_t *__restrict__ canon_out,
  uint16_t *__restrict__ amin_out, uint16_t *__restrict__ ql_out, uint16_t *__restrict__ qh_out,
  int d_stride = 1) {
  const int lane = threadIdx.x & 63;
  const float x[4] = {xv.x, xv.y, xv.z, xv.w};

  float amax = fmaxf(fmaxf(fabsf(x[0]), fabsf(x[1])), fmaxf(fabsf(x[2]), fabsf(x[3])));
  amax = hipq_wave_max(amax); /* the same value in every lane, without an exchange through LDS */

  int q[4];
  float d;
  if (amax == 0.0f) {
    q[0] = q[1] = q[2] = q[3] = 0;
    d = 0.f;
  } else if (m < mat_rows) {
    /* 4-row quantizer semantics */
    const bool hit = (x[0] == amax) | (x[1] == amax) | (x[2] == amax) | (x[3] == amax);
    const bool pos_hit = __ballot(hit) != 0ull;
    const float iscale = pos_hit ? __fdiv_rn(-127.f, amax) : __fdiv_rn(127.f, amax);
    d = __fdiv_rn(1.f, iscale);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int v = (int)rintf(__fmul_rn(x[i], iscale));
      q[i] = max(-128, min(127, v));
    }
  } else {
    /* row quantizer semantics: sign of the FIRST element of maximal magnitude */
    float cand = 0.f;
    bool has = false;
#pragma unroll
    for (int i = 3; i >= 0; --i)
      if (fabsf(x[i]) == amax) {
        cand = x[i];
        has = true;
      }
    const unsigned long long mask = __ballot(has);
    const int first = __ffsll((long long)mask) - 1;
    const float vmax = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, cand), first));
    const float iscale = __fdiv_rn(-127.f, vmax);
    d = __fdiv_rn(1.f, iscale);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      q[i] = min(127, magic_to_int(__fmaf_rn(iscale, x[i], kRoundMagic)));
  }

  const int packed = pack4(q[0], q[1], q[2], q[3]);
  int gsum = q[0] + q[1] + q[2] + q[3];
  gsum = hipq_group_sum_i<4>(gsum); /* 4 lanes = one 16-value group */

  if (MODE == Q8K_CANONICAL) {
    uint8_t *o = canon_out + sb * 292;
    if (lane == 0) *(float *)o = d;
    *(int *)(o + 4 + lane * 4) = packed;
    if ((lane & 3) == 0) *(int16_t *)(o + 260 + (lane >> 2) * 2) = (int16_t)gsum;
  } else if (MODE == Q8K_ROWMMA) {
    /* row-major, each 16-value group stored as its 8 even then its 8 odd values:
     * this lane's four values are elements 4l .. 4l+3 of group lane / 4 */
    const uint4 op = hipq_quad_operand(q);
    if ((lane & 3) == 0) *(uint4 *)(q_out + sb * 256 + (lane >> 2) * 16) = op;
    if (lane == 0) d_out[sb * d_stride] = d;
    const int bs = gsum + hipq_dpp_i<0x104>(gsum); /* row_shl:4: lane l takes lane l + 4; two 16-value groups = one sub-block (read in lanes 0 and 8 of a row) */
    if ((lane & 7) == 0) {
      const int l6 = bs & 63;
      amin_out[sb * 16 + (lane >> 3)] = __half_as_ushort(__float2half_rn((float)l6));
      amin_out[sb * 16 + 8 + (lane >> 3)] = __half_as_ushort(__float2half_rn((float)(bs - l6)));
    }
  } else {
    if (MODE != Q8K_DIGITS) *(int *)(q_out + sb * 256 + lane * 4) = packed;
    if (lane == 0) d_out[sb] = d;
    if (MODE != Q8K_BYTES) {
      if ((lane & 3) == 0) bsum_out[sb * 16 + (lane >> 2)] = (int16_t)gsum;
      /* 4-bit digits for the v_dot8_u32_u4 kernels: q = 16 * (qh - 8) + ql */
      uint32_t lo = 0, hi = 0;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        lo |= (uint32_t)(q[i] & 15) << (4 * i);
        hi |= (uint32_t)(((q[i] >> 4) + 8) & 15) << (4 * i);
      }
      ql_out[sb * 64 + lane] = (uint16_t)lo;
      qh_out[sb * 64 + lane] = (uint16_t)hi;
    }
  }
}

/* The row quantizer with sixteen consecutive values of the super-block in the calling lane, the super-block's sixteen
 * lanes consecutive, for one row quantized by a few wavefronts that wait for it: the reductions stay inside a row of
 * lanes, the two divisions serve four super-blocks a wavefront, and a 16-value group's sum needs no exchange. MODE
 * Q8K_DIGITS, Q8K_BYTES or Q8K_ROWMMA (the sums' fp16 parts then go to bsum_out); `at` is the lane's place in the row (values 16 at .. 16 at + 15), stored where `store`.
 *
 * The scale has the sign of the first value of largest magnitude: that of the largest value or of the smallest,
 * whichever is larger in magnitude, and only where both are the same has the first to be looked for. No value leaves
 * -127 .. 127 (|iscale x| <= 127 (1 + 2^-23)), so the low byte of the biased float is the value; where iscale is not
 * finite that byte is 0, as the plain form's is. */
template <int MODE>
__device__ __forceinline__ void hipq_quantize_q8_K_values16(const float4 (&x)[4], int at, bool store,
                                                            int8_t *__restrict__ q_out, float *__restrict__ d_out,
                                                            int16_t *__restrict__ bsum_out,
                                                            uint8_t *__restrict__ ql_out,
                                                            uint8_t *__restrict__ qh_out) {
  static_assert(MODE == Q8K_DIGITS || MODE == Q8K_BYTES || MODE == Q8K_ROWMMA, "the forms of one row's quantizer");
  const float v[16] = {x[0].x, x[0].y, x[0].z, x[0].w, x[1].x, x[1].y, x[1].z, x[1].w,
                       x[2].x, x[2].y, x[2].z, x[2].w, x[3].x, x[3].y, x[3].z, x[3].w};
  float hi = v[0], lo = v[0];
#pragma unroll
  for (int i = 1; i < 16; ++i) hi = fmaxf(hi, v[i]), lo = fminf(lo, v[i]);
  hi = hipq_group_max<16>(hi);
  lo = -hipq_group_max<16>(-lo);
  const float amax = fmaxf(fabsf(hi), fabsf(lo));
  float vmax = fabsf(hi) == amax ? hi : lo;
  if (__ballot(hi == -lo && amax != 0.f) != 0ull) {
    int key = 1 << 30; /* place of the first such value, twice, plus its sign */
#pragma unroll
    for (int i = 15; i >= 0; --i)
      if (fabsf(v[i]) == amax) key = (((int)(threadIdx.x & 15) * 16 + i) << 1) | (v[i] < 0.f ? 1 : 0);
    key = min(key, hipq_dpp_i<HIPQ_DPP_XOR1>(key));
    key = min(key, hipq_dpp_i<HIPQ_DPP_XOR2>(key));
    key = min(key, hipq_dpp_i<HIPQ_DPP_HALF_MIRROR>(key));
    key = min(key, hipq_dpp_i<HIPQ_DPP_MIRROR>(key));
    vmax = (key & 1) ? -amax : amax;
  }
  const float iscale = amax != 0.f ? __fdiv_rn(-127.f, vmax) : 0.f;
  uint32_t p[4];
  int sum = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    auto biased = [&](int j) { return __float_as_uint(__fmaf_rn(iscale, v[4 * i + j], kRoundMagic)); };
    p[i] = __builtin_amdgcn_perm(biased(1), biased(0), 0x0c0c0400u) | __builtin_amdgcn_perm(biased(3), biased(2), 0x04000c0cu);
    sum = hipq_dot4((int)p[i], 0x01010101, sum);
  }
  float d = amax != 0.f ? __fdiv_rn(1.f, iscale) : 0.f;
  asm volatile("" : "+v"(d)); /* here, beside the rest, and not behind the condition that stores it */
  if (MODE == Q8K_BYTES) {
    if (store) *(uint4 *)(q_out + 16 * at) = make_uint4(p[0], p[1], p[2], p[3]);
  } else if (MODE == Q8K_ROWMMA) {
    /* the group's 8 even values, then its 8 odd ones; two lanes are a sub-block */
    const int bs = sum + hipq_dpp_i<HIPQ_DPP_XOR1>(sum);
    if (store) {
      *(uint4 *)(q_out + (int64_t)16 * at) =
        make_uint4(__builtin_amdgcn_perm(p[1], p[0], 0x06040200u), __builtin_amdgcn_perm(p[3], p[2], 0x06040200u),
                   __builtin_amdgcn_perm(p[1], p[0], 0x07050301u), __builtin_amdgcn_perm(p[3], p[2], 0x07050301u));
      if ((at & 1) == 0) {
        const int l6 = bs & 63;
        uint16_t *amin = (uint16_t *)bsum_out + (at & ~15) + ((at & 15) >> 1);
        amin[0] = __half_as_ushort(__float2half_rn((float)l6));
        amin[8] = __half_as_ushort(__float2half_rn((float)(bs - l6)));
      }
    }
  } else {
    /* 4-bit digits, q = 16 * (qh - 8) + ql, eight values a dword in order */
    auto gather = [](uint32_t a, uint32_t b) { /* the nibbles of eight bytes 0x0n */
      return __builtin_amdgcn_perm(b | (b >> 4), a | (a >> 4), 0x06040200u);
    };
    uint32_t l[4], h[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) l[i] = p[i] & 0x0f0f0f0fu, h[i] = ((p[i] >> 4) & 0x0f0f0f0fu) ^ 0x08080808u;
    if (store) {
      *(uint2 *)(ql_out + 8 * at) = make_uint2(gather(l[0], l[1]), gather(l[2], l[3]));
      *(uint2 *)(qh_out + 8 * at) = make_uint2(gather(h[0], h[1]), gather(h[2], h[3]));
      bsum_out[at] = (int16_t)sum;
    }
  }
  if (store && (at & 15) == 0) d_out[at >> 4] = d;
}

/* The same with the values read from row m of A (rows M and beyond read as zeros). */
template <int MODE>
__device__ __forceinline__ void hipq_quantize_q8_K_wave(
  const float *__restrict__ A, int64_t M, int64_t sb, int nsb, int64_t lda, int64_t mat_rows,
  int8_t *__restrict__ q_out, float *__restrict__ d_out, int16_t *__restrict__ bsum_out,
  uint8_t *__restrict__ canon_out, uint16_t *__restrict__ amin_out, uint16_t *__restrict__ ql_out,
  uint16_t *__restrict__ qh_out) {
  const int lane = threadIdx.x & 63;
  const int64_t m = sb / nsb;
  const int b = (int)(sb - m * nsb);
  float4 xv = make_float4(0.f, 0.f, 0.f, 0.f);
  if (m < M) xv = *(const float4 *)(A + m * lda + (int64_t)b * 256 + lane * 4);
  hipq_quantize_q8_K_values<MODE>(xv, m, b, sb, nsb, mat_rows, q_out, d_out, bsum_out, canon_out, amin_out,
                                  ql_out, qh_out);
}

#endif /* HIPQ_QUANTIZE_DEVICE_H */
