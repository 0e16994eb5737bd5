// SPDX-License-Identifier: Apache-2.0
/**
 * @file   moe_tile_device.h
 * @brief  Q4_K expert products of many tokens: a workgroup's tile of 32 or 64
 *         gathered activation rows against 32 weight columns a wavefront.
 *
 * With dozens of tokens per expert the expert products are GEMMs and the vector
 * instructions per matrix step set their time. The kernels for a few tokens scale every
 * sub-block's sums on the vector ALU (a multiply-add per sum and 32-deep step: 290 vector
 * instructions per 32 x 32 x 256 of product); here the 6-bit scale goes into the weights,
 * split as sc = 8 hi + lo: both digit planes q4 * lo and q4 * hi (<= 105) are int8, two
 * chains of v_mfma_i32_32x32x32_i8 accumulate over the whole super-block and
 * I = Dlo + 8 Dhi is the exact integer the few-token kernels form. The fp32 chains behind it
 * are theirs (and the single-row product's), acc = fma(float(I), d * dA, acc) and
 * accm = fma(float(Im), dmin * dA, accm), so the outputs keep those bits. The expansion of the
 * weights is shared by the two row tiles of 32: 135 vector instructions per 32 x 32 x 256.
 *
 * Rows go from the quantized planes straight to one of two LDS buffers, a super-block ahead, with
 * buffer_load ... lds: sixteen lanes fetch the 256 consecutive bytes of a row (four rows an
 * instruction, whole cache lines), wherever the row lies, so nothing is gathered or copied
 * beforehand. What the mins' pass reads arrives during the products too: the row sums in LDS of their own (of the first eight
 * super-blocks), the headers in the row buffer that the last super-block leaves free. With the sums copied when they were due and one
 * header under way, the pass was a chain of L2 latencies, and a workgroup has three to twelve super-blocks in all. 1000 tokens
 * of 128 experts of 2048 x 768, top 8, traced, medians of 400 launches: gate/up 110 -> 98 us, with the activation evaluated four values
 * at a time and the outputs stored without conditions, down 67 -> 57. What is beyond eight super-blocks of a row is
 * copied when it is due, as all of it was: blocks of 2304 to 3072 hidden or intermediate columns take 2 to 14 % less all the same. A row's sixteen
 * 16-byte pieces are stored rotated by an exclusive-or with its number
 * (the lane asks for piece slot ^ row), which spreads the 128-bit reads of eight neighbouring rows
 * over all banks. Weights stream through registers from the expert tiles (hipq_internal.h), a
 * super-block ahead.
 */
#ifndef HIPQ_MOE_TILE_DEVICE_H
#define HIPQ_MOE_TILE_DEVICE_H
#include <type_traits>

#include "gemv_device.h"

namespace moe_tile {

typedef int v2i __attribute__((ext_vector_type(2)));
typedef int v3i __attribute__((ext_vector_type(3)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef __amdgpu_buffer_rsrc_t rsrc_t;

constexpr int ROWS = 64; /* rows of a work item, at most */

constexpr int MINS_SB = 8; /* super-blocks whose row sums are in LDS at once in the mins' pass */
struct MinsLds {
  uint8_t amin[MINS_SB][ROWS * 32]; /* [row][8 low parts, 8 high parts of the sub-block sums, fp16] */
  float dA[MINS_SB][ROWS];
};
struct Lds {
  int8_t q[2][ROWS * 256]; /* per buffer [row][16 pieces of 16 bytes, piece p of row r at place p ^ (r & 15)] */
  float dA[2][ROWS];
  int rows[ROWS]; /* where the item's rows lie in the activation planes */
  MinsLds m;
};
static_assert((sizeof(Lds) + 512) * 3 <= 158 * 1024, "three workgroups per CU must fit the 160 KB LDS");

__device__ __forceinline__ int out_row(int tm, int r, int lane) { return 32 * tm + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3); }

/* The wavefront's column tile (its first byte is tile[0]) over the whole of K for the item's 32 * TM rows. rows() fills l.rows (valid
 * plane rows, all of them), kept() may put into LDS what was asked for there, and done(acc, accm, free) receives the sums:
 * acc[tm][r] - accm[tm][r] is row out_row(tm, r, lane), column lane & 31. It may use 4 KB of LDS a wavefront from free on. */
template <int TM, typename Rows, typename Kept, typename Done>
__device__ __forceinline__ void run(Lds &l, const QView &a, uint32_t a_rows, const uint8_t *tile, Rows rows, Kept kept, Done done) {
  const int K = a.K, nsb = K >> 8;
  const int lane = threadIdx.x & 63, i32 = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const v16i zero16 = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
  const v16f zero16f = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};

  const uint32_t tile_bytes = (uint32_t)nsb * hipq::EXPERT_TILE_BYTES;
  const rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void *)tile, 0, (int)tile_bytes, 0x00020000);
  auto load_q = [&](int sb, int i) {
    return __builtin_bit_cast(
      v4i, __builtin_amdgcn_raw_buffer_load_b128(rw, lane * 16, sb * hipq::EXPERT_TILE_BYTES + i * 1024, 0));
  };
  auto load_hd = [&](int sb) {
    return __builtin_bit_cast(
      v3i, __builtin_amdgcn_raw_buffer_load_b96(rw, 4096 + i32 * 16, sb * hipq::EXPERT_TILE_BYTES, 0));
  };
  v4i W[4];
  v3i hd; /* the scales; the mins' pass reads the whole header */
  /* the weights are asked for before the rows are known */
#pragma unroll
  for (int i = 0; i < 4; ++i) W[i] = load_q(0, i);
  hd = load_hd(0);
  rows();
  __syncthreads();

  const rsrc_t rq = __builtin_amdgcn_make_buffer_rsrc((void *)a.q, 0, (int)(a_rows * (uint32_t)K), 0x00020000);
  const rsrc_t rm = __builtin_amdgcn_make_buffer_rsrc((void *)a.bsum, 0, (int)(a_rows * (uint32_t)nsb * 32), 0x00020000);
  const rsrc_t rd = __builtin_amdgcn_make_buffer_rsrc((void *)a.d, 0, (int)(a_rows * (uint32_t)nsb * 4), 0x00020000);
  auto lds_ptr = [](void *p) { return (__attribute__((address_space(3))) void *)p; };
  /* this lane's places: copy i of the wavefront moves rows 4 (2 TM wave + i) .. + 3 */
  uint32_t vq[2 * TM];
#pragma unroll
  for (int i = 0; i < 2 * TM; ++i) {
    const int r = 4 * (wave * 2 * TM + i) + (lane >> 4);
    vq[i] = (uint32_t)l.rows[r] * (uint32_t)K + (uint32_t)(((lane & 15) ^ (r & 15)) * 16);
  }
  const uint32_t vd = (uint32_t)l.rows[lane & (32 * TM - 1)] * (uint32_t)(nsb * 4); /* row lane's scale */
  auto copy_rows = [&](int sb, int buf) {
#pragma unroll
    for (int i = 0; i < 2 * TM; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rq, lds_ptr(l.q[buf] + (wave * 2 * TM + i) * 1024), 16, (int)vq[i], sb * 256,
                                               0, 0);
    if (wave == 0) __builtin_amdgcn_raw_ptr_buffer_load_lds(rd, lds_ptr(l.dA[buf]), 4, (int)vd, sb * 4, 0, 0);
  };
  /* row sums and scales of the super-blocks m0 .. of the mins' pass */
  const uint32_t vm = (uint32_t)l.rows[(32 * (wave & 1) + (lane >> 1)) & (32 * TM - 1)] * (uint32_t)(nsb * 32) + (lane & 1) * 16;
  auto copy_mins = [&](int m0, int mn) {
    for (int k = wave; k < TM * mn; k += 4) { /* 32 rows of a super-block; k % TM is wave % TM, as in vm */
      const int b = k / TM, part = k % TM;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rm, lds_ptr(l.m.amin[b] + part * 1024), 16, (int)vm, (m0 + b) * 32, 0, 0);
    }
    for (int b = wave; b < mn; b += 4)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rd, lds_ptr(l.m.dA[b]), 4, (int)vd, (m0 + b) * 4, 0, 0);
  };
  /* headers of the super-blocks m0 .. of the mins' pass, [super-block][column] in the wavefront's 4 KB of a row buffer */
  auto copy_headers = [&](int buf, int m0) {
#pragma unroll
    for (int b = 0; b < MINS_SB; b += 2) /* two of 32 columns an instruction; past the end the last one again: a fixed number of loads in flight */
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, lds_ptr(l.q[buf] + wave * 4096 + b * 512), 16,
                                               4096 + (lane & 31) * 16 + min(m0 + b + (lane >> 5), nsb - 1) * (int)hipq::EXPERT_TILE_BYTES,
                                               0, 0, 0);
  };

  /* LDS byte of this lane's operand of step j: row i32, piece 2 j + g */
  const uint32_t abase = (uint32_t)(i32 * 256 + ((g ^ (i32 & 15)) << 4));
  uint32_t m4 = HIPQ_M4;
  asm("" : "+v"(m4)); /* an operand in a scalar register halves an instruction's rate */
  float acc[TM][16];

  /* One super-block: the rows of the next are asked for first; a quarter of the nibbles is asked for
   * again (for the next super-block) as soon as its two steps have taken it, so one set of registers holds
   * the stream and most of a super-block's time covers every load. */
  auto super_block = [&](int sb, auto last) {
    constexpr bool LAST = decltype(last)::value;
    const int buf = sb & 1;
    if (LAST)
      copy_headers(buf ^ 1, 0);
    else
      copy_rows(sb + 1, buf ^ 1);
    const int8_t *pq = l.q[0] + buf * (ROWS * 256);
    HipqDigits dg;
    const float dw = hipq_h2f((uint16_t)((uint32_t)hd[0] & 0xffff));
    v16i Dlo[TM], Dhi[TM];
    v4i av[2][TM]; /* the rows of a step are read a step ahead: a block of 1000 tokens 0.4 % less */
    auto read_a = [&](int j) {
      uint32_t at = abase;
      asm("" : "+v"(at)); /* one instruction a step instead of eight registers */
#pragma unroll
      for (int tm = 0; tm < TM; ++tm) av[j & 1][tm] = *(const v4i *)(pq + (at ^ (j * 32)) + tm * 8192);
    };
    read_a(0);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (j + 1 < 8) read_a(j + 1);
      if (j % 4 == 0) dg = hipq_digits((uint32_t)hd[1 + j / 4]);
      const uint32_t x0 = (uint32_t)W[j >> 1][2 * (j & 1)], x1 = (uint32_t)W[j >> 1][2 * (j & 1) + 1];
      const uint32_t e0 = x0 & m4, e1 = x1 & m4, o0 = (x0 >> 4) & m4, o1 = (x1 >> 4) & m4;
      const v4i bl = {hipq_scale4(e0, dg.lo, j & 3), hipq_scale4(e1, dg.lo, j & 3), hipq_scale4(o0, dg.lo, j & 3),
                      hipq_scale4(o1, dg.lo, j & 3)};
      const v4i bh = {hipq_scale4(e0, dg.hi, j & 3), hipq_scale4(e1, dg.hi, j & 3), hipq_scale4(o0, dg.hi, j & 3),
                      hipq_scale4(o1, dg.hi, j & 3)};
#pragma unroll
      for (int tm = 0; tm < TM; ++tm) {
        Dlo[tm] = __builtin_amdgcn_mfma_i32_32x32x32_i8(av[j & 1][tm], bl, j == 0 ? zero16 : Dlo[tm], 0, 0, 0);
        Dhi[tm] = __builtin_amdgcn_mfma_i32_32x32x32_i8(av[j & 1][tm], bh, j == 0 ? zero16 : Dhi[tm], 0, 0, 0);
      }
      if (!LAST && (j & 1)) W[j >> 1] = load_q(sb + 1, j >> 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (!LAST) hd = load_hd(sb + 1);
#pragma unroll
    for (int tm = 0; tm < TM; ++tm) {
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        const v4i dv = *(const v4i *)((const int8_t *)l.dA[0] + buf * (ROWS * 4) + (32 * tm + 8 * q4 + 4 * g) * 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int r = 4 * q4 + e;
          acc[tm][r] = fmaf((float)((Dhi[tm][r] << 3) + Dlo[tm][r]), dw * __int_as_float(dv[e]), acc[tm][r]);
        }
      }
      /* keeps the arithmetic of a row tile here: sunk past the barrier its operands would all stay live */
#pragma unroll
      for (int r = 0; r < 16; ++r) asm volatile("" : "+v"(acc[tm][r]));
      __builtin_amdgcn_sched_barrier(0);
    }
    /* the rows copied above have arrived (they were issued before the five weight loads, which stay in flight) */
    if (!LAST) asm volatile("s_waitcnt vmcnt(5) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };

  copy_rows(0, 0);
  kept();
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  copy_mins(0, min(MINS_SB, nsb)); /* they arrive during the products */
#pragma unroll
  for (int tm = 0; tm < TM; ++tm)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[tm][r] = 0.f;
  for (int sb = 0; sb + 1 < nsb; ++sb) super_block(sb, std::false_type{});
  super_block(nsb - 1, std::true_type{});

  /* the mins: accm = fma(Im, dmin * dA, accm) over the super-blocks, in a pass of its own so that its
   * chains do not occupy registers during the products */
  const int hbuf = nsb & 1; /* the row buffer that the last super-block left free */
  float accm[TM][16];
#pragma unroll
  for (int tm = 0; tm < TM; ++tm)
#pragma unroll
    for (int r = 0; r < 16; ++r) accm[tm][r] = 0.f;
  for (int m0 = 0; m0 < nsb; m0 += MINS_SB) {
    const int mn = min(MINS_SB, nsb - m0);
    if (m0) {
      __syncthreads(); /* the sums in LDS have been read */
      copy_mins(m0, mn);
      copy_headers(hbuf, m0);
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    for (int b = 0; b < mn; ++b) {
      const v4i hm = *(const v4i *)(l.q[hbuf] + wave * 4096 + b * 512 + i32 * 16);
      const float dmin = hipq_h2f((uint16_t)((uint32_t)hm[0] >> 16));
      const v8h bmin = hipq_mins8((uint32_t)hm[1], (uint32_t)hm[2], (uint32_t)hm[3]);
#pragma unroll
      for (int tm = 0; tm < TM; ++tm) {
        const v8h amin = __builtin_bit_cast(v8h, *(const v4i *)(l.m.amin[b] + (32 * tm + i32) * 32 + g * 16));
        const v16f Sm = __builtin_amdgcn_mfma_f32_32x32x16_f16(amin, bmin, zero16f, 0, 0, 0);
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
          const v4i dv = *(const v4i *)((const int8_t *)l.m.dA[b] + (32 * tm + 8 * q4 + 4 * g) * 4);
#pragma unroll
          for (int e = 0; e < 4; ++e)
            accm[tm][4 * q4 + e] = fmaf(Sm[4 * q4 + e], dmin * __int_as_float(dv[e]), accm[tm][4 * q4 + e]);
        }
      }
    }
  }
  done(acc, accm, l.q[hbuf]);
}

} // namespace moe_tile

#endif /* HIPQ_MOE_TILE_DEVICE_H */
