// SPDX-License-Identifier: Apache-2.0
/**
 * @file   gemm_rows_q6k.hip
 * @brief  Q6_K x Q8_K for a few activation rows (passes of eight side by side in one launch) on the int8 matrix cores,
 *         with the reference's bits.
 *
 * The reference multiplies every row on its own (ggml_interface_mixed.cpp:776-821 in the reference checkout), and its
 * row product keeps eight fp32 sums: sum l takes, super-block after super-block, the values whose place in their block of
 * 32 is 4 l .. 4 l + 3 (gemv_device.h). Those are 32 values of a super-block: exactly one v_mfma_i32_32x32x32_i8, if its 32
 * steps of K are the l-th four values of the eight blocks. So a super-block is eight matrix steps, one for each sum, twice
 * (the scaled weights are two int8 planes as in gemm_q6k.hip, whose tile copy this kernel reads: a lane has half of a
 * super-block's blocks of its column, and its operand of sum l is the l-th dword of each). The rows are staged so that a
 * lane's operand of a sum is one 128-bit read.
 *
 * A workgroup owns 32 columns and the eight rows of its pass (blockIdx.y); its four wavefronts take a super-block each per
 * round and leave the eight exact sums of every output in LDS, and after a barrier every thread runs the eight chains of one
 * output over the round's super-blocks, ascending, as the few-rows kernel of Q4_K does. Bound by the expansion's vector
 * instructions (430 a super-block and wavefront) and a round's latency; what it takes against the GEMV engine stands at gemm_rows_q6k_fits.
 */
#include "hipq_internal.h"
#include "q6k_device.h"
#include <algorithm>

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef __amdgpu_buffer_rsrc_t rsrc_t;

constexpr int TC = 8;   /* activation rows a workgroup holds */
constexpr int SBR = 4;  /* super-blocks a round = wavefronts a workgroup */
constexpr int NT = 64 * SBR;
constexpr int NREG = 4; /* result registers of a matrix step that carry them */

constexpr int QROW = SBR * 256 + 16; /* a staged row, padded so that the lanes of a 128-bit read fall into different banks */
constexpr int ACT_BYTES = TC * QROW;
constexpr int LDS_DA = 2 * ACT_BYTES; /* the rows' scales, four rounds of them */
constexpr int LDS_REC = (LDS_DA + 4 * SBR * TC * 4 + 255) / 256 * 256; /* [wavefront][register][sums 0-3 | 4-7][lane][4] */
constexpr int LDS_DW = LDS_REC + SBR * NREG * 2 * 256 * 4;
constexpr int LDS_BYTES = LDS_DW + SBR * 32 * 4;
static_assert(ACT_BYTES % 16 == 0 && 3 * LDS_BYTES <= 160 * 1024, "three workgroups a CU");

struct Regs { /* a lane's half of a super-block: steps s = 0 .. 7 of sixteen weights, blocks s / 2 of its half */
  v4i q[4], h[2], hd;
};

template <bool HOST>
__global__ __launch_bounds__(NT, 2) void gemm_rows_q6k_kernel(WView w, QView a, int M_all, float *__restrict__ C, int64_t ldc,
                                                              hipq::HostDone hd) {
  extern __shared__ __attribute__((aligned(16))) unsigned char rows_lds[];
  if (HOST) asm volatile("" ::"s"(w.qs), "s"(w.qh), "s"(w.hdr), "s"(w.N), "s"(w.K), "s"(a.q), "s"(a.d), "s"(M_all), "s"(C), "s"(ldc), "s"(hd.word));
  const int tile = blockIdx.x, K = w.K, nsb = K >> 8;
  const int r0 = blockIdx.y * TC, M = min(TC, M_all - r0);
  a.q += (size_t)r0 * K;
  a.d += (size_t)r0 * nsb;
  C += (int64_t)r0 * ldc;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int lane = threadIdx.x & 63, i32 = lane & 31, g = lane >> 5;
  float *const lda_ = (float *)(rows_lds + LDS_DA);
  int *const lrec = (int *)(rows_lds + LDS_REC);
  float *const ldw = (float *)(rows_lds + LDS_DW);

  const rsrc_t rq = __builtin_amdgcn_make_buffer_rsrc((void *)(w.qs + (size_t)tile * (size_t)(nsb * 4096)), 0, nsb * 4096, 0x00020000);
  const rsrc_t rh = __builtin_amdgcn_make_buffer_rsrc((void *)(w.qh + (size_t)tile * (size_t)(nsb * 2048)), 0, nsb * 2048, 0x00020000);
  const rsrc_t rd = __builtin_amdgcn_make_buffer_rsrc((void *)(w.hdr + (size_t)tile * (size_t)(nsb * 1024)), 0, nsb * 1024, 0x00020000);
  auto load = [&](Regs &r, int sb) {
    sb = min(sb, nsb - 1); /* uniform; a wavefront past the end loads the last super-block and does not use it */
#pragma unroll
    for (int i = 0; i < 4; ++i)
      r.q[i] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rq, lane * 16, sb * 4096 + i * 1024, 2));
#pragma unroll
    for (int i = 0; i < 2; ++i)
      r.h[i] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rh, lane * 16, sb * 2048 + i * 1024, 2));
    r.hd = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rd, lane * 16, sb * 1024, 2));
  };
  /* A round's share of the rows, through registers into one of two buffers; rows M .. 7 repeat row M - 1 and pieces past
   * the end of a row its last piece (never used) */
  struct ActRegs {
    v4i q[2];
    float dA;
  };
  auto act_load = [&](ActRegs &r, int rho) {
    const int t = threadIdx.x;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int c = t + u * NT;
      const int row = min(c / (16 * SBR), M - 1), off = min(rho * (SBR * 256) + c % (16 * SBR) * 16, K - 16);
      r.q[u] = *(const v4i *)(a.q + (size_t)row * K + off);
    }
    const int tt = t & (8 * SBR - 1), row = min(tt / SBR, M - 1);
    r.dA = a.d[(size_t)row * nsb + min(rho * SBR + tt % SBR, nsb - 1)];
  };
  /* [row][super-block][half g][sum l][block of the half]: a sixteen is half of a block, four sums' dwords */
  auto act_store = [&](const ActRegs &r, int rho) {
    unsigned char *base = rows_lds + (rho & 1) * ACT_BYTES;
    const int t = threadIdx.x;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int c = t + u * NT, p = c % (16 * SBR), s = p & 7;
      int *o = (int *)(base + c / (16 * SBR) * QROW + (p >> 4) * 256 + ((p >> 3) & 1) * 128 + (s & 1) * 64) + (s >> 1);
#pragma unroll
      for (int k = 0; k < 4; ++k) o[4 * k] = r.q[u][k];
    }
    if (t < 8 * SBR) lda_[(rho & 3) * (SBR * TC) + t % SBR * TC + t / SBR] = r.dA; /* [round][super-block][row] */
  };
  ActRegs AR;
  act_load(AR, 0);
  constexpr int NB = 2; /* the next round's weights are in flight during a round */
  Regs buf[NB];
  const int rounds = (nsb + SBR - 1) / SBR;
  load(buf[0], wave);
  act_store(AR, 0);
  __syncthreads();

  /* the output this thread chains: row cm, column cn; its sums sit in register cr of lane cl */
  const int cn = threadIdx.x & 31, cm = threadIdx.x >> 5;
  const int cr = cm & 3, cl = (cm >> 2) * 32 + cn;
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};

  auto round = [&](const Regs &W, int rho) {
    const int sb = rho * SBR + wave;
    if (sb < nsb) { /* uniform per wavefront */
      const v16i zero16 = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
      const unsigned char *pa = rows_lds + (rho & 1) * ACT_BYTES + (i32 & (TC - 1)) * QROW + wave * 256 + g * 128;
      int *rec = lrec + wave * (NREG * 2 * 256) + lane * 4;
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) { /* sums 4 hh .. 4 hh + 3: the first, the second sixteen of every block */
        v4i A[4], bl[4], bh[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) A[k] = *(const v4i *)(pa + (hh * 4 + k) * 16);
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          const int s = 2 * b + hh;
          const uint32_t x0 = (uint32_t)W.q[s >> 1][2 * (s & 1)], x1 = (uint32_t)W.q[s >> 1][2 * (s & 1) + 1];
          const uint32_t hb = (uint32_t)W.h[s >> 2][s & 3];
          const hipq_q6k_planes p = hipq_q6k_expand(x0, x1, hb, __builtin_amdgcn_sbfe(W.hd[s >> 2], 8 * (s & 3), 8));
          /* weights 4 k .. 4 k + 3 in order: the block's dword of sum 4 hh + k */
          bl[0][b] = (int)__builtin_amdgcn_perm(p.l[2], p.l[0], 0x05010400u), bl[1][b] = (int)__builtin_amdgcn_perm(p.l[2], p.l[0], 0x07030602u);
          bl[2][b] = (int)__builtin_amdgcn_perm(p.l[3], p.l[1], 0x05010400u), bl[3][b] = (int)__builtin_amdgcn_perm(p.l[3], p.l[1], 0x07030602u);
          bh[0][b] = (int)__builtin_amdgcn_perm(p.h[2], p.h[0], 0x05010400u), bh[1][b] = (int)__builtin_amdgcn_perm(p.h[2], p.h[0], 0x07030602u);
          bh[2][b] = (int)__builtin_amdgcn_perm(p.h[3], p.h[1], 0x05010400u), bh[3][b] = (int)__builtin_amdgcn_perm(p.h[3], p.h[1], 0x07030602u);
        }
        int S[4][NREG];
        v16i Dl[2], Dh[2];
#pragma unroll
        for (int k = 0; k <= 4; ++k) { /* a sum's results are read behind the next one's steps, not waited for */
          if (k < 4) {
            Dl[k & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(A[k], bl[k], zero16, 0, 0, 0);
            Dh[k & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(A[k], bh[k], zero16, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
          }
          if (k > 0) {
#pragma unroll
            for (int r = 0; r < NREG; ++r) /* the planes hold four times the product */
              S[k - 1][r] = ((Dh[(k - 1) & 1][r] << 8) + Dl[(k - 1) & 1][r]) >> 2;
          }
        }
#pragma unroll
        for (int r = 0; r < NREG; ++r) *(v4i *)(rec + (r * 2 + hh) * 256) = v4i{S[0][r], S[1][r], S[2][r], S[3][r]};
      }
      if (g == 0) ldw[wave * 32 + i32] = hipq_h2f((uint16_t)(W.hd[2] & 0xffff));
    }
    act_store(AR, rho + 1);
    __syncthreads();
    v4i iv[SBR][2];
    float sd[SBR];
#pragma unroll
    for (int ws = 0; ws < SBR; ++ws) {
      const int *rec = lrec + ws * (NREG * 2 * 256) + (cr * 2) * 256 + cl * 4;
      iv[ws][0] = *(const v4i *)rec;
      iv[ws][1] = *(const v4i *)(rec + 256);
      sd[ws] = lda_[(rho & 3) * (SBR * TC) + ws * TC + cm] * ldw[ws * 32 + cn];
    }
#pragma unroll
    for (int ws = 0; ws < SBR; ++ws)
      if (rho * SBR + ws < nsb) { /* uniform */
#pragma unroll
        for (int l = 0; l < 8; ++l) acc[l] = fmaf(sd[ws], (float)iv[ws][l >> 2][l & 3], acc[l]);
      }
    __syncthreads(); /* the next round overwrites the records */
  };
  for (int rho0 = 0; rho0 < rounds; rho0 += NB) {
#pragma unroll
    for (int u = 0; u < NB; ++u) {
      const int rho = rho0 + u;
      if (rho < rounds) {
        act_load(AR, rho + 1); /* before the weights: its wait must not include theirs */
        load(buf[(u + 1) % NB], (rho + 1) * SBR + wave);
        round(buf[u], rho);
      }
    }
  }
  const int col = tile * 32 + cn;
  const float sum = ((acc[0] + acc[4]) + (acc[2] + acc[6])) + ((acc[1] + acc[5]) + (acc[3] + acc[7]));
  if (HOST) {
    if (cm < M && col < w.N) hipq::store_out(C + (int64_t)cm * ldc + col, sum);
    hipq::host_done(hd);
  } else if (cm < M && col < w.N)
    C[(int64_t)cm * ldc + col] = sum;
}

} // namespace

namespace hipq {

/* Against the GEMV engine, whose passes of eight take 6 us and, a row of the weight, 0.42, 0.78 or 1.72 ns with up to two,
 * four or eight activation rows, or a weight 0.185, 0.215 and 0.71 ps (0.31 and 0.92 for the latter two beyond rows of 4096).
 * This kernel takes 6.8 us and a round of four super-blocks 2.05, or more where a CU has more than 0.75 workgroups. Over 315
 * sizes 28 % less than the engine alone, within 1 % of the faster one each time. us, engine / this kernel: eight rows of 1000 x
 * 4096 9.7 / 14.7, of 2000 x 2048 11.3 / 10.8, of 12288 x 512 28.1 / 9.7, of 20000 x 8192 128 / 51; four of 6000 x 4096 12.2 / 15.8,
 * of 12288 x 1024 15.8 / 10.3; two of 20000 x 512 14.9 / 10.8; sixteen of 600 x 1024 15.1 / 9.4, of 4000 x 4096 28.8 / 17.0. */
bool gemm_rows_q6k_fits(const hipq_weight *w, int64_t M) {
  if (w->dtype != HIPQ_Q6_K || w->expert_tiles || M < 2 || M > 16 || w->K % 256 || 16 * w->K > 0x7fffffff) return false;
  const double n = 1e-3 * (double)w->N, mw = 1e-6 * (double)w->N * (double)w->K;
  const bool chunks = w->K > 4096;
  auto pass = [&](int64_t rows) {
    return rows <= 2   ? std::max(0.42 * n, 0.185 * mw)
           : rows <= 4 ? std::max(0.78 * n, (chunks ? 0.31 : 0.215) * mw)
                       : std::max(1.72 * n, (chunks ? 0.92 : 0.71) * mw);
  };
  double engine = 1.;
  for (int64_t r0 = 0; r0 < M; r0 += 8) engine += 6. + pass(std::min<int64_t>(8, M - r0));
  const double a_cu = (double)((w->N + 31) / 32 * ((M + TC - 1) / TC)) / 256.;
  return 6.8 + (double)((w->K + 1023) / 1024) * std::max(2.05, 0.6 + 1.95 * a_cu) < engine;
}

int launch_gemm_rows_q6k(const hipq_weight *w, const QAct *qa, int M, float *C, int64_t ldc, hipStream_t s, HostEnd *end) {
  if (!w->gt_base || w->dtype != HIPQ_Q6_K || qa->K != w->K || M < 1 || M > 16)
    return fail(HIPQ_ERR_INVALID_ARGUMENT, "the few-rows Q6_K product takes 1 to 16 rows and a weight with its tile copy");
  WView v = wview(w);
  v.qs = w->gt_qs;
  v.qh = w->gt_qh;
  v.hdr = w->gt_hdr;
  const dim3 grid((unsigned)((w->N + 31) / 32), (unsigned)((M + TC - 1) / TC));
  const HostDone hd = take_end(end, grid);
  auto go = [&](const char *name, auto kernel) { launch_kernel(name, kernel, grid, dim3(NT), LDS_BYTES, s, v, qview(*qa), M, C, ldc, hd); };
  hd.word ? go("gemm_rows_q6k_kernel<true>", gemm_rows_q6k_kernel<true>) : go("gemm_rows_q6k_kernel<false>", gemm_rows_q6k_kernel<false>);
  HIPQ_HIP(hipGetLastError());
  return HIPQ_OK;
}

} // namespace hipq
