// SPDX-License-Identifier: Apache-2.0
/**
 * @file   gemv.hip
 * @brief  Decode GEMV kernels (M = 1, and 2..8 activation rows in one pass over
 *         the weights) for Q4_0, Q4_K and Q6_K weights on gfx950.
 *
 * Replaces the M == 1 branches of __ggml_q4_0_8x8_q8_0_GEMM,
 * __ggml_q4_K_8x8_q8_K_GEMM and __ggml_gemm_q6_K
 * (nntrainer/tensor/cpu_backend/ggml_interface/ggml_interface_omp.cpp:303-329,
 * 404-431, 519-535 in the reference checkout) and the gemv / vec_dot kernels
 * they call; outputs are bit-identical to those kernels (see gemv_device.h).
 *
 * Launch shape: 4 wavefronts a workgroup, each wavefront owns G consecutive output
 * columns, 16, 32 or 64 lanes a column (fused_form); rows of more weights than a chunk
 * are shared by the wavefronts of a workgroup (gemv_split_kernel). The kernel is bound by
 * HBM where the matrix is large: per output column it reads the column's packed weights
 * exactly once, 16 bytes per lane per load, all loads of a group in flight together; and
 * by the chain of what waits for what where it is small.
 */
#include <string>
#include <type_traits>

#include "gemv_device.h"
#include "quantize_device.h"

namespace {

template <int DT, int T, int R, int G, bool PW, int FK>
__global__ __launch_bounds__(256) void gemv_kernel(WView w, QView qa, int M, int pair_rows,
                                                   float *__restrict__ C, int64_t ldc) {
  extern __shared__ uint32_t gemv_lds[];
  const int wave = threadIdx.x >> 6;
  uint32_t *lds = gemv_lds + wave * GemvLds<DT, R, G, PW>::DWORDS;
  const int row0 = (blockIdx.x * 4 + wave) * G;
  int arow[R];
#pragma unroll
  for (int r = 0; r < R; ++r) arow[r] = r < M ? r : M - 1;
  const GemvOut o = gemv_engine<DT, T, R, G, PW, HIPQ_KCHUNK, FK>(w, row0, qa, arow, pair_rows, lds);
  if (o.valid && row0 + o.g < w.N && o.r < M) C[(int64_t)o.r * ldc + row0 + o.g] = o.v;
}

/* Decode GEMV on the fp32 activation row itself: the workgroup quantizes the row
 * into LDS (the arithmetic of the quantizer kernels, so the blocks are the same
 * bits) while its weight loads are in flight, and the engine reads the activations
 * from there. Saves the quantizer's launch, which costs more than the redundant
 * quantization as long as the matrix is small. One chunk only (K <= 4096).
 *
 * Up to some millions of weights a launch is bound by the chain of what waits for what: the arguments, the row,
 * its quantization, the barrier, the products, the fp32 sums in order. A launch of nothing takes 1.5 us of a
 * stream's time. So the row is quantized in one pass, four to sixteen values a lane, the arguments are
 * asked for together (args_first), the sums read their records a batch ahead (GemvCore::chain_batched; the records
 * are rounded up to whole batches), and every load is issued unconditionally whatever the row length: with the
 * number of a lane's steps a constant of the instance and the sums in batches at every length, Q4_K 8192 x 3584 8.2 ->
 * 5.4 us a call, 5120 x 2560 5.4 -> 4.7, 4096 x 4096 4.6 -> 4.0, 20000 x 768 6.5 -> 4.6, Q4_0 20000 x 800 6.3 -> 4.4, Q6_K 8192
 * x 3584 9.0 -> 6.8.
 */
template <int DT> __host__ __device__ constexpr int fused_act_bytes(int K) {
  /* Q8_0: q [K], meta [K/32] u32; Q8_K: q [K], ql [K/2], qh [K/2], bsum [K/16] i16, d [K/256] f32 */
  return ((DT == HIPQ_Q4_0 ? K + K / 8 : 2 * K + K / 8 + K / 64) + 15) & ~15;
}

/* The row of K values in the workgroup's lanes, V each from V * at on (lanes beyond K / V repeat the last), quantized into
 * LDS at ap: what the engine reads of it */
template <int DT, int V = 16>
__device__ __forceinline__ QView quantize_row_lds(const float4 (&xs)[4], int at, int K, uint8_t *ap) {
  const bool store = (int)threadIdx.x < K / V;
  QView qa;
  qa.K = K;
  qa.q = (const int8_t *)ap;
  if constexpr (DT == HIPQ_Q4_0) {
    int8_t *q = (int8_t *)ap;
    uint32_t *meta = (uint32_t *)(ap + K);
    qa.meta = meta;
    qa.d = nullptr;
    qa.bsum = nullptr;
    qa.ql = qa.qh = nullptr;
    uint32_t qv[V / 4];
    float4 xv[V / 4];
    uint16_t dh;
    int bsum;
#pragma unroll
    for (int p = 0; p < V / 4; ++p) xv[p] = xs[p];
    hipq_quantize_q8_0_values<V>(xv, qv, dh, bsum);
    if (store) {
      if constexpr (V == 4)
        *(uint32_t *)(q + at * V) = qv[0];
      else if constexpr (V == 8)
        *(uint2 *)(q + at * V) = make_uint2(qv[0], qv[1]);
      else
        *(uint4 *)(q + at * V) = make_uint4(qv[0], qv[1], qv[2], qv[3]);
      if (at % (32 / V) == 0) meta[at / (32 / V)] = (uint32_t)dh | ((uint32_t)(bsum & 0xffff) << 16);
    }
  } else {
    static_assert(V == 16, "a super-block in sixteen lanes");
    int8_t *q = (int8_t *)ap;
    uint8_t *ql = ap + K, *qh = ap + K + (K >> 1);
    int16_t *bsum = (int16_t *)(ap + 2 * K);
    float *d = (float *)(ap + 2 * K + (K >> 3));
    qa.meta = nullptr;
    qa.d = d;
    qa.bsum = bsum;
    qa.ql = ql;
    qa.qh = qh;
    hipq_quantize_q8_K_values16<DT == HIPQ_Q4_K ? Q8K_DIGITS : Q8K_BYTES>(xs, at, store, q, d, bsum, ql, qh);
  }
  return qa;
}

template <int DT, int T, int G, int NW, int FK, typename Store>
__device__ __forceinline__ void gemv_fused_rows(const WView (&wv)[NW], const float *__restrict__ x, int block,
                                                Store store) {
  typedef GemvCore<DT, T, 1, G, false, FK < 0 ? -FK : HIPQ_KCHUNK, (FK < 0)> E;
  const WView &w = wv[0];
  extern __shared__ __attribute__((aligned(16))) uint32_t gemv_lds[];
  /* FK: the row length where it is one of the usual ones, or less than zero the instance's capacity (with_length). Either
   * way the number of steps a lane takes is a constant, every load of the row and of the weights is issued
   * unconditionally, and the waits can count them: a load behind a condition makes every wait in front of it a wait for
   * nearly all loads in flight. Steps past the row's end read its last unit again; their records are not written. */
  const int K = FK > 0 ? FK : w.K;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  uint8_t *ap = (uint8_t *)gemv_lds;
  uint32_t *lds = gemv_lds + fused_act_bytes<DT>(K) / 4 + wave * GemvLds<DT, 1, G, false>::DWORDS;
  const int row0 = (block * 4 + wave) * G;
  const int arow[1] = {0};

  /* the row first (it comes from the cache), then the weights: the wait for the row
   * leaves the weight loads in flight. Positions beyond the row re-read its end. */
  /* V values a lane, K / V lanes. Q8_0: as few values as one pass of the workgroup's lanes allows; Q8_K: sixteen. */
  float4 xs[4];
  int at; /* the lane's place in the row */
  auto with_v = [&](auto f) {
    const int most = FK < 0 ? -FK : K; /* a constant */
    if (DT == HIPQ_Q4_0 && most <= 1024)
      f(std::integral_constant<int, DT == HIPQ_Q4_0 ? 4 : 16>{});
    else if (DT == HIPQ_Q4_0 && most <= 2048)
      f(std::integral_constant<int, DT == HIPQ_Q4_0 ? 8 : 16>{});
    else
      f(std::integral_constant<int, 16>{});
  };
  with_v([&](auto v) {
    constexpr int V = decltype(v)::value;
    at = min((int)threadIdx.x, K / V - 1);
#pragma unroll
    for (int p = 0; p < V / 4; ++p) xs[p] = *(const float4 *)(x + at * V + 4 * p);
  });
  /* Half of a wavefront's passes over the weight rows are asked for in front of the row's quantization, the other half
   * behind it; a single pass in front. The row's quantization wants its own loads back first and the weights' requests
   * out early, and a wavefront that issues all of them in front of it is late for the barrier the workgroup waits at
   * (us a call, in front / behind / half and half, four rows a wavefront: Q4_K 4096 x 4096 4.26 / 4.73 / 4.02, 8192 x 3072
   * 4.92 / 5.20 / 4.84, 12288 x 2048 5.11 / 4.89 / 4.98, sums over sizes of 3072 to 32000 rows of 2048 to 4096: Q4_K 172 / 171
   * / 162, Q4_0 81 / 81 / 79.5, Q6_K 112 / 110 / 101; rows of one pass, 1024 x 512 to 1536: 53.3 / 54.4 in front and behind). */
  typename E::Wts W[NW];
  constexpr int HP = E::NP > 1 ? E::NP / 2 : 1;
#pragma unroll
  for (int i = 0; i < NW; ++i) E::template load_w<0, HP>(W[i], wv[i], row0, 0, K);

  QView qa;
  with_v([&](auto v) { qa = quantize_row_lds<DT, decltype(v)::value>(xs, at, K, ap); });
#pragma unroll
  for (int i = 0; i < NW; ++i) E::template load_w<HP, E::NP>(W[i], wv[i], row0, 0, K);
  __syncthreads();

  typename E::Act A;
  E::load_act(A, qa, arow, 0, K);
  GemvOut o[NW];
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    typename E::Chain c = E::begin(arow, 0);
    E::compute(W[i], A, K, lds);
    if constexpr (FK < 0 || FK % (E::PADB * E::BLOCK) != 0) E::pad(K, lds, E::PER);
    hipq_wave_lds_sync();
    E::template chain<true>(c, K, lds);
    hipq_wave_lds_sync();
    o[i] = E::finish(c);
  }
  /* the results of the NW weights' row row0 + o[0].g sit in the same lane */
  if (o[0].valid && row0 + o[0].g < w.N) store(row0 + o[0].g, o);
}

/* Asks for all of a kernel's arguments at once. One that is loaded where it is first used (the weights' pointers
 * behind the row's, the output's at the end) adds a round trip of its own to a kernel that is nothing but a chain of
 * them. */
template <int DT> __device__ __forceinline__ void args_first(const void *x, const void *C, const WView &w) {
  const void *scale = DT == HIPQ_Q4_K ? (const void *)w.hdr : w.d;
  const void *qh = DT == HIPQ_Q6_K ? (const void *)w.qh : x, *sc = DT == HIPQ_Q6_K ? (const void *)w.sc : x;
  asm volatile("" ::"s"(x), "s"(C), "s"(w.qs), "s"(scale), "s"(qh), "s"(sc), "s"(w.N), "s"(w.K));
}

template <int DT, int T, int G, int FK>
__device__ __forceinline__ void gemv_fused_body(const WView &w, const float *__restrict__ x,
                                                float *__restrict__ C, int block) {
  const WView wv[1] = {w};
  gemv_fused_rows<DT, T, G, 1, FK>(wv, x, block, [&](int row, const GemvOut(&o)[1]) { C[row] = o[0].v; });
}

/* out[n] = silu(x . Wact[n]) * (x . Wmul[n]): the two projections of a gated MLP and the
 * SwiGLU between them and the down projection as one launch. A wavefront forms the same G
 * rows of both matrices (their loads in flight together) and the lane that ends up with
 * row n of the one also holds row n of the other. The activation is the framework's swiglu
 * (X = (Y / (1 + exp(-Y))) * Z in fp32, fallback_internal.cpp:417-423), applied by
 * SwiGLULayer::incremental_forwarding to the outputs of ffn_up (Y) and ffn_gate (Z)
 * (Applications/CausalLM/layers/swiglu.cpp:40-62, causal_lm.cpp:690-695). */
template <int DT, int T, int G, int FK>
__global__ __launch_bounds__(256) void gemv_fused_swiglu_kernel(WView wact, WView wmul,
                                                                const float *__restrict__ x,
                                                                float *__restrict__ out) {
  const WView wv[2] = {wact, wmul};
  args_first<DT>(x, out, wact);
  args_first<DT>(x, out, wmul);
  gemv_fused_rows<DT, T, G, 2, FK>(wv, x, (int)blockIdx.x, [&](int row, const GemvOut(&o)[2]) {
    out[row] = hipq_swiglu(o[0].v, o[1].v);
  });
}

template <int DT, int T, int G, int FK>
__global__ __launch_bounds__(256) void gemv_fused_kernel(WView w, const float *__restrict__ x,
                                                         float *__restrict__ C) {
  args_first<DT>(x, C, w);
  gemv_fused_body<DT, T, G, FK>(w, x, C, (int)blockIdx.x);
}
/* dwords of LDS between two rows' records of gemv_split_kernel: whole batches, and a gap against bank conflicts */
template <int DT> __host__ __device__ constexpr int split_stride(int K) {
  return DT == HIPQ_Q4_0 ? ((K / 32 + 7) & ~7) * 2 + 2 : DT == HIPQ_Q4_K ? ((K / 256 + 3) & ~3) * 4 + 4 : ((K / 256 + 7) & ~7) * 9 + 1;
}
/* One row of more weights than one step of 64 lanes takes (2048, Q6_K 4096): the wavefronts of a workgroup share its rows'
 * K. Wavefront c + nch * g takes part c of the G rows of group g, kc weights, with every load issued unconditionally as
 * in the kernels above; the parts' records lie one after the other in the workgroup's LDS, and behind a barrier the first
 * wavefront of a group forms the sums, in the reference's order over the whole row. A wavefront that walked a long row
 * in chunks of 4096 by itself, behind the quantizer's launch, waited for each chunk's loads and summed up its records in
 * between: Q4_K 4096 x 12288 12.9 -> 8.5 us a call, 5000 x 8192 11.5 -> 7.7, Q4_0 2560 x 9728 13.4 -> 9.0, Q6_K 4096 x 12288 13.2 ->
 * 11.4. FUSED: the row is
 * quantized by the workgroup, 16 values a lane (K <= 1024 * wavefronts); else it comes from the quantizer's planes. */
template <int DT, int G, bool FUSED>
__global__ __launch_bounds__(1024) void gemv_split_kernel(WView w, const float *__restrict__ x, QView qv, int nch, int kc,
                                                          float *__restrict__ C) {
  constexpr int STEP = 64 * GemvRec<DT, false>::UNIT;
  typedef GemvCore<DT, 64, 1, G, false, STEP, true> E;
  extern __shared__ __attribute__((aligned(16))) uint32_t gemv_lds[];
  args_first<DT>(FUSED ? (const void *)x : qv.q, C, w);
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
  const int grp = wave / nch, c = wave - grp * nch, groups = (int)(blockDim.x >> 6) / nch;
  const int K = w.K, k0 = c * kc, len = min(kc, K - k0);
  const int row0 = ((int)blockIdx.x * groups + grp) * G;
  uint8_t *ap = (uint8_t *)gemv_lds;
  const int stride = split_stride<DT>(K);
  uint32_t *rec = gemv_lds + (FUSED ? fused_act_bytes<DT>(K) / 4 : 0) + grp * (G * stride);
  const int arow[1] = {0};
  float4 xs[4];
  const int at = min((int)threadIdx.x, K / 16 - 1);
  typename E::Act A;
  typename E::Wts W;
  constexpr int HP = E::NP > 1 ? E::NP / 2 : 1;
  if constexpr (FUSED) {
#pragma unroll
    for (int p = 0; p < 4; ++p) xs[p] = *(const float4 *)(x + at * 16 + 4 * p);
    E::template load_w<0, HP>(W, w, row0, k0, len);
    const QView qa = quantize_row_lds<DT>(xs, at, K, ap);
    E::template load_w<HP, E::NP>(W, w, row0, k0, len);
    __syncthreads();
    E::load_act(A, qa, arow, k0, len);
  } else {
    E::load_act(A, qv, arow, k0, len);
    __builtin_amdgcn_sched_barrier(0);
    E::load_w(W, w, row0, k0, len);
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int pass = 0; pass < E::NP; ++pass)
    E::F::compute(W.W[pass], A, lane, len, rec + pass * stride + k0 / E::BLOCK * E::RECORD);
  if (c == 0) E::pad(K, rec, stride);
  __syncthreads();
  if (c) return; /* uniform per wavefront */
  typename E::Chain ch = E::begin(arow, 0);
  if (ch.on) E::template sums<true>(rec + ch.cg * stride, K, ch.l, ch.acc, ch.accm);
  const GemvOut o = E::finish(ch);
  if (o.valid && row0 + o.g < w.N) C[row0 + o.g] = o.v;
}

/* Up to four weights of one format and K on the same row, one launch: the
 * workgroups of weight i are blocks end[i-1] .. end[i]-1 of the grid. */
constexpr int FUSED_MAXW = 4;
struct FusedMulti {
  WView w[FUSED_MAXW];
  float *C[FUSED_MAXW];
  int end[FUSED_MAXW];
};
template <int DT, int T, int G, int FK>
__global__ __launch_bounds__(256) void gemv_fused_multi_kernel(FusedMulti mw, const float *__restrict__ x) {
  const int b = (int)blockIdx.x;
  int i = 0, first = 0;
#pragma unroll
  for (int k = 0; k + 1 < FUSED_MAXW; ++k)
    if (b >= mw.end[k]) i = k + 1, first = mw.end[k];
  gemv_fused_body<DT, T, G, FK>(mw.w[i], x, mw.C[i], b - first);
}

/* The name a launch is noted under, with the instance's template arguments as numbers (what a kernel trace
 * prints): built once per instance. */
template <int FAMILY, int... V> const char *kernel_name(const char *base) { /* FAMILY: one number a kernel template */
  static const std::string name = [&] {
    std::string n = std::string(base) + "<";
    const int v[] = {V...};
    for (size_t i = 0; i < sizeof(v) / sizeof(v[0]); ++i) n += (i ? ", " : "") + std::to_string(v[i]);
    (void)FAMILY;
    return n + ">";
  }();
  return name.c_str();
}

/* f(FK) as a compile-time constant. FK: one of the usual row lengths, or less than zero the capacity of the instance, the
 * next whole number of steps of its lanes. What the constants gain is small launches: Q4_K with two rows a wavefront 7 %,
 * with four rows from 8192 on nothing. */
template <int DT, int T, typename F> void with_length(int64_t K, F f) {
  constexpr int STEP = T * GemvRec<DT, false>::UNIT; /* weights of a row that the lanes take at once */
  constexpr int MOST = HIPQ_KCHUNK / STEP;
  if (T == 64 && K == 4096) return f(std::integral_constant<int, T == 64 ? 4096 : -STEP>{});
  if (T >= 32 && K == 3072) return f(std::integral_constant<int, T >= 32 ? 3072 : -STEP>{});
  if (T >= 32 && K == 2048) return f(std::integral_constant<int, T >= 32 ? 2048 : -STEP>{});
  if (T == 16 && K == 1024) return f(std::integral_constant<int, T == 16 ? 1024 : -STEP>{});
  const int steps = (int)((K + STEP - 1) / STEP);
  if (MOST > 1 && steps <= 1) return f(std::integral_constant<int, -STEP>{});
  if (MOST > 2 && steps <= 2) return f(std::integral_constant<int, (MOST > 2 ? -2 * STEP : -STEP)>{});
  if (MOST > 3 && steps <= 3) return f(std::integral_constant<int, (MOST > 3 ? -3 * STEP : -STEP)>{});
  f(std::integral_constant<int, (MOST < 4 ? -MOST : -4) * STEP>{}); /* what fused_form sends to T lanes has no more */
}

/* f(T, G): lanes a row and rows a wavefront of the kernels that quantize their own row, for n rows of K weights in a
 * launch. The fewer lanes a row the fewer of them idle at its end (2560 weights: a step and a quarter of 64 lanes), the
 * more a lane keeps of the activations; and rows a wavefront share those, but few rows leave CUs idle. Measured over
 * 512 to 32000 rows of 512 to 4096 weights, the rule is within 1.5 % (Q4_K, Q6_K) and 0.9 % (Q4_0) of the fastest of
 * 16 / 32 / 64 lanes and 1 / 2 / 4 / 8 rows, in the geometric mean; us a call, Q4_K 16 lanes x 4 / 16 x 8 / 32 x 4 / 64 x 2 /
 * 64 x 4: 24576 x 512 4.2 / 4.1 / 4.9 / 6.2 / 5.1, 8192 x 3072 5.5 / 5.7 / 4.9 / 5.2 / 5.0, 2048 x 4096 4.0 / 5.0 / 3.6 / 3.1 / 3.5, 4096 x
 * 4096 5.1 / 6.1 / 4.1 / 4.3 / 4.0. Workgroups of twelve wavefronts, which quantize the row less often, were the fastest form
 * of rows of 4096 while the sums read their records one by one; they are level at 6144, 12288 and 24576 rows now and behind
 * elsewhere (4096 x 4096 4.6). */
template <int DT, typename F> int fused_form(int64_t n, int64_t K, F f) {
  constexpr int SHORT = DT == HIPQ_Q6_K ? 1280 : 2048, MID = DT == HIPQ_Q6_K ? 2048 : 3072;
  typedef std::integral_constant<int, 16> L16;
  typedef std::integral_constant<int, 32> L32;
  typedef std::integral_constant<int, 64> L64;
  if (K < SHORT) return n >= 6144 ? f(L16{}, std::integral_constant<int, 8>{}) : f(L16{}, std::integral_constant<int, 4>{});
  if (n <= 1024) return f(L64{}, std::integral_constant<int, 1>{});
  if (n <= 2048) return f(L64{}, std::integral_constant<int, 2>{});
  return K <= MID ? f(L32{}, std::integral_constant<int, 4>{}) : f(L64{}, std::integral_constant<int, 4>{});
}

template <int DT, int T, int G>
int launch_fused_many(int count, const hipq_weight *const *w, const float *x, float *const *C, hipStream_t s) {
  FusedMulti mw;
  int blocks = 0;
  for (int i = 0; i < FUSED_MAXW; ++i) {
    const int j = i < count ? i : count - 1;
    mw.w[i] = wview(w[j]);
    mw.C[i] = C[j];
    if (i < count) blocks += (int)((w[i]->N + 4 * G - 1) / (4 * G));
    mw.end[i] = blocks;
  }
  const size_t lds = fused_act_bytes<DT>((int)w[0]->K) + 4 * GemvLds<DT, 1, G, false>::DWORDS * sizeof(uint32_t);
  with_length<DT, T>(w[0]->K, [&](auto FK) {
    hipq::launch_kernel(kernel_name<1, DT, T, G, decltype(FK)::value>("gemv_fused_multi_kernel"),
                        (gemv_fused_multi_kernel<DT, T, G, decltype(FK)::value>), dim3((unsigned)blocks), dim3(256), lds, s, mw, x);
  });
  HIPQ_HIP(hipGetLastError());
  return HIPQ_OK;
}

template <int DT, int T, int G>
int launch_fused_one(const hipq_weight *w, const float *x, float *C, hipStream_t s) {
  const unsigned grid = (unsigned)((w->N + 4 * G - 1) / (4 * G));
  const size_t lds = fused_act_bytes<DT>((int)w->K) + 4 * GemvLds<DT, 1, G, false>::DWORDS * sizeof(uint32_t);
  with_length<DT, T>(w->K, [&](auto FK) {
    hipq::launch_kernel(kernel_name<3, DT, T, G, decltype(FK)::value>("gemv_fused_kernel"),
                        (gemv_fused_kernel<DT, T, G, decltype(FK)::value>), dim3(grid), dim3(256), lds, s, wview(w), x, C);
  });
  HIPQ_HIP(hipGetLastError());
  return HIPQ_OK;
}

template <int DT, int T, int R, int G, bool PW>
int launch_one(const hipq_weight *w, const QAct *qa, int M, int pair_rows, float *C, int64_t ldc,
               hipStream_t s) {
  const unsigned grid = (unsigned)((w->N + 4 * G - 1) / (4 * G));
  const size_t lds = 4 * GemvLds<DT, R, G, PW>::DWORDS * sizeof(uint32_t);
  auto go = [&](auto FK) {
    hipq::launch_kernel(kernel_name<5, DT, T, R, G, PW, decltype(FK)::value>("gemv_kernel"), (gemv_kernel<DT, T, R, G, PW, decltype(FK)::value>),
                        dim3(grid), dim3(256), lds, s, wview(w), qview(*qa), M, pair_rows, C, ldc);
  };
  if (w->K > HIPQ_KCHUNK)
    go(std::integral_constant<int, 0>{});
  else
    with_length<DT, T>(w->K, go);
  HIPQ_HIP(hipGetLastError());
  return HIPQ_OK;
}

template <int DT, int T, int G>
int launch_fused_swiglu_one(const hipq_weight *wa, const hipq_weight *wm, const float *x, float *out,
                            hipStream_t s) {
  const unsigned grid = (unsigned)((wa->N + 4 * G - 1) / (4 * G));
  const size_t lds = fused_act_bytes<DT>((int)wa->K) + 4 * GemvLds<DT, 1, G, false>::DWORDS * sizeof(uint32_t);
  with_length<DT, T>(wa->K, [&](auto FK) {
    hipq::launch_kernel(kernel_name<6, DT, T, G, decltype(FK)::value>("gemv_fused_swiglu_kernel"),
                        (gemv_fused_swiglu_kernel<DT, T, G, decltype(FK)::value>), dim3(grid), dim3(256), lds, s, wview(wa), wview(wm), x, out);
  });
  HIPQ_HIP(hipGetLastError());
  return HIPQ_OK;
}

/* The form of a pair of n x K matrices: G rows of each a wavefront, so the lanes a row weigh more (us a call, Q4_0
 * 12288 x 4096 with 32 lanes x 4 / 64 x 2 / 64 x 4 13.7 / 15.1 / 13.2, 12288 x 3072 10.5 / 13.6 / 12.2; Q4_K 12288 x 4096 13.0 / 11.6 /
 * 12.0, 12288 x 2560 8.9 / 10.6 / 9.9) */
template <int DT>
int launch_fused_swiglu(const hipq_weight *wa, const hipq_weight *wm, const float *x, float *out, hipStream_t s) {
  const int64_t n = wa->N, K = wa->K;
  if (K < (DT == HIPQ_Q6_K ? 1280 : 2048)) return launch_fused_swiglu_one<DT, 16, 4>(wa, wm, x, out, s);
  if (n <= 1024) return launch_fused_swiglu_one<DT, 64, 1>(wa, wm, x, out, s);
  if (K <= 3072) return n <= 2048 ? launch_fused_swiglu_one<DT, 32, 2>(wa, wm, x, out, s) : launch_fused_swiglu_one<DT, 32, 4>(wa, wm, x, out, s);
  if (n <= 2048 || DT == HIPQ_Q4_K) return launch_fused_swiglu_one<DT, 64, 2>(wa, wm, x, out, s);
  return launch_fused_swiglu_one<DT, 64, DT == HIPQ_Q4_K ? 2 : 4>(wa, wm, x, out, s);
}

/* Row parts of a long row: nch of kc weights (whole super-blocks, the last one shorter), and wavefronts a workgroup */
struct SplitRow {
  int nch, kc, waves;
};
template <int DT> SplitRow split_row(int64_t K, bool fused) {
  constexpr int STEP = 64 * GemvRec<DT, false>::UNIT;
  SplitRow r;
  r.nch = (int)((K + STEP - 1) / STEP);
  r.kc = (int)((K + 256 * r.nch - 1) / (256 * r.nch)) * 256;
  r.nch = (int)((K + r.kc - 1) / r.kc);
  /* the least that quantizes the row in one pass; on planes one group of rows a workgroup (us, Q4_K 32000 x 12288 with one
   * group 36, with two 38) */
  r.waves = r.nch * (fused ? STEP / 1024 : 1);
  return r;
}
template <int DT, int G, bool FUSED>
int launch_split(const hipq_weight *w, const float *x, const QAct *qa, float *C, hipStream_t s) {
  const SplitRow r = split_row<DT>(w->K, FUSED);
  const int rows = r.waves / r.nch * G;
  const size_t lds = (FUSED ? fused_act_bytes<DT>((int)w->K) : 0) + (size_t)rows * split_stride<DT>((int)w->K) * 4;
  hipq::launch_kernel(kernel_name<7, DT, G, FUSED>("gemv_split_kernel"), (gemv_split_kernel<DT, G, FUSED>),
                      dim3((unsigned)((w->N + rows - 1) / rows)), dim3(64 * r.waves), lds, s, wview(w), x,
                      FUSED ? QView{} : qview(*qa), r.nch, r.kc, C);
  HIPQ_HIP(hipGetLastError());
  return HIPQ_OK;
}

/* One activation row, quantized by a launch of its own: matrices of 32768 rows and more (gemv_fuses_quantizer) */
template <int DT>
int launch_m1(const hipq_weight *w, const QAct *qa, float *C, int64_t ldc, hipStream_t s) {
  const int64_t n = w->N, K = w->K;
  /* long rows: a workgroup's wavefronts share four rows (us with the quantizer's launch, walking the row -> this: Q4_K 65536 x
   * 8192 58 -> 46, 32000 x 12288 41 -> 36; Q4_0 65536 x 8192 61 -> 49; Q6_K 32000 x 6144 35 -> 29) */
  if (K > HIPQ_KCHUNK && split_row<DT>(K, false).nch <= 16) return launch_split<DT, 4, false>(w, nullptr, qa, C, s);
  auto one = [&](auto T, auto G) { return launch_one<DT, decltype(T)::value, 1, decltype(G)::value, false>(w, qa, 1, 0, C, ldc, s); };
  if (n < 8192 && K <= HIPQ_KCHUNK) return fused_form<DT>(n, K, one);
  typedef std::integral_constant<int, 16> L16;
  typedef std::integral_constant<int, 32> L32;
  typedef std::integral_constant<int, 64> L64;
  typedef std::integral_constant<int, 4> G4;
  typedef std::integral_constant<int, 8> G8;
  /* The most lanes a row of those that leave the fewest idle at its end, and eight rows a wavefront, which share the
   * activations, up to rows of 2048. us with the quantizer's launch, before (a wavefront that streamed two to four groups
   * of rows, its loads' count no constant but at K = 1024) -> now: Q4_K 151936 x 512 26.4 -> 10.9, x 1024 18.9 -> 16.8, x 1536
   * 46.8 -> 23.3, x 2560 46.2 -> 37.1, 65536 x 1792 26.0 -> 14.1; Q4_0 151936 x 1024 18.1 -> 17.2, x 2560 46.8 -> 35.9, 32768 x 3584
   * 19.7 -> 15.9; Q6_K 151936 x 768 24.0 -> 19.5, x 3584 80.7 -> 67.0 */
  if (DT == HIPQ_Q6_K) {
    if (K <= 1024) return one(L16{}, G8{});
    if (K <= 2048) return one(L32{}, G8{});
    return one(L64{}, G4{});
  }
  if (K <= 512) return one(L16{}, G8{});
  if (K > 1024 && K <= 2048) return one(L64{}, G8{});
  if (K <= 3072) return DT == HIPQ_Q4_0 ? one(L32{}, G4{}) : one(L32{}, std::integral_constant<int, DT == HIPQ_Q4_0 ? 4 : 8>{});
  return one(L64{}, G4{});
}

/* One activation row as it is, quantized by the kernel */
template <int DT> int launch_fused(const hipq_weight *w, const float *x, float *C, hipStream_t s) {
  if (w->K > HIPQ_KCHUNK) {
    /* rows a workgroup: four up to 1024 rows, eight beyond (us a call, Q4_K 1024 x 8192 4.8 / 4.35 / 4.9 with 2 / 4 / 8, 4096 x 8192
     * 8.7 with 4, 6.6 with 8); Q6_K has four groups of rows a workgroup where the four-bit formats have two */
    constexpr int MOST = DT == HIPQ_Q6_K ? 2 : 4;
    return w->N <= 1024 ? launch_split<DT, MOST / 2, true>(w, x, nullptr, C, s) : launch_split<DT, MOST, true>(w, x, nullptr, C, s);
  }
  return fused_form<DT>(w->N, w->K, [&](auto T, auto G) { return launch_fused_one<DT, decltype(T)::value, decltype(G)::value>(w, x, C, s); });
}

template <int DT>
int launch_fused_multi(int count, const hipq_weight *const *w, const float *x, float *const *C, hipStream_t s) {
  int64_t n = 0;
  for (int i = 0; i < count; ++i) n += w[i]->N;
  return fused_form<DT>(n, w[0]->K, [&](auto T, auto G) { return launch_fused_many<DT, decltype(T)::value, decltype(G)::value>(count, w, x, C, s); });
}

/* 2..8 activation rows in one pass (small prefill chunks, leftover rows). */
template <int DT>
int launch_mr(const hipq_weight *w, const QAct *qa, int M, int pair_rows, float *C, int64_t ldc,
              hipStream_t s) {
  constexpr bool K4 = DT == HIPQ_Q4_K;
  if (M == 2) return launch_one<DT, 64, 2, (K4 ? 4 : 2), false>(w, qa, M, 0, C, ldc, s);
  if (M == 3) return launch_one<DT, 64, 4, 2, false>(w, qa, M, 0, C, ldc, s);
  if (M == 4) return launch_one<DT, 64, 4, 2, K4>(w, qa, M, pair_rows, C, ldc, s);
  return launch_one<DT, 64, 8, 1, K4>(w, qa, M, pair_rows, C, ldc, s);
}

} // namespace

namespace hipq {

int launch_gemv(const hipq_weight *w, const QAct *qa, int M, int pair_rows, float *C, int64_t ldc,
                hipStream_t s) {
  if (M < 1 || M > 8) return fail(HIPQ_ERR_INVALID_ARGUMENT, "gemv handles 1..8 rows, got %d", M);
  switch (w->dtype) {
  case HIPQ_Q4_0:
    return M == 1 ? launch_m1<HIPQ_Q4_0>(w, qa, C, ldc, s)
                  : launch_mr<HIPQ_Q4_0>(w, qa, M, pair_rows, C, ldc, s);
  case HIPQ_Q4_K:
    return M == 1 ? launch_m1<HIPQ_Q4_K>(w, qa, C, ldc, s)
                  : launch_mr<HIPQ_Q4_K>(w, qa, M, pair_rows, C, ldc, s);
  case HIPQ_Q6_K:
    return M == 1 ? launch_m1<HIPQ_Q6_K>(w, qa, C, ldc, s)
                  : launch_mr<HIPQ_Q6_K>(w, qa, M, pair_rows, C, ldc, s);
  }
  return fail(HIPQ_ERR_INVALID_ARGUMENT, "unknown weight dtype %d", w->dtype);
}

/* Rows of one chunk, 16-byte aligned, and matrices below 32768 rows (the sizes that
 * launch_m1 does not stream): beyond that the quantizer's launch is a few per cent of
 * the GEMV and thousands of workgroups quantizing the row again cost more (measured
 * on a 151936 x 4096 Q6_K matrix: 92.9 us against 81.6 us with two launches). */
bool gemv_fuses_quantizer(const hipq_weight *w, const float *x) {
  if ((uintptr_t)x & 15) return false;
  /* rows shared by a workgroup's wavefronts: few rows a workgroup, so the quantizer's launch is the cheaper sooner (us a
   * call, the row quantized in the kernel / by a launch: Q4_K 8192 x 8192 9.7 / 11.1, 8192 x 14336 19.6 / 15.6, 12288 x 9728 18.3 /
   * 15.3; the kernel before, which walked the row, 13.3, 17.6 and 18.7) */
  if (w->K > HIPQ_KCHUNK) return w->K <= 16384 && w->N <= (w->K <= 12288 ? 8192 : 4096);
  return w->N < 32768;
}

bool gemv_fuses_quantizer_multi(int count, const hipq_weight *const *w, const float *x) {
  if (count < 1 || count > FUSED_MAXW) return false;
  int64_t n = 0;
  for (int i = 0; i < count; ++i) {
    if (w[i]->dtype != w[0]->dtype || w[i]->K != w[0]->K || w[i]->K > HIPQ_KCHUNK || !gemv_fuses_quantizer(w[i], x)) return false;
    n += w[i]->N;
  }
  return n < 32768;
}

int launch_gemv_fused_multi(int count, const hipq_weight *const *w, const float *x, float *const *C,
                            hipStream_t s) {
  if (!gemv_fuses_quantizer_multi(count, w, x))
    return fail(HIPQ_ERR_INVALID_ARGUMENT, "these matrices do not take the GEMV that quantizes its own row");
  switch (w[0]->dtype) {
  case HIPQ_Q4_0:
    return launch_fused_multi<HIPQ_Q4_0>(count, w, x, C, s);
  case HIPQ_Q4_K:
    return launch_fused_multi<HIPQ_Q4_K>(count, w, x, C, s);
  case HIPQ_Q6_K:
    return launch_fused_multi<HIPQ_Q6_K>(count, w, x, C, s);
  }
  return fail(HIPQ_ERR_INVALID_ARGUMENT, "unknown weight dtype %d", w[0]->dtype);
}

bool gemv_fuses_swiglu(const hipq_weight *wa, const hipq_weight *wm, const float *x) {
  return wa->dtype == wm->dtype && wa->K == wm->K && wa->N == wm->N && wa->K <= HIPQ_KCHUNK && gemv_fuses_quantizer(wa, x) &&
         2 * wa->N < 32768;
}

int launch_gemv_fused_swiglu(const hipq_weight *wa, const hipq_weight *wm, const float *x, float *out,
                             hipStream_t s) {
  if (!gemv_fuses_swiglu(wa, wm, x))
    return fail(HIPQ_ERR_INVALID_ARGUMENT, "these matrices do not take the fused gated-MLP GEMV");
  switch (wa->dtype) {
  case HIPQ_Q4_0:
    return launch_fused_swiglu<HIPQ_Q4_0>(wa, wm, x, out, s);
  case HIPQ_Q4_K:
    return launch_fused_swiglu<HIPQ_Q4_K>(wa, wm, x, out, s);
  case HIPQ_Q6_K:
    return launch_fused_swiglu<HIPQ_Q6_K>(wa, wm, x, out, s);
  }
  return fail(HIPQ_ERR_INVALID_ARGUMENT, "unknown weight dtype %d", wa->dtype);
}

/* out[m][n] = (y / (1 + exp(-y))) * z, elementwise (the same activation for M > 1 rows) */
__global__ __launch_bounds__(256) void swiglu_rows_kernel(const float *__restrict__ y, const float *__restrict__ z,
                                                          int64_t n_total, int64_t N, int64_t ldo,
                                                          float *__restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n_total) return;
  out[(i / N) * ldo + i % N] = hipq_swiglu(y[i], z[i]);
}

int launch_swiglu_rows(const float *y, const float *z, int64_t M, int64_t N, float *out, int64_t ldo, hipStream_t s) {
  const int64_t n = M * N;
  hipq::launch_kernel("swiglu_rows_kernel", swiglu_rows_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, y, z, n, N, ldo, out);
  HIPQ_HIP(hipGetLastError());
  return HIPQ_OK;
}

int launch_gemv_fused(const hipq_weight *w, const float *x, float *C, hipStream_t s) {
  if (!gemv_fuses_quantizer(w, x))
    return fail(HIPQ_ERR_INVALID_ARGUMENT, "this matrix does not take the GEMV that quantizes its own row");
  switch (w->dtype) {
  case HIPQ_Q4_0:
    return launch_fused<HIPQ_Q4_0>(w, x, C, s);
  case HIPQ_Q4_K:
    return launch_fused<HIPQ_Q4_K>(w, x, C, s);
  case HIPQ_Q6_K:
    return launch_fused<HIPQ_Q6_K>(w, x, C, s);
  }
  return fail(HIPQ_ERR_INVALID_ARGUMENT, "unknown weight dtype %d", w->dtype);
}

} // namespace hipq
