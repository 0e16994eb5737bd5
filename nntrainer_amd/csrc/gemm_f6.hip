// SPDX-License-Identifier: Apache-2.0
/**
 * @file   gemm_f6.hip
 * @brief  Prefill GEMM of Q4_0 x Q8_0 on the gfx950 six-bit matrix instructions.
 *
 * Replaces the M > 1 branch of __ggml_q4_0_8x8_q8_0_GEMM
 * (nntrainer/tensor/cpu_backend/ggml_interface/ggml_interface_omp.cpp:330-389 in the
 * reference checkout) and the nntr_gemm_q4_0_8x8_q8_0 kernel behind it
 * (nntr_ggml_impl/nntr_ggml_impl.cpp:650-3259).
 *
 * What bounds the product is the vector ALU, not the matrix core: every 32 weights have a scale of their
 * own, so a matrix step can cover 32 values of K and each of its sums is then scaled and added in the
 * reference's block order. Measured on this device with two wavefronts a SIMD: a plain fp32 or logical
 * instruction holds the SIMD 2.1 clk, a conversion, a packed, DPP or three-operand integer one 4 clk, and a
 * 32 x 32 matrix instruction of 32 clk leaves room for four vector instructions under it. An int8 step
 * leaves integers: a conversion, the scales' product and a multiply-add a sum, 10 clk (gemm.hip).
 * v_mfma_f32_32x32x64_f8f6f4 with six-bit operands runs at twice the int8 rate and leaves fp32, and
 * six-bit floats hold the quantized integers exactly:
 *   - a weight q - 8 (-8 .. 7) is one fp6 (e2m3) number, in units of 1/8;
 *   - an activation (-127 .. 127) is the sum of two bf6 (e3m2) numbers in units of 1/16: its magnitude
 *     rounded to three significant bits, and the rest, which is at most 8.
 * One instruction takes the 32 values of a block as 64 products, both parts of an activation against the same
 * weight: lane (row, g) holds the first parts of values 16 g .. + 15, then their second parts, lane
 * (column, g) the sixteen weights twice. Every product and every sum is a whole number below 2^24 in those
 * units (the instruction's own block scales turn the units into ones): D is the exact dot product. The
 * scales' products dw * da (22 bits: exact in fp32) come as a rank-one v_mfma_f32_32x32x8_f16. Behind the
 * two, one fused multiply-add a sum is left, acc = fma(D, dw * da, acc): the reference's chain and bits.
 * Per 32 x 32 x 32 that is two matrix instructions and 16 multiply-adds, 90 clk of a SIMD by themselves
 * (210 with the int8 step).
 * Measured, kernel us, int8 kernel -> this one: 512 rows of 12288 x 4096 151 -> 62, of 3072 x 1024 14.7 -> 9.6,
 * 1024 x 1024 7.6 -> 6.7, 1024 x 3072 14.1 -> 12.0 (10.4 with two wavefronts a tile); 333 of 5000 x 2048 29 -> 14; 300 of 1000 x 896 (a K that the int8
 * kernel does not take: eight-row GEMV passes) 135 us a call -> 11. At the first shape the clock falls to about
 * 1.85 GHz under this mix, and 115 clk a step at that clock are 48 us of the 62.
 *
 * Tiling: a workgroup (4 wavefronts side by side) owns 32 rows x 128 columns, each wavefront one 32 x 32
 * tile: 512 rows by 1024 columns, the smallest product of the small decoder's prompt, make 512 wavefronts, and the
 * order of the sums does not let K be split. (Tiles of 64 rows share the weights' operand among two steps, but were
 * not faster at any size: 63 us at the first shape, 9 at 1024 x 1024.)
 * A chunk is 256 of K. Activations come from the quantizer in operand order, one run of consecutive bytes per 64 rows
 * and chunk (hipq_internal.h, QActF6), and go straight to one of three LDS buffers (buffer_load ... lds). Weights
 * stream through registers, up to two chunks ahead, from a copy in operand order (gf_base: 0.81 bytes a weight). The
 * steps run on through the chunks: an operand is read from LDS LOOK steps ahead and a step's matrix instructions are
 * issued before the multiply-adds of the step before it, also across the end of a chunk; the one barrier a chunk lies
 * in its middle. Workgroup ids are mapped so that the row tiles sharing weights run on one XCD.
 */
#include <algorithm>
#include <atomic>
#include <mutex>
#include <new>

#include "gemv_device.h"
#include "quantize_device.h"

namespace {

typedef int v2i __attribute__((ext_vector_type(2)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef __amdgpu_buffer_rsrc_t rsrc_t;
typedef __attribute__((address_space(3))) void *lds_ptr;

constexpr int BM = 32, BN = 128, NT = 256;
constexpr int PARTS = 32 * 384;     /* the activations' parts of 32 rows and one chunk: [block 8]{[64 lanes][16], [64 lanes][8]} */
constexpr int BUF = PARTS + 32 * 16; /* a row buffer in LDS: the parts, then the block scales [32 rows][8] fp16 */
constexpr int MAX_Y = 65535; /* of a grid */
/* Whether `groups` workgroup columns of `mtiles` row tiles leave every workgroup a CU of its own: an XCD takes every eighth
 * column with all its row tiles and has 32 CUs. */
inline bool f6_alone(int mtiles, int64_t groups) { return mtiles * ((groups + 7) / 8) <= 32; }
constexpr int CHUNK = hipq::F6_CHUNK, WTILE = hipq::F6_WTILE; /* bytes of 64 rows / 32 columns and one chunk */

__device__ __forceinline__ rsrc_t make_rsrc(const void *p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void *)p, 0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ v4i ld16(rsrc_t r, uint32_t voff, uint32_t soff) {
  return __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(r, (int)voff, (int)soff, 0));
}
__device__ __forceinline__ v16f zero16() { return v16f{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0}; }

struct MultiF6 { /* up to four weights of one K, their column tiles side by side in the grid */
  const uint8_t *w[4];
  float *C[4];
  int64_t ldc[4];
  int N[4];
  int tile_end[4]; /* running sum of the weights' workgroup columns */
  uint32_t *word;  /* or null: set_word */
};

/* The copies made in front of this launch are complete, by stream order: said to the host (no fence is needed for it) */
__device__ __forceinline__ void set_word(uint32_t *word) {
  if (word && blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) __hip_atomic_store(word, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

/* What a launch reads its rows from (QActF6). */
struct ActF6 {
  const uint8_t *p;
  const uint32_t *flags;
  uint32_t token;
};

/* The sums of f6_sums for a row tile with a scale that is not finite (magnitudes of 8.3e6 and more). There the rank-one
 * instruction may have nothing but the one block's scales on either side: infinity times the zeros that stand for the
 * other blocks would be NaN in all of them. Masking the rows' side as well in the loop below cost 8 % of every product;
 * this plain one runs for such tiles only. */
template <int NS>
__device__ __forceinline__ void f6_sums_plain(const uint8_t *wbase, int N, int chunks, const ActF6 &act, int mt, int tile,
                                              int swap, float (&acc)[NS]) {
  const int lane = threadIdx.x & 63, i32 = lane & 31, g = lane >> 5;
#pragma unroll
  for (int r = 0; r < NS; ++r) acc[r] = 0.f;
  const uint8_t *w = wbase + (size_t)min(tile, ((N + 31) >> 5) - 1) * chunks * WTILE;
  const uint8_t *rows = act.p + (size_t)(mt >> 1) * chunks * CHUNK;
#pragma unroll 1
  for (int c = 0; c < chunks; ++c, w += WTILE, rows += CHUNK)
#pragma unroll 1
    for (int j = 0; j < 8; ++j) {
      const uint8_t *p = rows + (mt & 1) * PARTS + j * 1536;
      const v4i a0 = *(const v4i *)(p + (lane ^ swap) * 16);
      const v2i a1 = *(const v2i *)(p + 1024 + (lane ^ swap) * 8);
      v8i b;
#pragma unroll
      for (int e = 0; e < 3; ++e) {
        const int q = 3 * j + e;
        b[e] = b[3 + e] = *(const int *)(w + (q >> 2) * 1024 + lane * 16 + (q & 3) * 4);
      }
      b[6] = b[7] = 0;
      const v2i da{g ? 0 : (int)*(const uint16_t *)(rows + 2 * PARTS + (mt & 1) * 512 + (i32 ^ swap) * 16 + j * 2), 0},
        dw{g ? 0 : (int)*(const uint16_t *)(w + 6144 + i32 * 16 + j * 2), 0};
      const v16f D = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(v8i{a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], 0, 0}, b, zero16(),
                                                                     3, 2, 0, 127 + 4, 0, 127 + 3);
      const v16f P = __builtin_amdgcn_mfma_f32_32x32x8f16(__builtin_bit_cast(v4h, da), __builtin_bit_cast(v4h, dw), zero16(), 0, 0, 0);
#pragma unroll
      for (int r = 0; r < NS; ++r) acc[r] = fmaf(D[r], P[r], acc[r]);
    }
}

/* The sums of row tile mt and the wavefront's column tile `tile` (lane (column, g), sum r: row 8 (r / 4) + 4 g + r % 4).
 * LOOK: steps an operand is read ahead of its matrix instruction, 1 or 3. ALONE: the wavefront has a SIMD to itself. NS = 8: the
 * sums of half of the rows only; swap: 16 for a wavefront whose half is the upper one, which takes the rows with the halves
 * exchanged. */
template <int LOOK, bool ALONE, int NS = 16>
__device__ __forceinline__ void f6_sums(const uint8_t *wbase, int N, int chunks, const ActF6 &act, int mt, int tile,
                                        float (&acc)[NS], int swap = 0) {
  const uint32_t flag = act.flags[mt]; /* the same for the whole workgroup */
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int lane = threadIdx.x & 63, i32 = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int half = mt & 1; /* of the quantizer's 64 rows */
  const int al = NS == 16 ? lane : lane ^ swap;
  const rsrc_t ra = make_rsrc(act.p + (size_t)(mt >> 1) * chunks * CHUNK, (uint32_t)chunks * CHUNK);
  /* a tile past the last repeats it; it is not stored */
  const rsrc_t rw = make_rsrc(wbase + (size_t)min(tile, ((N + 31) >> 5) - 1) * chunks * WTILE, (uint32_t)chunks * WTILE);

  /* the rows of chunk c into the buffer at byte `at`: kilobytes in turn to the four wavefronts */
  auto copy = [&](int c, int at) {
    unsigned char *to = smem + at;
#pragma unroll
    for (int k0 = 0; k0 < 12; k0 += 4)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_ptr)(to + (k0 + wave) * 1024), 16, lane * 16,
                                               c * CHUNK + half * PARTS + (k0 + wave) * 1024, 0, 0);
    if (wave < 2) /* uniform per wavefront */
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_ptr)(to + PARTS + wave * 256), 4, lane * 4,
                                               c * CHUNK + 2 * PARTS + half * 512 + wave * 256, 0, 0);
  };

  /* Two sets of weight registers: chunk c's in set c & 1; a half of a set takes the loads of chunk c + 2 as soon as
   * chunk c has used it */
  v4i W[2][6], dw[2];
  auto load_w = [&](int c, int k, int p0, int p1) {
#pragma unroll
    for (int p = p0; p < p1; ++p) W[k][p] = ld16(rw, lane * 16, (uint32_t)c * WTILE + p * 1024);
  };
  auto load_dw = [&](int c, int k) { dw[k] = ld16(rw, 6144 + i32 * 16, (uint32_t)c * WTILE); };
  const int last = chunks - 1; /* past the end the last chunk again: a fixed number of loads in flight */
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    copy(min(k, last), k * BUF);
    __builtin_amdgcn_sched_barrier(0); /* the counted waits here and in the first chunk rest on this order */
    load_w(min(k, last), k, 0, 6);
    load_dw(min(k, last), k);
    __builtin_amdgcn_sched_barrier(0);
  }
  /* chunk 0 is there; the second chunk's loads, three or four of rows and seven of weights, may be under way */
  asm volatile("s_waitcnt vmcnt(10)\n\ts_barrier" ::: "memory");
  if (flag == act.token) { /* looked at only here, behind the other loads */
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); /* the copies under way: the caller uses the LDS */
    f6_sums_plain(wbase, N, chunks, act, mt, tile, swap, acc);
    return;
  }

#pragma unroll
  for (int r = 0; r < NS; ++r) acc[r] = 0.f;
  v8i a[LOOK + 1], b;
  v16f D[2], P[2];
  v4h da[2]; /* the row's block scales of an even and an odd chunk */
  auto read_a = [&](int st, int at) {
    const unsigned char *p = smem + at + st * 1536;
    const v4i a0 = *(const v4i *)(p + al * 16);
    const v2i a1 = *(const v2i *)(p + 1024 + al * 8);
    a[st & LOOK] = v8i{a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], 0, 0};
  };
  auto read_da = [&](int k, int at) { da[k] = *(const v4h *)(smem + at + PARTS + (al & 31) * 16 + g * 8); };
  /* Block j of the chunk whose weights are in set k. ALONE: half of a step's sums stand between the two matrix instructions,
   * since the second waits for the first to leave the matrix core (us a call, both instructions first / so: 512 rows of 2048 x 4096
   * 23.1 / 22.8, 525 of 865 x 7168 32.9 / 32.0). With a second wavefront on the SIMD that one has the gap, and the fences of the
   * split cost: 512 of 4096 x 12288 73.0 / 76.9, 77 of 12288 x 7168 36.2 / 38.0. */
  auto start_d = [&](int j, int k) {
#pragma unroll
    for (int e = 0; e < 3; ++e) b[e] = b[3 + e] = W[k][(3 * j + e) >> 2][(3 * j + e) & 3];
    b[6] = b[7] = 0;
    /* 2^4 and 2^3 make whole numbers of the units 1/16 and 1/8 */
    D[j & 1] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a[j & LOOK], b, zero16(), 3, 2, 0, 127 + 4, 0, 127 + 3);
    if (ALONE) asm volatile("" ::"v"(D[j & 1])); /* a use here: the instruction is not moved down to its sums */
  };
  auto start_p = [&](int j, int k) {
    /* lane (row, g) supplies the row's scales of blocks 4 g .. 4 g + 3, lane (column, g) the column's scale of block j
     * at the place of block j and zeros elsewhere */
    const uint32_t h = (uint32_t)dw[k][j >> 1] & (g == (j >> 2) ? ((j & 1) ? 0xffff0000u : 0xffffu) : 0u);
    const v2i dw2 = (j & 2) ? v2i{0, (int)h} : v2i{(int)h, 0};
    P[j & 1] = __builtin_amdgcn_mfma_f32_32x32x8f16(da[k], __builtin_bit_cast(v4h, dw2), zero16(), 0, 0, 0);
    asm volatile("" ::"v"(D[j & 1]), "v"(P[j & 1]));
  };
  auto sums = [&](int j, int r0, int r1) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = r0; r < r1; ++r) acc[r] = fmaf(D[j & 1][r], P[j & 1][r], acc[r]);
#pragma unroll
    for (int r = r0; r < r1; ++r) asm volatile("" : "+v"(acc[r])); /* the sums stay at this step */
    /* half of the sums: the other half's registers are not free either while the instructions write them */
    if (NS == 8) asm volatile("" ::"v"(D[j & 1]), "v"(P[j & 1]));
    __builtin_amdgcn_sched_barrier(0);
  };
  /* Chunk c: its rows at `at`, the next chunk's at at_next, its weights in set k. The middle of the chunk waits for the
   * next chunk's rows (copied since the middle of the previous one), publishes them and gives the previous chunk's buffer
   * to the copy of the chunk after next. */
  auto chunk = [&](int c, int k, int at, int at_next, int at_free) {
    const int c2 = min(c + 2, last);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      read_a((j + LOOK) & 7, j + LOOK < 8 ? at : at_next);
      if (j == 8 - LOOK - 1) read_da(k ^ 1, at_next);
      start_d((j + 1) & 7, j + 1 < 8 ? k : k ^ 1);
      if (ALONE) sums(j, 0, NS / 2);
      start_p((j + 1) & 7, j + 1 < 8 ? k : k ^ 1);
      sums(j, ALONE ? NS / 2 : 0, NS);
      if (j == 3) {
        /* the seven weight loads behind the next chunk's rows may be under way */
        asm volatile("s_waitcnt vmcnt(7)\n\ts_barrier" ::: "memory");
        copy(c2, at_free);
        __builtin_amdgcn_sched_barrier(0);
        load_w(c2, k, 0, 3);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    load_w(c2, k, 3, 6);
    load_dw(c2, k);
    __builtin_amdgcn_sched_barrier(0);
  };
#pragma unroll
  for (int i = 0; i < LOOK; ++i) read_a(i, 0);
  read_da(0, 0);
  start_d(0, 0);
  start_p(0, 0);
  int c = 0, at = 0, at_next = BUF, at_free = 2 * BUF;
  auto turn = [&]() {
    const int t = at;
    at = at_next;
    at_next = at_free;
    at_free = t;
  };
  for (; c + 1 < chunks; c += 2) {
    chunk(c, 0, at, at_next, at_free);
    turn();
    chunk(c + 1, 1, at, at_next, at_free);
    turn();
  }
  if (c < chunks) chunk(c, 0, at, at_next, at_free);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

template <int LOOK, bool ALONE, int NS>
__device__ __forceinline__ void f6_tile(const uint8_t *wbase, int N, int chunks, const ActF6 &act, int M, int mt, int nt,
                                        float *__restrict__ C, int64_t ldc) {
  const int lane = threadIdx.x & 63, i32 = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int tile = NS == 16 ? nt * 4 + wave : nt * 2 + (wave & 1), swap = NS == 16 ? 0 : (wave >> 1) * 16;
  float acc[NS];
  f6_sums<LOOK, ALONE, NS>(wbase, N, chunks, act, mt, tile, acc, swap);

  const int m0 = mt * BM + swap, n = tile * 32 + i32;
  const uint32_t off = (uint32_t)(4 * g) * (uint32_t)ldc + (uint32_t)n; /* the rest of an address is uniform */
  if (m0 + 2 * NS <= M && tile * 32 + 32 <= N) { /* uniform: the whole tile */
#pragma unroll
    for (int r = 0; r < NS; ++r) (C + (int64_t)(m0 + 8 * (r >> 2) + (r & 3)) * ldc)[off] = acc[r];
    return;
  }
#pragma unroll
  for (int r = 0; r < NS; ++r) {
    const int m = m0 + 8 * (r >> 2) + (r & 3);
    if (m + 4 * g < M && n < N) (C + (int64_t)m * ldc)[off] = acc[r];
  }
}

/* Grid: (8 XCDs x row tiles, eighths of the workgroup columns), so that the row tiles sharing weights run on one XCD. All
 * arguments are asked for at once: each that is loaded where it is first used adds a round trip in front of the first
 * load of the tile, and so does a division by the number of row tiles (together with the stores of a whole tile without a
 * condition each, us a call: 512 rows of 2048 x 1024 10.6 -> 9.8, of 1024 x 3072 18.5 -> 17.6).
 * LOOK = 3 takes 184 registers, 188 ALONE and 196 with NS = 8 (two workgroups a CU), LOOK = 1 takes 163 and fits three. NS = 8: two wavefronts a tile, half of its sums
 * each, the matrix instructions twice. */
template <int LOOK, bool ALONE, int NS>
__global__ __launch_bounds__(NT, LOOK == 1 ? 3 : 2) void gemm_f6_kernel(MultiF6 mw, int chunks, ActF6 act, int M, int y0) {
#pragma unroll
  for (int i = 0; i < 4; ++i) asm volatile("" ::"s"(mw.w[i]), "s"(mw.C[i]), "s"(mw.ldc[i]), "s"(mw.N[i]), "s"(mw.tile_end[i]));
  asm volatile("" ::"s"(mw.word), "s"(chunks), "s"(act.p), "s"(act.flags), "s"(act.token), "s"(M), "s"(y0));
  const int mt = (int)(blockIdx.x >> 3);
  int nt = (int)((y0 + blockIdx.y) * 8 + (blockIdx.x & 7));
  if (nt >= mw.tile_end[3]) return; /* uniform per workgroup */
  const uint8_t *w = mw.w[0];
  float *C = mw.C[0];
  int64_t ldc = mw.ldc[0];
  int N = mw.N[0], begin = 0;
#pragma unroll
  for (int i = 1; i < 4; ++i)
    if (nt >= mw.tile_end[i - 1]) w = mw.w[i], C = mw.C[i], ldc = mw.ldc[i], N = mw.N[i], begin = mw.tile_end[i - 1];
  f6_tile<LOOK, ALONE, NS>(w, N, chunks, act, M, mt, nt - begin, C, ldc);
  set_word(mw.word);
}

/* A value of magnitude at most 128 as two bf6 (e3m2) codes in units of 1/16: the magnitude rounded to three
 * significant bits, and the rest (at most 8: codes up to 8 are the number itself). */
__device__ __forceinline__ void bf6_parts(int v, uint32_t &first, uint32_t &second) {
  const int mag = v < 0 ? -v : v;
  const uint32_t t = (__float_as_uint((float)mag) + (1u << 20)) >> 21; /* exponent and two mantissa bits */
  const bool small = mag < 4;
  const int rest = small ? 0 : mag - (int)__uint_as_float(t << 21);
  const uint32_t sign = v < 0 ? 0x20u : 0u;
  first = sign | (small ? (uint32_t)mag : t - 512u);
  second = (rest < 0 ? (sign ^ 0x20u) | (uint32_t)(-rest) : sign | (uint32_t)rest);
}

/* Block b (of nbp a row) of row m: the calling lane's four of its values in x, the block's eight lanes consecutive */
__device__ __forceinline__ void f6_quantize_block(const float4 &x, int64_t m, int b, int nbp, uint8_t *__restrict__ out,
                                                  uint32_t *__restrict__ flags, uint32_t token) {
  const int lane = threadIdx.x & 63, sub = lane & 7;
  constexpr int PARTS = hipq::F6_ROWS * 384;
  uint16_t dh;
  int qsum;
  const uint32_t q = (uint32_t)hipq_quantize_q8_0_lane(x, dh, qsum);
  uint32_t part[2] = {0, 0}; /* this lane's four codes of each part, 24 bits */
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    uint32_t first, second;
    bf6_parts((int)(int8_t)(q >> (8 * k)), first, second);
    part[0] |= first << (6 * k);
    part[1] |= second << (6 * k);
  }
  uint32_t w[6]; /* the quad's sixteen values: 96 bits of each part */
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int mine = (int)part[h];
    const uint32_t x0 = (uint32_t)hipq_dpp_i<0x00>(mine), x1 = (uint32_t)hipq_dpp_i<0x55>(mine),
                   x2 = (uint32_t)hipq_dpp_i<0xAA>(mine), x3 = (uint32_t)hipq_dpp_i<0xFF>(mine);
    w[3 * h] = x0 | (x1 << 24);
    w[3 * h + 1] = (x1 >> 8) | (x2 << 16);
    w[3 * h + 2] = (x2 >> 16) | (x3 << 8);
  }
  const int r = (int)(m & (hipq::F6_ROWS - 1)), g = sub >> 2, j = b & 7;
  uint8_t *dst = out + ((m / hipq::F6_ROWS) * (nbp >> 3) + (b >> 3)) * hipq::F6_CHUNK;
  uint8_t *o = dst + (r >> 5) * (PARTS / 2) + j * 1536;
  const int at = g * 32 + (r & 31);
  if ((lane & 3) == 0) *(uint4 *)(o + at * 16) = make_uint4(w[0], w[1], w[2], w[3]);
  if ((lane & 3) == 1) *(uint2 *)(o + 1024 + at * 8) = make_uint2(w[4], w[5]);
  if (sub == 0) {
    *(uint16_t *)(dst + PARTS + r * 16 + j * 2) = dh;
    if ((dh & 0x7c00) == 0x7c00) flags[m >> 5] = token; /* not finite: f6_sums_plain */
  }
}

/* The gated pair of an MLP: out = swiglu(act sums) * mul sums. Two wavefronts of a workgroup take 32 columns each of the
 * one matrix, the other two the same columns of the other; at the end each keeps half of its tile's rows and hands the
 * other half over through LDS. The two products never reach memory: as products and a launch of the activation 512 rows of
 * 3072 columns wrote and read 25 MB more (294 -> 273 us for four decoder layers). QUANT: the result goes out quantized, as the
 * operand of the down projection behind it: 32 columns of a tile are the blocks of 32 rows, which pass through LDS to the
 * lanes that the quantizer gives them. As fp32 rows and a quantizer's launch 512 rows of 3072 columns wrote and read 12.6 MB
 * more (four decoder layers of 1024 and 3072 over 512 rows 271.6 -> 253.7 us). */
struct GatedF6 {
  const uint8_t *act, *mul;
  float *out;
  int64_t ldo;
  int N, ntiles; /* columns, workgroup columns of 64 (QUANT: with those that fill the last chunk, written as zeros) */
  uint32_t *word; /* or null: set_word */
  uint8_t *q;     /* QUANT: where the quantized rows go (QActF6) */
  uint32_t *flags, token;
};
template <int LOOK, bool ALONE, bool QUANT>
__device__ __forceinline__ void f6_gated_tile(const GatedF6 &p, int chunks, const ActF6 &act, int M, int mt, int nt) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int lane = threadIdx.x & 63, i32 = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const bool second = wave >= 2;
  const int tile = nt * 2 + (wave & 1);
  float acc[16];
  f6_sums<LOOK, ALONE>(second ? p.mul : p.act, p.N, chunks, act, mt, tile, acc);

  __syncthreads(); /* no wavefront reads or fills its row buffers any more */
  float *mine = (float *)smem + wave * 512, *other = (float *)smem + (wave ^ 2) * 512;
#pragma unroll
  for (int r = 0; r < 8; ++r) mine[r * 64 + lane] = second ? acc[r] : acc[8 + r];
  __syncthreads();
  if constexpr (QUANT) {
    constexpr int LD = 36; /* floats between the rows of a tile: whole 16 bytes, and rows on different banks */
    float *hs = (float *)smem + 4 * 512, *ht = hs + (wave & 1) * (32 * LD) + i32;
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const float o = other[r * 64 + lane];
      ht[((second ? 16 : 0) + 8 * (r >> 2) + (r & 3) + 4 * g) * LD] = second ? hipq_swiglu(o, acc[8 + r]) : hipq_swiglu(acc[r], o);
    }
    __syncthreads();
    const int row = threadIdx.x >> 3;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int b = nt * 2 + t;
      float4 x = *(const float4 *)(hs + t * (32 * LD) + row * LD + (threadIdx.x & 7) * 4);
      if (b * 32 >= p.N) x = make_float4(0.f, 0.f, 0.f, 0.f); /* uniform */
      f6_quantize_block(x, (int64_t)mt * BM + row, b, p.ntiles * 2, p.q, p.flags, p.token);
    }
    return;
  }
  const int m0 = mt * BM + (second ? 16 : 0), n = tile * 32 + i32;
  const uint32_t off = (uint32_t)(4 * g) * (uint32_t)p.ldo + (uint32_t)n;
#pragma unroll
  for (int r = 0; r < 8; ++r) {
    const float o = other[r * 64 + lane];
    const float h = second ? hipq_swiglu(o, acc[8 + r]) : hipq_swiglu(acc[r], o);
    const int m = m0 + 8 * (r >> 2) + (r & 3);
    if (m + 4 * g < M && n < p.N) (p.out + (int64_t)m * p.ldo)[off] = h;
  }
}
template <int LOOK, bool ALONE, bool QUANT>
__global__ __launch_bounds__(NT, LOOK == 1 ? 3 : 2) void gemm_f6_gated_kernel(GatedF6 p, int chunks, ActF6 act, int M, int y0) {
  asm volatile("" ::"s"(p.act), "s"(p.mul), "s"(p.out), "s"(p.ldo), "s"(p.N), "s"(p.ntiles), "s"(p.word), "s"(p.q), "s"(p.flags),
               "s"(p.token), "s"(chunks), "s"(act.p), "s"(act.flags), "s"(act.token), "s"(M), "s"(y0));
  const int mt = (int)(blockIdx.x >> 3), nt = (int)((y0 + blockIdx.y) * 8 + (blockIdx.x & 7));
  if (nt < p.ntiles) f6_gated_tile<LOOK, ALONE, QUANT>(p, chunks, act, M, mt, nt); /* uniform per workgroup */
  set_word(p.word);
}

/* ---- the copy of a weight in operand order ---- */

struct CopyF6 { /* up to four weights of one K; the workgroups of weight i end at end[i] */
  const uint8_t *qs[4];
  const uint16_t *d[4];
  uint8_t *out[4];
  int N[4], end[4];
  int nb, chunks; /* blocks and chunks a row */
};

/* The fp6 codes of four weights, one nibble a byte, as 24 bits: v - 8 is the number itself from 0 to 7, the sign bit and
 * its magnitude below */
__device__ __forceinline__ uint32_t f6_codes(uint32_t v) {
  const uint32_t t = v ^ 0x08080808u, m = (t >> 3) & 0x01010101u; /* m: below zero, where t = v + 8 */
  const uint32_t code = (((t ^ ((m << 8) - m)) + m) & 0x0f0f0f0fu) | (m << 5);
  const uint32_t pairs = (code & 0x003f003fu) | ((code >> 2) & 0x0fc00fc0u);
  return (pairs & 0xfffu) | ((pairs >> 4) & 0xfff000u);
}

/* A wavefront takes half a chunk (four blocks) of a tile's 32 rows: 64 bytes a row in, four lanes a row, through LDS to
 * lane (column, g), which writes twelve of its 24 dwords, three whole kilobytes a wavefront. */
__device__ __forceinline__ void f6_copy(const uint8_t *__restrict__ qs, const uint16_t *__restrict__ d, int N, int nb, int chunks,
                                        uint8_t *__restrict__ out, int block) {
  __shared__ __attribute__((aligned(16))) uint4 rows[4][32][5]; /* a row's four blocks, and a gap against bank conflicts */
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, i32 = lane & 31, g = lane >> 5;
  const uint32_t unit = (uint32_t)block * 4 + wave; /* (tile, chunk, half) */
  const uint32_t tc = unit >> 1, tile = tc / (uint32_t)chunks; /* tc: tile * chunks + chunk */
  const int half = (int)(unit & 1);
  const int64_t n0 = (int64_t)tile * 32;
  const int b0 = (int)(tc - tile * (uint32_t)chunks) * 8 + half * 4; /* first block in the row */
  const bool live = n0 < N;                         /* the last workgroup may have wavefronts to spare */
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = i * 16 + (lane >> 2), b = b0 + (lane & 3);
    uint4 x = make_uint4(0x88888888u, 0x88888888u, 0x88888888u, 0x88888888u); /* weights of zero */
    if (n0 + r < N && b < nb) x = *(const uint4 *)(qs + ((n0 + r) * nb + b) * 16);
    rows[wave][r][lane & 3] = x;
  }
  uint32_t sc = 0; /* the scales of blocks 2 g and 2 g + 1 of the half */
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int b = b0 + 2 * g + i;
    if (n0 + i32 < N && b < nb) sc |= (uint32_t)d[(n0 + i32) * nb + b] << (16 * i);
  }
  __syncthreads();
  if (!live) return;
  uint32_t w[12];
#pragma unroll
  for (int j = 0; j < 4; ++j) { /* byte i of a block = elements i (low nibble) and i + 16 */
    const uint4 x = rows[wave][i32][j];
    const uint32_t a = f6_codes((x.x >> (4 * g)) & 0x0f0f0f0fu), b = f6_codes((x.y >> (4 * g)) & 0x0f0f0f0fu),
                   c = f6_codes((x.z >> (4 * g)) & 0x0f0f0f0fu), e = f6_codes((x.w >> (4 * g)) & 0x0f0f0f0fu);
    w[3 * j] = a | (b << 24);
    w[3 * j + 1] = (b >> 8) | (c << 16);
    w[3 * j + 2] = (c >> 16) | (e << 8);
  }
  uint8_t *dst = out + (size_t)tc * WTILE;
#pragma unroll
  for (int p = 0; p < 3; ++p)
    *(uint4 *)(dst + (3 * half + p) * 1024 + lane * 16) = make_uint4(w[4 * p], w[4 * p + 1], w[4 * p + 2], w[4 * p + 3]);
  *(uint32_t *)(dst + 6144 + i32 * 16 + half * 8 + g * 4) = sc;
}

/* f6_copy of workgroup `block`. A macro, so that the struct's members are picked where it is a kernel's argument: picked
 * through a reference it went to scratch memory */
#define F6_COPY(cw, block)                                                                                       \
  do {                                                                                                           \
    int wi = 0, begin = 0;                                                                                       \
    if ((block) >= cw.end[0]) wi = 1, begin = cw.end[0];                                                         \
    if ((block) >= cw.end[1]) wi = 2, begin = cw.end[1];                                                         \
    if ((block) >= cw.end[2]) wi = 3, begin = cw.end[2];                                                         \
    f6_copy(wi == 0 ? cw.qs[0] : wi == 1 ? cw.qs[1] : wi == 2 ? cw.qs[2] : cw.qs[3],                             \
            wi == 0 ? cw.d[0] : wi == 1 ? cw.d[1] : wi == 2 ? cw.d[2] : cw.d[3],                                 \
            wi == 0 ? cw.N[0] : wi == 1 ? cw.N[1] : wi == 2 ? cw.N[2] : cw.N[3], cw.nb, cw.chunks,               \
            wi == 0 ? cw.out[0] : wi == 1 ? cw.out[1] : wi == 2 ? cw.out[2] : cw.out[3], (block)-begin);         \
  } while (0)

__global__ __launch_bounds__(256) void f6_weights_kernel(CopyF6 cw) { F6_COPY(cw, (int)blockIdx.x); }

/* ---- the activations ---- */

/* Q8_0 in the form of the six-bit GEMM (QActF6). A wavefront takes one block of eight consecutive rows, eight lanes a
 * row (128 bytes of a row in, two whole lines of operands out). Rows M and beyond of the last 64 and blocks of K and
 * beyond are written as zeros. */
struct RowsF6 {
  const float *A;
  int64_t M, lda;
  uint32_t n_units; /* octets of rows (padding included) x blocks */
  int nbp, K;
  uint8_t *out;
  uint32_t *flags;
  uint32_t token;
};
__device__ __forceinline__ void f6_quantize(const RowsF6 &p, int block) {
  const int64_t M = p.M;
  const int K = p.K, nbp = p.nbp;
  const uint32_t unit = (uint32_t)block * 4 + (threadIdx.x >> 6);
  if (unit >= p.n_units) return; /* uniform per wavefront */
  const int lane = threadIdx.x & 63, sub = lane & 7;
  const uint32_t octet = unit / (uint32_t)nbp; /* a 64-bit quotient was half of the kernel's instructions */
  const int b = (int)(unit - octet * (uint32_t)nbp);
  const int64_t m = (int64_t)octet * 8 + (lane >> 3);
  float4 x = *(const float4 *)(p.A + (m < M ? m : M - 1) * p.lda + min(b * 32 + 4 * sub, K - 4));
  if (m >= M || b * 32 >= K) x = make_float4(0.f, 0.f, 0.f, 0.f);
  f6_quantize_block(x, m, b, nbp, p.out, p.flags, p.token);
}

__global__ __launch_bounds__(256) void quantize_q8_0_f6_kernel(RowsF6 p) { f6_quantize(p, (int)blockIdx.x); }

/* Both in one launch, for the call that makes the copies: the copies' workgroups in front, their reads of weights that
 * no cache holds beside the quantization. First pass of four decoder layers of 1024 / 3072 over 512 rows, fresh weights:
 * 470 us with an allocation, an event and a launch a weight, 380 with the copies of a call in a launch of their own in
 * front of the quantizer's, 329 this way (272 from the second pass on; 360 with the int8 kernel, which needs no copy). */
__global__ __launch_bounds__(256) void quantize_copy_f6_kernel(RowsF6 p, CopyF6 cw) {
  if ((int)blockIdx.x < cw.end[3]) /* uniform */
    F6_COPY(cw, (int)blockIdx.x);
  else
    f6_quantize(p, (int)blockIdx.x - cw.end[3]);
}

} // namespace

namespace hipq {

/* ---- who may read a copy ----
 * A copy is made by the product that asks for it, in the launch of its quantizer, and nothing waits. Until it is known
 * to be complete it is PENDING, and only the stream it was made on may read it; a product on another stream takes the
 * kernels that read the weight as stored (the same bits). Complete is what the page-locked word of its batch says, which
 * the product behind the quantizer sets: a plain read, so also a call that is being captured into a graph, where events
 * may not be queried, finds out. A graph may be launched on any stream, so a captured product reads complete copies
 * only.
 * The same stream is known by its handle alone, and one handle can stand for two streams (hipStreamPerThread; a stream
 * made after another was destroyed): the event of the batch orders those. */
struct F6Batch {
  uint32_t *word, *word_dev;
  hipEvent_t ev;
  hipStream_t s;
  int refs; /* PENDING weights that point here */
  F6Batch *next;
};

/* The copies' memory: blocks of 64 MiB (a copy of more than half that has one of its own size), the first gap that is
 * large enough, given back with the last copy in it; one empty block is kept for the next weights. A hipMalloc for each
 * copy took 13 to 30 us of the first product. */
struct F6Block;
struct F6Copy {
  F6Block *block;
  size_t at, bytes; /* multiples of 256 */
  F6Copy *next;     /* the block's copies in the order of their places */
};
struct F6Block {
  uint8_t *base;
  size_t size;
  F6Copy *first;
  F6Block *next;
};

namespace {
std::atomic<uint32_t> f6_calls{0}; /* the calls' tokens */
std::mutex f6_mu; /* guards what follows and every weight's gf_ fields */
struct F6Page { /* batches and the page-locked page of their words; given back by f6_shutdown */
  static constexpr int COUNT = 1024;
  F6Batch batch[COUNT];
  uint32_t *words;
  F6Page *next;
};
F6Page *f6_pages = nullptr;
F6Batch *f6_idle = nullptr; /* batches no weight points to */

void batch_idle(F6Batch *b) {
  b->next = f6_idle;
  f6_idle = b;
}

constexpr size_t F6_BLOCK = (size_t)64 << 20;
F6Block *f6_blocks = nullptr;

int mem_get(size_t bytes, F6Copy **out) {
  F6Copy *c = new (std::nothrow) F6Copy();
  if (!c) return fail(HIPQ_ERR_OUT_OF_MEMORY, "host allocation failed");
  c->bytes = bytes;
  for (F6Block *b = f6_blocks; b && !c->block; b = b->next) {
    size_t end = 0; /* of the copy in front */
    F6Copy **at = &b->first;
    for (; *at && (*at)->at - end < bytes; at = &(*at)->next) end = (*at)->at + (*at)->bytes;
    if (!*at && b->size - end < bytes) continue;
    c->block = b, c->at = end, c->next = *at;
    *at = c;
  }
  if (!c->block) {
    F6Block *b = new (std::nothrow) F6Block();
    hipError_t e = hipErrorOutOfMemory;
    if (b) {
      b->size = bytes > F6_BLOCK / 2 ? bytes : F6_BLOCK;
      e = hipMalloc((void **)&b->base, b->size);
      if (e != hipSuccess && b->size > bytes) { /* a full device may still have room for this one */
        (void)hipGetLastError();
        b->size = bytes;
        e = hipMalloc((void **)&b->base, b->size);
      }
    }
    if (e != hipSuccess) {
      delete b;
      delete c;
      return fail(HIPQ_ERR_OUT_OF_MEMORY, "six-bit copy of %zu bytes: %s", bytes, hipGetErrorString(e));
    }
    c->block = b, b->first = c;
    b->next = f6_blocks;
    f6_blocks = b;
  }
  *out = c;
  return HIPQ_OK;
}
/* gives back the empty blocks, one of which may stay for the next weights */
void mem_trim(bool keep) {
  for (F6Block **at = &f6_blocks; *at;) {
    F6Block *b = *at;
    if (!b->first && keep && b->size == F6_BLOCK) {
      keep = false;
    } else if (!b->first) {
      *at = b->next;
      (void)hipFree(b->base);
      delete b;
      continue;
    }
    at = &b->next;
  }
}
void copy_put(hipq_weight *w) {
  F6Copy *c = w->gf_copy;
  if (!c) return;
  F6Copy **at = &c->block->first;
  while (*at != c) at = &(*at)->next;
  *at = c->next;
  if (!c->block->first) mem_trim(true);
  delete c;
  w->gf_copy = nullptr;
  w->gf_base = nullptr;
}

int batch_get(hipStream_t s, F6Batch **out) {
  if (!f6_idle) {
    F6Page *pg = new (std::nothrow) F6Page();
    if (!pg) return fail(HIPQ_ERR_OUT_OF_MEMORY, "host allocation failed");
    uint32_t *dev = nullptr;
    hipError_t e = hipHostMalloc((void **)&pg->words, F6Page::COUNT * 4, hipHostMallocDefault);
    if (e == hipSuccess && (e = hipHostGetDevicePointer((void **)&dev, pg->words, 0)) != hipSuccess) (void)hipHostFree(pg->words);
    if (e != hipSuccess) {
      delete pg;
      return fail(HIPQ_ERR_OUT_OF_MEMORY, "page-locked words: %s", hipGetErrorString(e));
    }
    pg->next = f6_pages;
    f6_pages = pg;
    for (int i = F6Page::COUNT; i-- > 0;) {
      pg->batch[i] = F6Batch{pg->words + i, dev + i, nullptr, nullptr, 0, nullptr};
      batch_idle(&pg->batch[i]);
    }
  }
  F6Batch *b = f6_idle;
  if (!b->ev) HIPQ_HIP(hipEventCreateWithFlags(&b->ev, hipEventDisableTiming));
  f6_idle = b->next;
  __atomic_store_n(b->word, 0u, __ATOMIC_RELAXED);
  b->s = s;
  *out = b;
  return HIPQ_OK;
}
void batch_drop(hipq_weight *w) {
  F6Batch *b = w->gf_batch;
  w->gf_batch = nullptr;
  if (b && --b->refs == 0) batch_idle(b);
}

void make_undo(F6Make &m) {
  for (int i = 0; i < m.count; ++i) {
    copy_put(m.w[i]);
    m.w[i]->gf_state = F6_NONE;
  }
  m.count = 0;
  batch_idle(m.batch);
}

/* Whether the weight's copy is complete; looks up to `spins` times more */
bool complete(hipq_weight *w, int &spins) {
  if (w->gf_state == F6_PENDING) {
    while (!__atomic_load_n(w->gf_batch->word, __ATOMIC_ACQUIRE)) {
      if (spins <= 0) return false;
      --spins;
      __builtin_ia32_pause();
    }
    batch_drop(w);
    __atomic_store_n(&w->gf_state, F6_COMPLETE, __ATOMIC_RELEASE);
  }
  return w->gf_state == F6_COMPLETE;
}
} // namespace

/* *ready: the products a call enqueues on s next may read the copies of the weights. For those that are missing, where
 * may_make and the stream is not being captured, `make` has the memory; the call hands it to its quantizer. */
int f6_copies(int count, const hipq_weight *const *cw, hipStream_t s, bool may_make, bool *ready, F6Make *make) {
  *ready = false;
  int done = 0;
  for (int i = 0; i < count; ++i) done += __atomic_load_n(&cw[i]->gf_state, __ATOMIC_ACQUIRE) == F6_COMPLETE;
  if (done == count) {
    *ready = true;
    return HIPQ_OK;
  }
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &cs) != hipSuccess) (void)hipGetLastError();
  const bool capturing = cs != hipStreamCaptureStatusNone;
  hipq_weight *const *w = const_cast<hipq_weight *const *>(cw);
  std::lock_guard<std::mutex> lk(f6_mu);
  int missing = 0;
  /* the graph keeps the kernels that are chosen now: a copy that is about to complete is waited for, up to about a
   * millisecond a call */
  int spins = capturing ? 20000 : 0;
  F6Batch *behind = nullptr;
  for (int i = 0; i < count; ++i) {
    if (w[i]->gf_state == F6_MAKING) return HIPQ_OK; /* another thread is about to enqueue it */
    if (w[i]->gf_state == F6_NONE) {
      if (w[i]->dtype != HIPQ_Q4_0 || w[i]->expert_tiles)
        return fail(HIPQ_ERR_INVALID_ARGUMENT, "only Q4_0 weights in the plane layout have a six-bit copy");
      if (w[i]->K != w[0]->K) return fail(HIPQ_ERR_INVALID_ARGUMENT, "the copies of one call are of one K");
      ++missing;
    } else if (!complete(w[i], spins)) {
      F6Batch *b = w[i]->gf_batch;
      if (capturing || b->s != s) return HIPQ_OK;
      if (b != behind) HIPQ_HIP(hipStreamWaitEvent(s, b->ev, 0));
      behind = b;
    }
  }
  if (missing) {
    if (!may_make || capturing || missing > F6Make::MOST) return HIPQ_OK;
    if (int rc = batch_get(s, &make->batch)) return rc;
    const int64_t chunks = (w[0]->K + 255) / 256;
    for (int i = 0; i < count; ++i) {
      hipq_weight *x = w[i];
      if (x->gf_state != F6_NONE) continue; /* has one, or stands in the list twice */
      if (int rc = mem_get((size_t)((x->N + 31) / 32 * chunks) * F6_WTILE, &x->gf_copy)) {
        make_undo(*make);
        return rc;
      }
      x->gf_base = x->gf_copy->block->base + x->gf_copy->at;
      x->gf_state = F6_MAKING;
      make->w[make->count++] = x;
    }
  }
  *ready = true;
  return HIPQ_OK;
}

F6Make::~F6Make() { /* a call that failed between f6_copies and its quantizer's launch */
  if (!count) return;
  std::lock_guard<std::mutex> lk(f6_mu);
  make_undo(*this);
}

size_t qact_f6_bytes(int64_t M, int64_t K) {
  const size_t tiles = (size_t)((M + F6_ROWS - 1) / F6_ROWS);
  return tiles * (size_t)((K + 255) / 256) * F6_CHUNK + ((tiles * 8 + 255) & ~(size_t)255); /* the flags: two a tile of 64 rows */
}
QActF6 qact_f6_carve(void *mem, int64_t M, int64_t K) {
  const int64_t chunks = (K + 255) / 256;
  return QActF6{(uint8_t *)mem, (uint32_t *)((uint8_t *)mem + (size_t)((M + F6_ROWS - 1) / F6_ROWS) * chunks * F6_CHUNK), 0, (int)M, (int)K,
                (int)chunks, nullptr};
}

int launch_quantize_q8_0_f6(const float *A, int64_t M, int64_t K, int64_t lda, QActF6 *qa, F6Make *make, hipStream_t s) {
  if (M <= 0) return HIPQ_OK;
  if (K % 32 || lda < K) return fail(HIPQ_ERR_INVALID_ARGUMENT, "Q8_0: K=%lld must be a multiple of 32 and lda >= K", (long long)K);
  if (((uintptr_t)A & 15) || (lda & 3))
    return fail(HIPQ_ERR_INVALID_ARGUMENT, "activation rows must be 16-byte aligned");
  const int64_t units = (M + F6_ROWS - 1) / F6_ROWS * (F6_ROWS / 8) * (qa->chunks * 8); /* padding included */
  if (units > INT32_MAX) return fail(HIPQ_ERR_NOT_SUPPORTED, "%lld x %lld values in one call", (long long)M, (long long)K);
  qa->token = ++f6_calls;
  const RowsF6 rows{A, M, lda, (uint32_t)units, qa->chunks * 8, (int)K, qa->p, qa->flags, qa->token};
  const unsigned blocks = (unsigned)((units + 3) / 4);
  if (!make || !make->count) {
    launch_kernel("quantize_q8_0_f6_kernel", quantize_q8_0_f6_kernel, dim3(blocks), dim3(256), 0, s, rows);
    HIPQ_HIP(hipGetLastError());
    return HIPQ_OK;
  }
  for (int i = (make->count - 1) / 4 * 4; i >= 0; i -= 4) { /* four copies a launch, the last ones with the rows */
    CopyF6 cw;
    cw.nb = (int)(K / 32);
    cw.chunks = qa->chunks;
    int end = 0;
    for (int k = 0; k < 4; ++k) {
      const hipq_weight *x = make->w[std::min(i + k, make->count - 1)];
      cw.qs[k] = x->qs, cw.d[k] = x->d, cw.out[k] = x->gf_base, cw.N[k] = (int)x->N;
      if (i + k < make->count) end += (int)(((x->N + 31) / 32 * cw.chunks + 1) / 2); /* four half chunks a workgroup */
      cw.end[k] = end;
    }
    if (i)
      launch_kernel("f6_weights_kernel", f6_weights_kernel, dim3((unsigned)end), dim3(256), 0, s, cw);
    else
      launch_kernel("quantize_copy_f6_kernel", quantize_copy_f6_kernel, dim3((unsigned)end + blocks), dim3(256), 0, s, rows, cw);
  }
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipEventRecord(make->batch->ev, s);
  if (e != hipSuccess) {
    (void)hipStreamSynchronize(s); /* before ~F6Make gives the copies' memory back */
    return fail(HIPQ_ERR_RUNTIME, "six-bit copies: %s", hipGetErrorString(e));
  }
  qa->word = make->batch->word_dev;
  std::lock_guard<std::mutex> lk(f6_mu);
  for (int i = 0; i < make->count; ++i) {
    make->w[i]->gf_batch = make->batch;
    __atomic_store_n(&make->w[i]->gf_state, F6_PENDING, __ATOMIC_RELEASE);
  }
  make->batch->refs = make->count;
  make->count = 0;
  return HIPQ_OK;
}

void f6_release(hipq_weight *w) {
  std::lock_guard<std::mutex> lk(f6_mu);
  batch_drop(w);
  copy_put(w);
  w->gf_state = F6_NONE;
}

void f6_shutdown() {
  std::lock_guard<std::mutex> lk(f6_mu);
  while (F6Page *pg = f6_pages) {
    f6_pages = pg->next;
    for (F6Batch &b : pg->batch)
      if (b.ev) (void)hipEventDestroy(b.ev);
    (void)hipHostFree(pg->words);
    delete pg;
  }
  f6_idle = nullptr;
  mem_trim(false);
}

int launch_gemm_f6(int count, const hipq_weight *const *w, const QActF6 *qa, int M, float *const *C, const int64_t *ldc,
                   hipStream_t s) {
  if (count < 1 || count > 4) return fail(HIPQ_ERR_INVALID_ARGUMENT, "1 to 4 weights per launch, got %d", count);
  MultiF6 mw;
  int tiles = 0;
  int64_t halves = 0; /* workgroup columns of 64, of two tiles */
  for (int i = 0; i < 4; ++i) {
    const int k = i < count ? i : count - 1;
    if (!w[k]->gf_base || w[k]->K != w[0]->K || w[k]->K != qa->K || M != qa->M)
      return fail(HIPQ_ERR_INVALID_ARGUMENT, "the weights of one launch share K and have their six-bit copy");
    mw.w[i] = w[k]->gf_base;
    mw.N[i] = (int)w[k]->N;
    mw.C[i] = C[k];
    mw.ldc[i] = ldc[k];
    if (i < count) tiles += (int)((w[k]->N + BN - 1) / BN), halves += (w[k]->N + BN / 2 - 1) / (BN / 2);
    mw.tile_end[i] = tiles; /* unused entries repeat the total: no workgroup lands in them */
  }
  mw.word = qa->word;
  const int mtiles = (M + BM - 1) / BM;
  auto go = [&](const char *name, auto kernel) {
    for (int y0 = 0, end = (tiles + 7) / 8; y0 < end; y0 += MAX_Y)
      launch_kernel(name, kernel, dim3((unsigned)(8 * mtiles), (unsigned)std::min(end - y0, MAX_Y)), dim3(NT), 3 * BUF, s, mw, qa->chunks,
                    ActF6{qa->p, qa->flags, qa->token}, M, y0);
  };
  /* up to two workgroups a CU: the deeper read-ahead (512 rows of 1024 x 3072 13.1 -> 12.0 us, 1024 x 1024 7.5 -> 6.7);
   * beyond, three workgroups a CU cover the reads (512 of 12288 x 4096 67 -> 62 us) */
  if (f6_alone(mtiles, halves) || (halves <= 8 && mtiles * (int64_t)tiles <= 128)) {
    /* Two wavefronts a tile (NS = 8), where their workgroups, twice as many, still have a CU each: a wavefront alone on its SIMD
     * takes a step's vector instructions one after the other, 150 clk with sixteen sums and 115 with eight. us a call, a
     * wavefront a tile / two: 512 rows of 1024 x 1024 9.8 / 9.2, x 3072 17.9 / 16.8, x 12288 47.2 / 43.7, 128 of 4096 x 4096 17.3 / 15.8.
     * With more of them the halves take a CU twice: 525 rows of 865 x 1024 10.2 / 11.0, x 7168 32.5 / 37.3, x 12288 48.3 / 56.5 (238
     * workgroups, 34 of them on an XCD), 512 of 1536 x 2048 13.7 / 15.0. Not with up to eight workgroup columns, where an XCD has one
     * of either kind and the halves run on twice the XCDs: 2000 of 256 x 1024 17.6 / 15.9, 4096 of 128 x 4096 66.0 / 59.4. */
    tiles = 0;
    for (int i = 0; i < 4; ++i) {
      if (i < count) tiles += (int)((w[i]->N + BN / 2 - 1) / (BN / 2));
      mw.tile_end[i] = tiles;
    }
    go("gemm_f6_kernel<3, true, 8>", gemm_f6_kernel<3, true, 8>);
  } else if (f6_alone(mtiles, tiles))
    go("gemm_f6_kernel<3, true, 16>", gemm_f6_kernel<3, true, 16>);
  else if (mtiles * (int64_t)tiles <= 512)
    go("gemm_f6_kernel<3, false, 16>", gemm_f6_kernel<3, false, 16>);
  else
    go("gemm_f6_kernel<1, false, 16>", gemm_f6_kernel<1, false, 16>);
  HIPQ_HIP(hipGetLastError());
  return HIPQ_OK;
}

/* out: the products' rows, or null and qh: the operand of a product with K = N (carved; its token is set here) */
int launch_gemm_f6_gated(const hipq_weight *wa, const hipq_weight *wm, const QActF6 *qa, int M, float *out, int64_t ldo,
                         hipStream_t s, QActF6 *qh) {
  if (!wa->gf_base || !wm->gf_base || wa->K != wm->K || wa->N != wm->N || wa->K != qa->K || M != qa->M ||
      (qh && (qh->K != wa->N || qh->M != M || wa->N % 32)))
    return fail(HIPQ_ERR_INVALID_ARGUMENT, "the gated pair has one shape and its six-bit copies");
  GatedF6 p{wa->gf_base, wm->gf_base, out, ldo, (int)wa->N, (int)((wa->N + 63) / 64), qa->word, nullptr, nullptr, 0};
  if (qh) {
    qh->token = ++f6_calls;
    p.ntiles = 4 * qh->chunks;
    p.q = qh->p, p.flags = qh->flags, p.token = qh->token;
  }
  const int mtiles = (M + BM - 1) / BM;
  /* the bounds of launch_gemm_f6 */
  const bool alone = f6_alone(mtiles, p.ntiles), few = (int64_t)mtiles * p.ntiles <= 512;
  auto go = [&](const char *name, auto kernel) {
    for (int y0 = 0, end = (p.ntiles + 7) / 8; y0 < end; y0 += MAX_Y)
      launch_kernel(name, kernel, dim3((unsigned)(8 * mtiles), (unsigned)std::min(end - y0, MAX_Y)), dim3(NT), 3 * BUF, s, p, qa->chunks,
                    ActF6{qa->p, qa->flags, qa->token}, M, y0);
  };
  if (qh) {
    if (alone)
      go("gemm_f6_gated_kernel<3, true, true>", gemm_f6_gated_kernel<3, true, true>);
    else if (few)
      go("gemm_f6_gated_kernel<3, false, true>", gemm_f6_gated_kernel<3, false, true>);
    else
      go("gemm_f6_gated_kernel<1, false, true>", gemm_f6_gated_kernel<1, false, true>);
  } else {
    if (alone)
      go("gemm_f6_gated_kernel<3, true, false>", gemm_f6_gated_kernel<3, true, false>);
    else if (few)
      go("gemm_f6_gated_kernel<3, false, false>", gemm_f6_gated_kernel<3, false, false>);
    else
      go("gemm_f6_gated_kernel<1, false, false>", gemm_f6_gated_kernel<1, false, false>);
  }
  HIPQ_HIP(hipGetLastError());
  return HIPQ_OK;
}

} // namespace hipq
