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
 * 1024 x 1024 7.6 -> 6.7, 1024 x 3072 14.1 -> 12.0; 333 of 5000 x 2048 29 -> 14; 300 of 1000 x 896 (a K that the int8
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
#include <mutex>
#include <new>

#include "gemv_device.h"

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
};

/* The sums of row tile mt and the wavefront's column tile `tile` (lane (column, g), sum r: row 8 (r / 4) + 4 g + r % 4).
 * LOOK: steps an operand is read ahead of its matrix instruction, 1 or 3 */
template <int LOOK>
__device__ __forceinline__ void f6_sums(const uint8_t *wbase, int N, int chunks, const uint8_t *act, int mt, int tile,
                                        float (&acc)[16]) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int lane = threadIdx.x & 63, i32 = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int half = mt & 1; /* of the quantizer's 64 rows */
  const rsrc_t ra = make_rsrc(act + (size_t)(mt >> 1) * chunks * CHUNK, (uint32_t)chunks * CHUNK);
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
    load_w(min(k, last), k, 0, 6);
    load_dw(min(k, last), k);
  }
  asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");

#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  v8i a[LOOK + 1], b;
  v16f D[2], P[2];
  v4h da[2]; /* the row's block scales of an even and an odd chunk */
  auto read_a = [&](int st, int at) {
    const unsigned char *p = smem + at + st * 1536;
    const v4i a0 = *(const v4i *)(p + lane * 16);
    const v2i a1 = *(const v2i *)(p + 1024 + lane * 8);
    a[st & LOOK] = v8i{a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], 0, 0};
  };
  auto read_da = [&](int k, int at) { da[k] = *(const v4h *)(smem + at + PARTS + i32 * 16 + g * 8); };
  auto start = [&](int j, int k) { /* block j of the chunk whose weights are in set k */
#pragma unroll
    for (int e = 0; e < 3; ++e) b[e] = b[3 + e] = W[k][(3 * j + e) >> 2][(3 * j + e) & 3];
    b[6] = b[7] = 0;
    /* 2^4 and 2^3 make whole numbers of the units 1/16 and 1/8 */
    D[j & 1] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a[j & LOOK], b, zero16(), 3, 2, 0, 127 + 4, 0, 127 + 3);
    /* lane (row, g) supplies the row's scales of blocks 4 g .. 4 g + 3, lane (column, g) the column's scale of block j
     * at the place of block j and zeros elsewhere */
    const uint32_t h = (uint32_t)dw[k][j >> 1] & (g == (j >> 2) ? ((j & 1) ? 0xffff0000u : 0xffffu) : 0u);
    const v2i dw2 = (j & 2) ? v2i{0, (int)h} : v2i{(int)h, 0};
    P[j & 1] = __builtin_amdgcn_mfma_f32_32x32x8f16(da[k], __builtin_bit_cast(v4h, dw2), zero16(), 0, 0, 0);
    asm volatile("" ::"v"(D[j & 1]), "v"(P[j & 1])); /* a use here: the instructions are not moved down to their sums */
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
      start((j + 1) & 7, j + 1 < 8 ? k : k ^ 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[r] = fmaf(D[j & 1][r], P[j & 1][r], acc[r]);
#pragma unroll
      for (int r = 0; r < 16; ++r) asm volatile("" : "+v"(acc[r])); /* the sums stay at this step */
      __builtin_amdgcn_sched_barrier(0);
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
  start(0, 0);
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

template <int LOOK>
__device__ __forceinline__ void f6_tile(const uint8_t *wbase, int N, int chunks, const uint8_t *act, int M, int mt, int nt,
                                        float *__restrict__ C, int64_t ldc) {
  const int lane = threadIdx.x & 63, i32 = lane & 31, g = lane >> 5;
  const int tile = nt * 4 + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  float acc[16];
  f6_sums<LOOK>(wbase, N, chunks, act, mt, tile, acc);

  const int m0 = mt * BM, n = tile * 32 + i32;
  const uint32_t off = (uint32_t)(4 * g) * (uint32_t)ldc + (uint32_t)n; /* the rest of an address is uniform */
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int m = m0 + 8 * (r >> 2) + (r & 3);
    if (m + 4 * g < M && n < N) (C + (int64_t)m * ldc)[off] = acc[r];
  }
}

/* LOOK = 3 takes 182 registers (two workgroups a CU), LOOK = 1 fits three */
template <int LOOK>
__global__ __launch_bounds__(NT, LOOK == 1 ? 3 : 2) void gemm_f6_kernel(MultiF6 mw, int chunks, const uint8_t *act, int M,
                                                                        int mtiles) {
  const int id = blockIdx.x;
  const int xcd = id & 7, qd = id >> 3;
  const int mt = qd % mtiles;
  int nt = (qd / mtiles) * 8 + xcd;
  if (nt >= mw.tile_end[3]) return; /* uniform per workgroup */
  int wi = 0;
  if (nt >= mw.tile_end[0]) wi = 1;
  if (nt >= mw.tile_end[1]) wi = 2;
  if (nt >= mw.tile_end[2]) wi = 3;
  if (wi) nt -= mw.tile_end[wi - 1];
  const uint8_t *w = wi == 0 ? mw.w[0] : wi == 1 ? mw.w[1] : wi == 2 ? mw.w[2] : mw.w[3];
  float *C = wi == 0 ? mw.C[0] : wi == 1 ? mw.C[1] : wi == 2 ? mw.C[2] : mw.C[3];
  const int64_t ldc = wi == 0 ? mw.ldc[0] : wi == 1 ? mw.ldc[1] : wi == 2 ? mw.ldc[2] : mw.ldc[3];
  const int N = wi == 0 ? mw.N[0] : wi == 1 ? mw.N[1] : wi == 2 ? mw.N[2] : mw.N[3];
  f6_tile<LOOK>(w, N, chunks, act, M, mt, nt, C, ldc);
}

/* The gated pair of an MLP: out = swiglu(act sums) * mul sums. Two wavefronts of a workgroup take 32 columns each of the
 * one matrix, the other two the same columns of the other; at the end each keeps half of its tile's rows and hands the
 * other half over through LDS. The two products never reach memory: as products and a launch of the activation 512 rows of
 * 3072 columns wrote and read 25 MB more (294 -> 273 us for four decoder layers). */
struct GatedF6 {
  const uint8_t *act, *mul;
  float *out;
  int64_t ldo;
  int N, ntiles; /* columns, workgroup columns of 64 */
};
template <int LOOK>
__device__ __forceinline__ void f6_gated_tile(const GatedF6 &p, int chunks, const uint8_t *act, int M, int mt, int nt) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int lane = threadIdx.x & 63, i32 = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const bool second = wave >= 2;
  const int tile = nt * 2 + (wave & 1);
  float acc[16];
  f6_sums<LOOK>(second ? p.mul : p.act, p.N, chunks, act, mt, tile, acc);

  __syncthreads(); /* no wavefront reads or fills its row buffers any more */
  float *mine = (float *)smem + wave * 512, *other = (float *)smem + (wave ^ 2) * 512;
#pragma unroll
  for (int r = 0; r < 8; ++r) mine[r * 64 + lane] = second ? acc[r] : acc[8 + r];
  __syncthreads();
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
template <int LOOK>
__global__ __launch_bounds__(NT, LOOK == 1 ? 3 : 2) void gemm_f6_gated_kernel(GatedF6 p, int chunks, const uint8_t *act, int M,
                                                                              int mtiles) {
  const int id = blockIdx.x;
  const int xcd = id & 7, qd = id >> 3;
  const int mt = qd % mtiles, nt = (qd / mtiles) * 8 + xcd;
  if (nt < p.ntiles) f6_gated_tile<LOOK>(p, chunks, act, M, mt, nt); /* uniform per workgroup */
}

/* ---- the copy of a weight in operand order ---- */

/* thread = lane (column, g) of one (tile, chunk, block): its sixteen weights as 96 bits, dwords 3 j .. 3 j + 2 of the
 * lane's 24, and the block's scale */
__global__ __launch_bounds__(256) void f6_weights_kernel(const uint8_t *__restrict__ qs, const uint16_t *__restrict__ d, int N,
                                                         int nb /* blocks a row */, int chunks, int64_t threads,
                                                         uint8_t *__restrict__ out) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= threads) return;
  const int lane = (int)(t & 63), j = (int)((t >> 6) & 7), g = lane >> 5, i32 = lane & 31;
  const int64_t tc = t >> 9; /* tile * chunks + chunk */
  const int c = (int)(tc % chunks);
  const int64_t n = tc / chunks * 32 + i32;
  uint8_t *dst = out + tc * WTILE;
  const int b = c * 8 + j;
  const bool in = n < N && b < nb;
  uint4 x = make_uint4(0x88888888u, 0x88888888u, 0x88888888u, 0x88888888u); /* weights of zero */
  if (in) x = *(const uint4 *)(qs + (n * nb + b) * 16);
  const uint32_t x4[4] = {x.x, x.y, x.z, x.w};
  uint32_t w[3] = {0, 0, 0};
#pragma unroll
  for (int i = 0; i < 16; ++i) { /* byte i of a block = elements i (low nibble) and i + 16 */
    const int v = (int)((x4[i >> 2] >> (8 * (i & 3) + 4 * g)) & 15u) - 8;
    const uint32_t code = v < 0 ? 0x20u | (uint32_t)(-v) : (uint32_t)v; /* fp6 codes up to 15 are the number itself */
    const int bit = 6 * i;
    w[bit >> 5] |= code << (bit & 31);
    if ((bit & 31) > 26) w[(bit >> 5) + 1] |= code >> (32 - (bit & 31));
  }
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const int k = 3 * j + i;
    *(uint32_t *)(dst + (k >> 2) * 1024 + lane * 16 + (k & 3) * 4) = w[i];
  }
  if (!g) *(uint16_t *)(dst + 6144 + i32 * 16 + j * 2) = in ? d[n * nb + b] : (uint16_t)0;
}

} // namespace

namespace hipq {

/* ---- who may read a copy ----
 * A copy is made on the stream of the product that asks for it, in front of that product, and nothing waits. Until it
 * is known to be complete it is PENDING, and only the stream it was made on may read it; a product on another stream
 * takes the kernels that read the weight as stored (the same bits). Complete is what the page-locked word of its batch
 * says, which the quantizer behind the copies sets: a plain read, so also a call that is being captured into a graph,
 * where events may not be queried, finds out. A graph may be launched on any stream, so a captured product reads
 * complete copies only.
 * The same stream is known by its handle alone, and one handle can stand for two streams (hipStreamPerThread; a stream
 * made after another was destroyed): the event of the batch orders those. */
struct F6Batch {
  uint32_t *word, *word_dev;
  hipEvent_t ev;
  hipStream_t s;
  int refs; /* PENDING weights that point here */
  F6Batch *next;
};

namespace {
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

/* *ready: what is enqueued on s next may read the copies of the weights. Missing ones are made where may_make and the
 * stream is not being captured; the caller then hands *word to the quantizer it launches behind them. */
int f6_copies(int count, const hipq_weight *const *cw, hipStream_t s, bool may_make, bool *ready, uint32_t **word) {
  *ready = false;
  *word = nullptr;
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
    if (w[i]->gf_state == F6_NONE) {
      if (w[i]->dtype != HIPQ_Q4_0 || w[i]->expert_tiles)
        return fail(HIPQ_ERR_INVALID_ARGUMENT, "only Q4_0 weights in the plane layout have a six-bit copy");
      ++missing;
    } else if (!complete(w[i], spins)) {
      F6Batch *b = w[i]->gf_batch;
      if (capturing || b->s != s) return HIPQ_OK;
      if (b != behind) HIPQ_HIP(hipStreamWaitEvent(s, b->ev, 0));
      behind = b;
    }
  }
  if (missing) {
    if (!may_make || capturing) return HIPQ_OK;
    F6Batch *b = nullptr;
    if (int rc = batch_get(s, &b)) return rc;
    int made = 0, rc = HIPQ_OK;
    hipq_weight *fresh[64];
    for (int i = 0; i < count && !rc && made < 64; ++i) {
      hipq_weight *x = w[i];
      if (x->gf_state != F6_NONE || x->gf_base) continue; /* a weight may stand in the list twice */
      const int nb = (int)(x->K / 32), chunks = (nb + 7) / 8;
      const int64_t tiles = (x->N + 31) / 32, threads = tiles * chunks * 512;
      const size_t bytes = (size_t)tiles * chunks * F6_WTILE;
      uint8_t *p = nullptr;
      hipError_t e = hipMalloc((void **)&p, bytes);
      if (e != hipSuccess) {
        rc = fail(HIPQ_ERR_OUT_OF_MEMORY, "six-bit copy of %zu bytes: %s", bytes, hipGetErrorString(e));
        break;
      }
      x->gf_base = p;
      fresh[made++] = x;
      launch_kernel("f6_weights_kernel", f6_weights_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s, x->qs, x->d,
                    (int)x->N, nb, chunks, threads, p);
      if ((e = hipGetLastError()) != hipSuccess) rc = fail(HIPQ_ERR_RUNTIME, "six-bit copy: %s", hipGetErrorString(e));
    }
    if (!rc) {
      const hipError_t e = hipEventRecord(b->ev, s);
      if (e != hipSuccess) rc = fail(HIPQ_ERR_RUNTIME, "six-bit copy: %s", hipGetErrorString(e));
    }
    if (rc) {
      if (made) (void)hipStreamSynchronize(s);
      for (int i = 0; i < made; ++i) {
        (void)hipFree(fresh[i]->gf_base);
        fresh[i]->gf_base = nullptr;
      }
      batch_idle(b);
      return rc;
    }
    for (int i = 0; i < made; ++i) {
      fresh[i]->gf_batch = b;
      __atomic_store_n(&fresh[i]->gf_state, F6_PENDING, __ATOMIC_RELEASE);
    }
    b->refs = made;
    *word = b->word_dev;
  }
  *ready = true;
  return HIPQ_OK;
}

void f6_release(hipq_weight *w) {
  std::lock_guard<std::mutex> lk(f6_mu);
  batch_drop(w);
  if (w->gf_base) (void)hipFree(w->gf_base);
  w->gf_base = nullptr;
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
}

int launch_gemm_f6(int count, const hipq_weight *const *w, const QActF6 *qa, int M, float *const *C, const int64_t *ldc,
                   hipStream_t s) {
  if (count < 1 || count > 4) return fail(HIPQ_ERR_INVALID_ARGUMENT, "1 to 4 weights per launch, got %d", count);
  MultiF6 mw;
  int tiles = 0;
  for (int i = 0; i < 4; ++i) {
    const int k = i < count ? i : count - 1;
    if (!w[k]->gf_base || w[k]->K != w[0]->K || w[k]->K != qa->K || M != qa->M)
      return fail(HIPQ_ERR_INVALID_ARGUMENT, "the weights of one launch share K and have their six-bit copy");
    mw.w[i] = w[k]->gf_base;
    mw.N[i] = (int)w[k]->N;
    mw.C[i] = C[k];
    mw.ldc[i] = ldc[k];
    if (i < count) tiles += (int)((w[k]->N + BN - 1) / BN);
    mw.tile_end[i] = tiles; /* unused entries repeat the total: no workgroup lands in them */
  }
  const int mtiles = (M + BM - 1) / BM;
  const dim3 grid((unsigned)(mtiles * ((tiles + 7) / 8) * 8));
  /* up to two workgroups a CU: the deeper read-ahead (512 rows of 1024 x 3072 13.1 -> 12.0 us, 1024 x 1024 7.5 -> 6.7);
   * beyond, three workgroups a CU cover the reads (512 of 12288 x 4096 67 -> 62 us) */
  if ((int64_t)mtiles * tiles <= 512)
    launch_kernel("gemm_f6_kernel<3>", gemm_f6_kernel<3>, grid, dim3(NT), 3 * BUF, s, mw, qa->chunks, (const uint8_t *)qa->p, M,
                  mtiles);
  else
    launch_kernel("gemm_f6_kernel<1>", gemm_f6_kernel<1>, grid, dim3(NT), 3 * BUF, s, mw, qa->chunks, (const uint8_t *)qa->p, M,
                  mtiles);
  HIPQ_HIP(hipGetLastError());
  return HIPQ_OK;
}

int launch_gemm_f6_gated(const hipq_weight *wa, const hipq_weight *wm, const QActF6 *qa, int M, float *out, int64_t ldo,
                         hipStream_t s) {
  if (!wa->gf_base || !wm->gf_base || wa->K != wm->K || wa->N != wm->N || wa->K != qa->K || M != qa->M)
    return fail(HIPQ_ERR_INVALID_ARGUMENT, "the gated pair has one shape and its six-bit copies");
  const GatedF6 p{wa->gf_base, wm->gf_base, out, ldo, (int)wa->N, (int)((wa->N + 63) / 64)};
  const int mtiles = (M + BM - 1) / BM;
  const dim3 grid((unsigned)(mtiles * ((p.ntiles + 7) / 8) * 8));
  /* the bound of launch_gemm_f6 */
  if ((int64_t)mtiles * p.ntiles <= 512)
    launch_kernel("gemm_f6_gated_kernel<3>", gemm_f6_gated_kernel<3>, grid, dim3(NT), 3 * BUF, s, p, qa->chunks,
                  (const uint8_t *)qa->p, M, mtiles);
  else
    launch_kernel("gemm_f6_gated_kernel<1>", gemm_f6_gated_kernel<1>, grid, dim3(NT), 3 * BUF, s, p, qa->chunks,
                  (const uint8_t *)qa->p, M, mtiles);
  HIPQ_HIP(hipGetLastError());
  return HIPQ_OK;
}

} // namespace hipq
