// bf16 products of many rows (prompt portions) with float32 sums: C[M,N] = A[M,K] W[N,K]^T in shares of K as partial sums, or
// gated (W = [gate; up], C = act(A gate^T) * (A up^T)) with no array of gate and up in between.
//
// A block of four waves owns a tile, a wave a quarter of it, all of whose sums stay in accumulation registers (a 256 x 256 tile
// takes half of a CU's registers, so a wave has its SIMD to itself).  Both operands go from memory to LDS without passing
// through registers (global_load_lds), whole 128-byte lines of a row, weights three steps of 64 k deep and activations two (all
// 160 KB at 256 x 256): a step's loads have two steps' or one step's products to come.  In a wave a product, an LDS read
// of the half step after it or one of the loads follow one another at fixed distances, so that the matrix unit never waits for
// an instruction; one barrier a step, ahead of which the next half's operands have been read.  16x16x32 products: half of the
// accumulators' traffic of 32x32x16, which at full load let the clock rise 1.68 -> 1.87 GHz (the card's power bounds large
// products: 24,576 x 4,096 at 2,048 rows of zeros takes 250 us where random numbers take 285).  Rows of 64-byte pieces
// (steps of 32 k) fetched every line twice: 1,470 cycles a 32 k where these take 1,340, and instructions in bunches
// between products another 100.
//
// Beside the library's fastest candidate and the gate's kernel, gated, us: 24,576 x 4,096 at 256 / 512 / 1,024 / 2,048 rows 67 / 98 /
// 253 / 317, here 62 / 90 / 170 / 288 (1.43 PFLOP/s); 19,456 x 2,560 at 512 / 1,024 / 2,048 rows 96 / 148 / 213, here 57 / 99 / 179;
// 6,144 x 1,024 at 256 / 1,024 / 2,048 rows 15.1 / 33.1 / 35.5, here 11.9 / 18.5 / 28.6.  In shares of K, with what the sums cost
// their reader, beside the library's first choice: 4,096 x 12,288 at 200 / 512 / 1,024 rows 45 / 75 / 106, here 37 / 55 / 93; 2,560 x
// 9,728 32 / 46 / 62, here 26 / 36 / 53; 5,120 x 17,408 226 / 168 / 246, here 57 / 90 / 149.
//
// Several products of one shape (a time mix's four projections) are one list of tiles: one alone is 64 to 256 tiles, a part of a round
// or one that ends unevenly.  Four of 4,096 x 4,096 at 129 / 512 / 1,000 / 2,048 rows, us: the library's launches 91 / 123 / 164 / 241, here 44
// / 59 / 96 / 184 (1.50 PFLOP/s).
#include "common.h"
#include "gate.h"
#include "lds_copy.h"
#include "slots.h"

using namespace tk;

namespace {

enum { EPI_PARTS, EPI_SILU, EPI_CLAMPED, EPI_GELU, EPI_SEVERAL };     // the three in the middle: gated; SEVERAL: independent products, bfloat16

constexpr int kCus = 256;       // blocks that run at once
constexpr int kXcds = 8;        // dies, each with an L2 of its own; blocks go to them in turn
constexpr int kStep = 64;       // k of a step: rows of 128 bytes, a line of the caches

struct Job {
  const bf16_t *a, *w;
  void* c;
  int M, N, K;
  long lda, ldw, ldc, part_stride;
  int tiles_m, tiles_n, parts;      // parts: shares of K, or products (EPI_SEVERAL)
  float limit;                      // of the clamped gate
  long a_next, w_next;              // EPI_SEVERAL: from a product's operands to the next one's (part_stride: of the results)
};

template <int EPI>
__device__ __forceinline__ float gated(float z, float u, float limit) {
  if (EPI == EPI_GELU) return gelu_by_exp(z, u);
  return gated_value(z, u, EPI == EPI_SILU ? 0 : 2, limit);
}

// The same number, which the compiler cannot follow: what is computed from it is computed where it stands and not kept in
// registers over the loop around it (the loop has none to spare).
__device__ __forceinline__ int here(int v) {
  asm volatile("" : "+v"(v));
  return v;
}

// Where a wave's loads of one operand stand: a unit, the step of it that is loaded next, its ring slot.
struct Cursor {
  int unit, step, steps;
  uint32_t slot;
  const char* base;
};

// Blocks that a CU holds at once: one whose sums take half of the registers, or two small ones.
constexpr int blocks_a_cu(int mt, int nt) { return mt * nt <= 4 ? 2 : 1; }

template <int MT, int NT, int EPI>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(blocks_a_cu(MT, NT), blocks_a_cu(MT, NT)))) void gemm_many_kernel(Job job) {
  constexpr int kSlots = kCus * blocks_a_cu(MT, NT);      // blocks that run at once
  constexpr bool GATED = EPI == EPI_SILU || EPI == EPI_CLAMPED || EPI == EPI_GELU, SEVERAL = EPI == EPI_SEVERAL;
  constexpr int BM = 64 * MT, BN = 64 * NT, OUT = GATED ? BN / 2 : BN;   // OUT: output channels of a tile
  constexpr uint32_t WB = BN * 128, XB = BM * 128, WRING = 3 * WB, XRING = 2 * XB;
  extern __shared__ __attribute__((aligned(1024))) unsigned char many_lds[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave & 1, wn = wave >> 1, r = lane & 15, g = lane >> 4;
  const uint32_t lds = (uint32_t)(uintptr_t)(TK_LDS unsigned char*)many_lds, lds_wave = lds + wave * 1024;
  const int tiles = job.tiles_m * job.tiles_n, total = tiles * job.parts, all_steps = job.K / kStep;

  // A round's units go to the dies in runs, so that a die's blocks share rows of both operands in its L2.
  const auto place = [&](int u, int& tm, int& tn, int& part) {
    const int round = u / kSlots, in = u % kSlots, left = min(kSlots, total - round * kSlots);
    const int die = in % kXcds, nth = in / kXcds, more = left % kXcds, least = left / kXcds;
    const int at = round * kSlots + die * least + min(die, more) + nth;
    part = at / tiles;
    const int tile = at - part * tiles;
    tn = tile / job.tiles_m;
    tm = tile - tn * job.tiles_m;
  };
  uint32_t xo[2 * MT], wo[2 * NT];
  const auto begin = [&](Cursor& c, int part, const bf16_t* rows, long next) {
    const int first = SEVERAL ? 0 : (int)((unsigned)(part * all_steps) / (unsigned)job.parts);
    c.steps = SEVERAL ? all_steps : (int)((unsigned)((part + 1) * all_steps) / (unsigned)job.parts) - first;
    c.step = 0;
    c.base = reinterpret_cast<const char*>(rows + (SEVERAL ? part * next : (long)first * kStep));
  };
  const auto aim_x = [&](Cursor& c) {
    int tm, tn, part;
    place(c.unit, tm, tn, part);
    const int at = here(lane), piece = (at & 7) ^ ((4 * (wave & 1) + (at >> 4)) & 7), m0 = tm * BM;
#pragma unroll
    for (int j = 0; j < 2 * MT; ++j)
      xo[j] = (uint32_t)min(8 * (4 * j + wave) + (at >> 3), job.M - 1 - m0) * (uint32_t)(job.lda * 2) + piece * 16;
    begin(c, part, job.a + (size_t)m0 * job.lda, job.a_next);
  };
  const auto aim_w = [&](Cursor& c) {
    int tm, tn, part;
    place(c.unit, tm, tn, part);
    const int at = here(lane), piece = (at & 7) ^ ((2 * wave + ((at >> 4) & 1)) & 7), n0 = tn * OUT;
#pragma unroll
    for (int j = 0; j < 2 * NT; ++j) {
      const int row = 8 * (4 * j + wave) + (at >> 3);
      int from = min(row, job.N - 1 - n0);
      if (GATED) {      // each half of the tile: the gate's channels, then the same ones' of up
        const int half = row / (32 * NT), in = row % (32 * NT);
        from = min(half * (16 * NT) + in % (16 * NT), job.N - 1 - n0) + in / (16 * NT) * job.N;
      }
      wo[j] = (uint32_t)from * (uint32_t)(job.ldw * 2) + piece * 16;
    }
    begin(c, part, job.w + (size_t)n0 * job.ldw, job.w_next);
  };
  const auto next_w = [](uint32_t s) { return s == WRING - WB ? 0u : s + WB; };
  const auto next_x = [](uint32_t s) { return s == WRING ? WRING + XB : WRING; };
  const auto next_unit = [&](Cursor& c, const auto& aim) {      // (behind the last unit: that one again, which nobody reads)
    if (++c.step == c.steps) {
      if (c.unit + (int)gridDim.x < total) c.unit += gridDim.x;
      aim(c);
    }
  };
  Cursor cx{(int)blockIdx.x, 0, 0, WRING, nullptr}, cw{(int)blockIdx.x, 0, 0, 0, nullptr};
  aim_x(cx);
  aim_w(cw);
  const auto load_x = [&](auto j) { copy_to_lds_at<decltype(j)::value * 4096>(lds_wave + cx.slot, xo[decltype(j)::value], cx.base); };
  const auto load_w = [&](auto j) { copy_to_lds_at<decltype(j)::value * 4096>(lds_wave + cw.slot, wo[decltype(j)::value], cw.base); };
  constexpr int READS = 2 * (MT + NT), PRODS = 4 * MT * NT;      // of half a step
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    each<0, 2 * NT>(load_w);
    cw.slot = next_w(cw.slot);
    cw.base += 128;
    next_unit(cw, aim_w);
    each<0, 2 * MT>(load_x);
    cx.slot = next_x(cx.slot);
    cx.base += 128;
    next_unit(cx, aim_x);
  }
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(READS) : "memory");
  __builtin_amdgcn_sched_barrier(0);

  // Operands in LDS: rows of eight 16-byte pieces, xored with the row so that sixteen rows' reads of a piece meet all banks.  A
  // pair of blocks of 16 channels has row 4 a + q of its block e as channel 8 a + 4 e + q: a lane's results are eight channels in a row.
  uint32_t xat[2], wat[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    xat[h] = lds + (wm * (MT * 32) + r) * 128 + (((4 * h + g) ^ (r >> 1)) & 7) * 16;
    wat[h] = lds + (wn * (NT * 32) + 8 * (r >> 2) + (r & 3)) * 128 + (((4 * h + g) ^ (2 * (r >> 2) + ((r >> 1) & 1))) & 7) * 16;
  }
  uint32_t ws = 0, xs = WRING;      // slots of the step that is read
  Frag8 wf[2][2 * NT], xf[2][2 * MT];
  const auto read = [&](int set, int h, int i) {
    if (i < 2 * NT) wf[set][i].u = *reinterpret_cast<TK_LDS const u32x4*>((uintptr_t)(wat[h] + ws + (i >> 1) * 4096 + (i & 1) * 512));
    else xf[set][i - 2 * NT].u = *reinterpret_cast<TK_LDS const u32x4*>((uintptr_t)(xat[h] + xs + (i - 2 * NT) * 2048));
  };
#pragma unroll
  for (int i = 0; i < READS; ++i) read(0, 0, i);

  for (int unit = blockIdx.x; unit < total; unit += gridDim.x) {
    int tm, tn, part;
    place(unit, tm, tn, part);
    const int steps = SEVERAL ? all_steps
                              : (int)((unsigned)((part + 1) * all_steps) / (unsigned)job.parts) - (int)((unsigned)(part * all_steps) / (unsigned)job.parts);
    float4v acc[2 * NT][2 * MT];
#pragma unroll
    for (int i = 0; i < 2 * NT; ++i)
#pragma unroll
      for (int j = 0; j < 2 * MT; ++j) acc[i][j] = float4v{0.f, 0.f, 0.f, 0.f};
    constexpr int TAIL = PRODS / 4, READ_EVERY = (PRODS - TAIL) / READS, W_EVERY = (PRODS - TAIL) / (2 * NT), X_EVERY = (PRODS - TAIL) / (2 * MT);
    static_assert(READ_EVERY >= 1 && W_EVERY >= 1 && X_EVERY >= 1, "a half step has room for its reads and loads");
    for (int k = 0; k < steps; ++k) {
      // The step's first half; its second half's operands are read, the weights of the step after the next two asked for.
      each<0, PRODS>([&](auto P) {
        constexpr int p = decltype(P)::value, i = p / (2 * MT), j = p % (2 * MT);
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[0][i].v, xf[0][j].v, acc[i][j], 0, 0, 0);
        if constexpr (p % READ_EVERY == 0 && p / READ_EVERY < READS) read(1, 1, p / READ_EVERY);
        if constexpr (p % W_EVERY == W_EVERY - 1 && p / W_EVERY < 2 * NT) load_w(std::integral_constant<int, p / W_EVERY>{});
        if constexpr (p == PRODS - TAIL) cw.slot = next_w(cw.slot);
        if constexpr (p == PRODS - TAIL * 3 / 4) cw.base += 128;
        if constexpr (p == PRODS - TAIL / 2) next_unit(cw, aim_w);
        __builtin_amdgcn_sched_barrier(0);
      });
      // All waves have read this step, and all of the next one has come: its loads are older than the last 2 NT.
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(2 * NT) : "memory");
      __builtin_amdgcn_sched_barrier(0);
      ws = next_w(ws);
      xs = next_x(xs);
      each<0, PRODS>([&](auto P) {
        constexpr int p = decltype(P)::value, i = p / (2 * MT), j = p % (2 * MT);
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[1][i].v, xf[1][j].v, acc[i][j], 0, 0, 0);
        if constexpr (p % READ_EVERY == 0 && p / READ_EVERY < READS) read(0, 0, p / READ_EVERY);
        if constexpr (p % X_EVERY == X_EVERY - 1 && p / X_EVERY < 2 * MT) load_x(std::integral_constant<int, p / X_EVERY>{});
        if constexpr (p == PRODS - TAIL) cx.slot = next_x(cx.slot);
        if constexpr (p == PRODS - TAIL * 3 / 4) cx.base += 128;
        if constexpr (p == PRODS - TAIL / 2) next_unit(cx, aim_x);
        __builtin_amdgcn_sched_barrier(0);
      });
    }
    // (in accumulation registers over the whole walk: vector registers are short, and some would be moved there and back)
#pragma unroll
    for (int i = 0; i < 2 * NT; ++i)
#pragma unroll
      for (int j = 0; j < 2 * MT; ++j) asm volatile("" : "+a"(acc[i][j]));
    const int at = here(lane), first_m = tm * BM + wm * (MT * 32) + (at & 15), first_n = tn * OUT + wn * (OUT / 2) + 8 * (at >> 4);
    // acc[2 b + e][j][q]: channel 32 b + 8 g + 4 e + q of the wave, row 16 j + r
#pragma unroll
    for (int j = 0; j < 2 * MT; ++j) {
      const int m = first_m + j * 16;
#pragma unroll
      for (int b = 0; b < (GATED ? NT / 2 : NT); ++b) {
        const int n = first_n + 32 * b;
        float v[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          v[q] = acc[2 * b + (q >> 2)][j][q & 3];
          if (GATED) v[q] = gated<EPI>(v[q], acc[(NT + 2 * b + (q >> 2)) % (2 * NT)][j][q & 3], job.limit);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (m >= job.M || n >= job.N) continue;      // (N is a multiple of 8)
        if (EPI == EPI_PARTS) {
          float* dst = static_cast<float*>(job.c) + part * job.part_stride + (size_t)m * job.ldc + n;
          *reinterpret_cast<float4*>(dst) = make_float4(v[0], v[1], v[2], v[3]);
          *reinterpret_cast<float4*>(dst + 4) = make_float4(v[4], v[5], v[6], v[7]);
        } else {
          *reinterpret_cast<uint4*>(static_cast<bf16_t*>(job.c) + (SEVERAL ? part * job.part_stride : 0) + (size_t)m * job.ldc + n) =
              make_uint4(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7]));
        }
      }
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // (the loads behind the last unit's end before the block's LDS is given away)
}

template <int MT, int NT, int EPI>
int launch(Job job, hipStream_t stream) {
  constexpr int BM = 64 * MT, OUT = EPI == EPI_PARTS || EPI == EPI_SEVERAL ? 64 * NT : 32 * NT, bytes = (3 * NT + 2 * MT) * 64 * 128;
  static bool raised[64] = {};      // (the attribute belongs to a function on a device)
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return -1;
  if (!raised[dev]) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_many_kernel<MT, NT, EPI>), hipFuncAttributeMaxDynamicSharedMemorySize,
                            bytes) != hipSuccess)
      return -1;
    raised[dev] = true;
  }
  job.tiles_m = (job.M + BM - 1) / BM;
  job.tiles_n = (job.N + OUT - 1) / OUT;
  const long total = (long)job.tiles_m * job.tiles_n * job.parts;
  constexpr int slots = kCus * blocks_a_cu(MT, NT);
  if (total > 0x7fffffffL - slots) return -1;
  gemm_many_kernel<MT, NT, EPI><<<(unsigned)(total < slots ? total : slots), 256, bytes, stream>>>(job);
  return launch_status();
}

}  // namespace

// mode 0: C float32 [parts][M, N], part_stride elements apart: the sums over `parts` shares of K; modes 1 to 3: W = [W_gate;
// W_up] of 2 N rows and C[M, N] bfloat16 = act(A W_gate^T) * (A W_up^T), act silu, (2) the gate whose halves are clamped at
// `limit` or (3) the tanh form of gelu.  rows, columns: a tile's rows of A and of W (256 x 256, 128 x 256, 256 x 128, 128 x 128).  K a multiple of 64, N of 8;
// rows of all operands 16-byte aligned.
TK_API int tk_gemm_many(int mode, const void* A, const void* W, void* C, int M, int N, int K, long lda, long ldw, long ldc,
                        int parts, long part_stride, float limit, int rows, int columns, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  const bool gate = mode >= EPI_SILU;
  if (mode < 0 || mode > EPI_GELU) return -1;
  if (K < kStep || K % kStep != 0 || N % 8 != 0 || lda % 8 != 0 || ldw % 8 != 0 || ldc % 8 != 0 || part_stride % 4 != 0) return -1;
  if (((uintptr_t)A | (uintptr_t)W | (uintptr_t)C) & 15) return -1;
  if (parts < 1 || parts > K / kStep || (mode != EPI_PARTS && parts != 1)) return -1;
  // offsets within a tile are 32 bits
  if (lda < K || ldw < K || lda * 2 * 256 > 0xffffffffL || ldw * 2 * ((gate ? (long)N : 0) + 256) > 0xffffffffL) return -1;
  const Job job{(const bf16_t*)A, (const bf16_t*)W, C, M, N, K, lda, ldw, ldc, part_stride, 0, 0, parts, limit, 0, 0};
#define TK_SHAPE(MT_, NT_)                                                             \
  if (rows == 64 * MT_ && columns == 64 * NT_) {                                       \
    if (mode == EPI_PARTS) return launch<MT_, NT_, EPI_PARTS>(job, stream);            \
    if (mode == EPI_SILU) return launch<MT_, NT_, EPI_SILU>(job, stream);              \
    if (mode == EPI_GELU) return launch<MT_, NT_, EPI_GELU>(job, stream);              \
    return launch<MT_, NT_, EPI_CLAMPED>(job, stream);                                 \
  }
  TK_SHAPE(4, 4)
  TK_SHAPE(2, 4)
  TK_SHAPE(4, 2)
  TK_SHAPE(2, 2)
#undef TK_SHAPE
  return -1;
}

// `count` products of one shape: C_i[M, N] bfloat16 = A_i W_i^T, the operands and results a_next, w_next and c_next numbers apart.
TK_API int tk_gemm_several(const void* A, const void* W, void* C, int M, int N, int K, long lda, long ldw, long ldc, int count, long a_next,
                           long w_next, long c_next, int rows, int columns, hipStream_t stream) {
  if (M <= 0 || N <= 0 || count <= 0) return 0;
  if (K < kStep || K % kStep != 0 || N % 8 != 0 || lda % 8 != 0 || ldw % 8 != 0 || ldc % 8 != 0) return -1;
  if ((((uintptr_t)A | (uintptr_t)W | (uintptr_t)C) & 15) || a_next % 8 != 0 || w_next % 8 != 0 || c_next % 8 != 0 || count > 64) return -1;
  // offsets within a tile are 32 bits
  if (lda < K || ldw < K || lda * 2 * 256 > 0xffffffffL || ldw * 2 * 256 > 0xffffffffL) return -1;
  const Job job{(const bf16_t*)A, (const bf16_t*)W, C, M, N, K, lda, ldw, ldc, c_next, 0, 0, count, 0.f, a_next, w_next};
#define TK_SHAPE(MT_, NT_) \
  if (rows == 64 * MT_ && columns == 64 * NT_) return launch<MT_, NT_, EPI_SEVERAL>(job, stream);
  TK_SHAPE(4, 4)
  TK_SHAPE(2, 4)
  TK_SHAPE(4, 2)
  TK_SHAPE(2, 2)
#undef TK_SHAPE
  return -1;
}

TK_SLOTS(tk_gemm_many)
TK_SLOTS(tk_gemm_several)
