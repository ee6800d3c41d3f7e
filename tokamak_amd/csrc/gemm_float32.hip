// float32 products of many rows: C[M,N] = A[M,K] W[N,K]^T with float32 multiply-add on the matrix cores, every output the sum that
// gemm_tiled.hip describes (k ascending within pieces of 256, the pieces' sums one after the other), bit for bit:
// v_mfma_f32_16x16x4_f32 gives the bits of fmaf over its four k in ascending order.
//
// Bound by the matrix unit (142 TFLOP/s on random numbers, where the clock falls to 2.2 GHz; 157 published), which a vector instruction
// of the same wave holds up for its whole time (a lane swap a product: 140 -> 99 TFLOP/s).  So nothing but products, LDS
// reads and loads stands in the walk: both operands go from memory to LDS without passing through registers (global_load_lds,
// rows of 128 bytes, three stages of 32 k), and a lane reads each step's number by itself (piece p of a row holds four k, a lane of
// group g takes word g: 64 banks), into the register that the step's last product has just read.  One barrier a stage, in its
// middle, ahead of which the second half's operands have been read.  Two blocks share a CU and fill each other's gaps (of 32 x 32 six; 160
// x 64, whose rings are 84 KB, has the CU to itself).
//
// Tiles come in five sizes, so that the CUs' shares of a product are even (1,053 rows, 2,048 columns: 144 blocks of 128 x 128 or 544 of
// 64 x 64 for the 512 that ran at once, here 242 of 96 x 96); which, ops.float32_tile prices.  Beside tiles of 64 x 64 and 128 x
// 128 in 32x32x2 products through registers, us: 1,053 rows, weights of 4,096 x 2,048 309 -> 154, 2,048 x 2,048 139 -> 87, 12,288 x
// 2,048 597 -> 438, 2,048 x 6,144 403 -> 251; 2,048 rows, 12,288 x 2,048 871 -> 780 (132 TFLOP/s); 80 rows, 12,288 x 2,048 91 ->
// 57, 1,024 x 2,048 54 -> 30; 247 sizes of 65 to 2,048 rows 1.10 to 2.08 times as fast, others of K of 512 to 1,024 0.95 to 2.1.  A short K of
// many results is left to that kernel (ops.float32_through_registers).
#include "common.h"
#include "lds_copy.h"
#include "slots.h"

using namespace tk;

namespace {

constexpr int kPiece = 256;     // k summed before they join the total
constexpr int kStep = 32;       // k of a stage: rows of 128 bytes, a line of the caches
constexpr int kXcds = 8;        // dies, each with an L2 of its own; blocks go to them in turn
constexpr int kRing = 3;        // stages in LDS

struct Job {
  const float *a, *w;
  float* c;
  int M, N, K;
  long lda, ldw, ldc;
  int tiles_m, tiles_n;
};

// RT, CT: 16-row tiles of a wave along M and N; the block's four waves are two by two.
template <int RT, int CT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void gemm_float32_kernel(Job job) {
  constexpr int BM = 32 * RT, BN = 32 * CT, LOADS = RT + CT;
  constexpr uint32_t W_AT = kRing * BM * 128;      // in LDS: the stages of A's rows, then those of W's
  extern __shared__ __attribute__((aligned(1024))) unsigned char float32_lds[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, g = lane >> 4;
  const int wm = wave & 1, wn = wave >> 1;
  const uint32_t lds = (uint32_t)(uintptr_t)(TK_LDS unsigned char*)float32_lds;

  // Blocks go to the dies in runs, rows of a column of tiles first, so that a die's blocks share rows of both operands in its L2.
  const int total_tiles = job.tiles_m * job.tiles_n;
  const int die = (int)blockIdx.x % kXcds, nth = (int)blockIdx.x / kXcds, more = total_tiles % kXcds;
  const int at = die * (total_tiles / kXcds) + min(die, more) + nth;
  const int tn = at / job.tiles_m, tm = at - tn * job.tiles_m;
  const int m0 = tm * BM, n0 = tn * BN;

  // A lane's place in the eight rows of a load: row lane / 8, and of the row the piece of four numbers that goes to place lane % 8
  // (xored with the row so that sixteen rows' reads of a piece meet all banks).  Rows past M or N: a valid row, never stored.
  const int piece = (lane & 7) ^ ((4 * (wave & 1) + (lane >> 4)) & 7);
  uint32_t xo[RT], wo[CT];
#pragma unroll
  for (int j = 0; j < RT; ++j) xo[j] = (uint32_t)min(32 * j + 8 * wave + (lane >> 3), job.M - 1 - m0) * (uint32_t)(job.lda * 4) + piece * 16;
#pragma unroll
  for (int j = 0; j < CT; ++j) wo[j] = (uint32_t)min(32 * j + 8 * wave + (lane >> 3), job.N - 1 - n0) * (uint32_t)(job.ldw * 4) + piece * 16;
  const int stages = (job.K + kStep - 1) / kStep, ragged = job.K % kStep;
  const char* xb = reinterpret_cast<const char*>(job.a + (size_t)m0 * job.lda);
  const char* wb = reinterpret_cast<const char*>(job.w + (size_t)n0 * job.ldw);
  const uint32_t to = lds + wave * 1024;
  const auto load = [&](auto SLOT, auto J) {
    constexpr int slot = decltype(SLOT)::value, j = decltype(J)::value;
    if constexpr (j < RT) copy_to_lds_at<slot * BM * 128 + j * 4096>(to, xo[j], xb);
    else copy_to_lds_at<W_AT + slot * BN * 128 + (j - RT) * 4096>(to, wo[j - RT], wb);
  };
  // Behind the loads of a stage: on to the next, `stage`.  Of one that K ends in, what lies past K is read at the row's end.
  const auto next_load = [&](int stage) {
    xb += kStep * 4;
    wb += kStep * 4;
    if (ragged != 0 && stage == stages - 1) {
      const int past = min(0, ragged - 4 - 4 * piece) * 4;
#pragma unroll
      for (int j = 0; j < RT; ++j) xo[j] += past;
#pragma unroll
      for (int j = 0; j < CT; ++j) wo[j] += past;
    }
  };

  // Operands: a lane's number of step p (four k) of a stage is word g of row r's piece p.
  uint32_t xat[8], wat[8];
#pragma unroll
  for (int p = 0; p < 8; ++p) {
    const uint32_t in_row = ((p ^ (r >> 1)) & 7) * 16 + g * 4;
    xat[p] = lds + (wm * (RT * 16) + r) * 128 + in_row;
    wat[p] = lds + W_AT + (wn * (CT * 16) + r) * 128 + in_row;
  }
  float held[LOADS][4];       // of half a stage
  const auto read = [&](auto SLOT, auto STEP) {
    constexpr int slot = decltype(SLOT)::value, p = decltype(STEP)::value;
#pragma unroll
    for (int i = 0; i < RT; ++i) held[i][p & 3] = *reinterpret_cast<TK_LDS const float*>((uintptr_t)(xat[p] + (slot * BM * 128 + i * 2048)));
#pragma unroll
    for (int i = 0; i < CT; ++i) held[RT + i][p & 3] = *reinterpret_cast<TK_LDS const float*>((uintptr_t)(wat[p] + (slot * BN * 128 + i * 2048)));
  };
  float4v acc[RT][CT], total[RT][CT];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < CT; ++j) acc[i][j] = total[i][j] = float4v{0.f, 0.f, 0.f, 0.f};
  // Half a stage's products.  Behind a step's its operands make room for the same step's of the next half (`follows`: there is one),
  // and in the second half the stage after the next is asked for (`more`).
  constexpr int PRODS = 4 * RT * CT, APART = PRODS / LOADS;
  static_assert(APART >= 1, "half a stage has room for a stage's loads");
  const auto multiply = [&](auto H, auto NEXT_SLOT, auto LOAD_SLOT, bool follows, bool more) {
    constexpr int h = decltype(H)::value;
    each<0, PRODS>([&](auto P) {
      constexpr int p = decltype(P)::value, s = p / (RT * CT), i = p % (RT * CT) / CT, j = p % CT;
      acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(held[RT + j][s], held[i][s], acc[i][j], 0, 0, 0);
      if constexpr (p % (RT * CT) == RT * CT - 1) {
        if (follows) read(NEXT_SLOT, std::integral_constant<int, 4 * (1 - h) + s>{});
      }
      if constexpr (h == 1 && p % APART == 0 && p / APART < LOADS) {
        if (more) load(LOAD_SLOT, std::integral_constant<int, p / APART>{});
      }
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  const auto stage = [&](auto SLOT, int s) {
    constexpr int slot = decltype(SLOT)::value;
    const std::integral_constant<int, (slot + 1) % kRing> next{};
    const std::integral_constant<int, (slot + 2) % kRing> after{};
    if (s == stages - 1 && ragged != 0) {      // K ends in this one
      each<0, 8>([&](auto STEP) {
        constexpr int p = decltype(STEP)::value;
        if (4 * p >= ragged) return;
        read(SLOT, STEP);
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
          for (int j = 0; j < CT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(held[RT + j][p & 3], held[i][p & 3], acc[i][j], 0, 0, 0);
      });
      return;
    }
    const bool follows = s + 1 < stages, more = s + 2 < stages;
    multiply(std::integral_constant<int, 0>{}, SLOT, after, true, false);
    // the next stage has come, for all waves, and the slot of the one before this has been read
    if (follows) asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    multiply(std::integral_constant<int, 1>{}, next, after, follows, more);
    if (more) next_load(s + 3);
    if ((s + 1) % (kPiece / kStep) == 0 && follows) {
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < CT; ++j) {
          total[i][j] += acc[i][j];
          acc[i][j] = float4v{0.f, 0.f, 0.f, 0.f};
        }
    }
  };

  const std::integral_constant<int, 0> slot0{};
  const std::integral_constant<int, 1> slot1{};
  const std::integral_constant<int, 2> slot2{};
  xb -= kStep * 4;
  wb -= kStep * 4;
  next_load(0);
  each<0, LOADS>([&](auto J) { load(slot0, J); });
  next_load(1);
  if (stages > 1) {
    each<0, LOADS>([&](auto J) { load(slot1, J); });
    next_load(2);
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(LOADS) : "memory");
  } else {
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
  }
  __builtin_amdgcn_sched_barrier(0);
  each<0, 4>([&](auto STEP) { read(slot0, STEP); });
  for (int s = 0; s < stages; s += kRing) {
    stage(slot0, s);
    if (s + 1 < stages) stage(slot1, s + 1);
    if (s + 2 < stages) stage(slot2, s + 2);
  }
  // acc[i][j][e]: row 16 i + r of the wave, column 16 j + 4 g + e
  const bool wide = rows_take_wide_stores(job.c, job.ldc);
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    const int m = m0 + wm * (RT * 16) + 16 * i + r;
    if (m >= job.M) continue;
#pragma unroll
    for (int j = 0; j < CT; ++j) {
      const int n = n0 + wn * (CT * 16) + 16 * j + 4 * g;
      const float4v v = total[i][j] + acc[i][j];
      if (n < job.N) store_four<float>(job.c + (size_t)m * job.ldc + n, v[0], v[1], v[2], v[3], job.N - n, wide);
    }
  }
}

template <int RT, int CT>
int launch(Job job, hipStream_t stream) {
  constexpr int BM = 32 * RT, BN = 32 * CT, bytes = kRing * (BM + BN) * 128;
  static bool raised[64] = {};      // (the attribute belongs to a function on a device)
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return -1;
  if (!raised[dev]) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_float32_kernel<RT, CT>), hipFuncAttributeMaxDynamicSharedMemorySize,
                            bytes) != hipSuccess)
      return -1;
    raised[dev] = true;
  }
  job.tiles_m = (job.M + BM - 1) / BM;
  job.tiles_n = (job.N + BN - 1) / BN;
  const long total = (long)job.tiles_m * job.tiles_n;
  if (total > 0x7fffffffL) return -1;
  gemm_float32_kernel<RT, CT><<<(unsigned)total, 256, bytes, stream>>>(job);
  return launch_status();
}

}  // namespace

// C[M, N] = A[M, K] W[N, K]^T, float32.  K and the row strides multiples of 4, A's and W's rows on 16-byte borders.  rows, columns: of a
// tile, 32 RT and 32 CT.
TK_API int tk_gemm_float32(const float* A, const float* W, float* C, int M, int N, int K, long lda, long ldw, long ldc, int rows,
                           int columns, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K < 4 || K % 4 != 0 || lda % 4 != 0 || ldw % 4 != 0 || ((uintptr_t)A | (uintptr_t)W) % 16 != 0) return -1;
  // offsets within a tile's rows are 32 bits
  if (lda < 0 || ldw < 0 || lda * 4 * 160 + 128 > 0xffffffffL || ldw * 4 * 160 + 128 > 0xffffffffL) return -1;
  const Job job{A, W, C, M, N, K, lda, ldw, ldc, 0, 0};
#define TK_SHAPE(RT_, CT_) \
  if (rows == 32 * RT_ && columns == 32 * CT_) return launch<RT_, CT_>(job, stream);
  TK_SHAPE(1, 1)
  TK_SHAPE(2, 3)
  TK_SHAPE(2, 4)
  TK_SHAPE(3, 3)
  TK_SHAPE(5, 2)
#undef TK_SHAPE
  return -1;
}

TK_SLOTS(tk_gemm_float32)
