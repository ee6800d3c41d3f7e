// bf16 products of up to 128 rows (decode steps of many requests; the routes take 3 to 96): C[M,N] = A[M,K] W[N,K]^T, the weights
// streamed through LDS.
//
// What bounds it is the weights' bytes.  Weights and activations go from memory to LDS without passing through registers
// (global_load_lds): a ring of three steps of 128 k, two of which are asked for ahead, 256 contiguous bytes of a row (with 128 the memory
// behind the caches served 5 to 20 % less, which weights that fit the last cache do not show; deeper rings gain nothing); a barrier
// a step.  A wave owns 16 channels and multiplies all rows, so every weight is read from LDS once, and
// the four waves read the same activations.  Blocks start at unlike places along K and wrap around: rows lie a power of two
// apart, and blocks that ask for the same k at once meet in a few memory channels.
// K is cut into shares only as far as the CUs need blocks.
//
// Beside the form that stages weights through registers (gemm_mfma.hip) and its partial sums, each with the sums' way to their
// reader, weights from memory, us at 64 / 24 / 8 rows: 4,096 x 12,288 28.6 / 23.7 / 21.3 -> 24.7 / 20.9 / 19.2 (5.2 TB/s), 4,096 x 4,096
// 14.1 / 10.3 / 8.7 -> 11.1 / 8.7 / 7.9, 2,560 x 9,728 19.2 / 15.1 / 12.5 -> 15.6 / 12.4 / 11.3, 1,024 x 3,072 6.4 / 5.0 / 4.3 -> 6.4 / 4.7 /
// 4.0; 6,144 x 1,024 gated 9.9 / 7.7 / - -> 8.2 / 6.5 / -; 12,800 x 4,096 into bfloat16 46 / 30 / - -> 27 / 22 / -.
#include "common.h"
#include "gate.h"
#include "lds_copy.h"
#include "slots.h"

using namespace tk;

namespace {

enum { EPI_BF16, EPI_FLOAT, EPI_SILU, EPI_GELU, EPI_CLAMPED };      // the last three: gated

constexpr int kStep = 128;            // k of a step
constexpr int kRow = kStep * 2;       // bytes of a row of it

struct Job {
  const bf16_t *a, *w;
  void* c;
  int M, N, K;
  long lda, ldw, ldc, part_stride;
  int tiles, parts;
  int squared;          // C = max(., 0)^2
  float limit;          // of the clamped gate
};

constexpr int D = 3;                  // steps of the ring
constexpr int kWeightRows = 64;       // of a block

// T: tiles of 16 rows of A.
template <int T, int EPI>
__global__ __launch_bounds__(256) void gemm_flow_kernel(Job job) {
  constexpr bool GATED = EPI >= EPI_SILU;
  constexpr int OUT = GATED ? kWeightRows / 2 : kWeightRows;
  constexpr int WI = kWeightRows / 16, XI = T;      // loads of a step, of four rows each: a wave's of weights and of activations
  constexpr uint32_t WB = kWeightRows * kRow, STAGE = WB + 16 * T * kRow;
  extern __shared__ __attribute__((aligned(1024))) unsigned char flow_lds[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, g = lane >> 4;
  const uint32_t lds = (uint32_t)(uintptr_t)(TK_LDS unsigned char*)flow_lds;
  const int tile = (int)(blockIdx.x % (unsigned)job.tiles), part = (int)(blockIdx.x / (unsigned)job.tiles);
  const unsigned all = (unsigned)job.K / kStep, first = (unsigned)part * all / (unsigned)job.parts;
  const int steps = (int)((unsigned)(part + 1) * all / (unsigned)job.parts - first);
  const int n0 = tile * OUT;

  // A lane's place in the four rows of a load: row lane / 16, and of the row the piece that goes to place lane % 16 (pieces are
  // xored with the row so that sixteen rows' reads of one piece meet all banks).  Rows past M or N: a valid row, never stored.
  uint32_t wo[WI], xo[XI];
#pragma unroll
  for (int j = 0; j < WI; ++j) {
    const int row = 4 * (4 * j + wave) + (lane >> 4), piece = (lane ^ row) & 15;
    int from = min(row, job.N - 1 - n0);
    if (GATED) {      // a wave's rows: its channels' gate, then the same ones' up
      const int of = row / 16, in = row % 16;
      from = min(of * 8 + in % 8, job.N - 1 - n0) + in / 8 * job.N;
    }
    wo[j] = (uint32_t)from * (uint32_t)(job.ldw * 2) + piece * 16;
  }
#pragma unroll
  for (int j = 0; j < XI; ++j) {
    const int row = 4 * (4 * j + wave) + (lane >> 4), piece = (lane ^ row) & 15;
    xo[j] = (uint32_t)min(row, job.M - 1) * (uint32_t)(job.lda * 2) + piece * 16;
  }
  int at = (int)((unsigned)tile % (unsigned)steps);      // the step that is loaded next
  const char* wb = reinterpret_cast<const char*>(job.w + (size_t)n0 * job.ldw) + (size_t)(first + at) * kRow;
  const char* xb = reinterpret_cast<const char*>(job.a) + (size_t)(first + at) * kRow;
  uint32_t to = lds;
  const auto load = [&]() {
#pragma unroll
    for (int j = 0; j < WI; ++j) copy_to_lds<true>(to + (4 * j + wave) * 1024, wo[j], wb);
#pragma unroll
    for (int j = 0; j < XI; ++j) copy_to_lds<false>(to + WB + (4 * j + wave) * 1024, xo[j], xb);
    to = to == lds + (D - 1) * STAGE ? lds : to + STAGE;
    wb += kRow;
    xb += kRow;
    if (++at == steps) {
      at = 0;
      wb -= (size_t)steps * kRow;
      xb -= (size_t)steps * kRow;
    }
  };
#pragma unroll
  for (int t = 0; t < D - 1; ++t) load();

  float4v acc[T];
#pragma unroll
  for (int t = 0; t < T; ++t) acc[t] = float4v{0.f, 0.f, 0.f, 0.f};
  uint32_t slot = lds;
  const auto multiply = [&]() {
#pragma unroll
    for (int h = 0; h < kStep / 32; ++h) {
      const uint32_t piece = ((4 * h + g) ^ r) * 16;      // (blocks of 16 rows: the row's own bits alone)
      Frag8 wf, xf[T];
      wf.u = *reinterpret_cast<TK_LDS const u32x4*>((uintptr_t)(slot + (wave * 16 + r) * kRow + piece));
#pragma unroll
      for (int t = 0; t < T; ++t) xf[t].u = *reinterpret_cast<TK_LDS const u32x4*>((uintptr_t)(slot + WB + (t * 16 + r) * kRow + piece));
#pragma unroll
      for (int t = 0; t < T; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf.v, xf[t].v, acc[t], 0, 0, 0);
    }
    slot = slot == lds + (D - 1) * STAGE ? lds : slot + STAGE;
  };
  // Ahead of the barrier a wave's own loads of the step have come and its reads of the step before are done; behind it
  // so have all waves', and the place of the step before takes the step D - 1 ahead.
  for (int k = 0; k < steps - (D - 1); ++k) {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((D - 2) * (WI + XI)) : "memory");
    load();
    multiply();
  }
  each<0, D - 1>([&](auto I) {      // the last steps, all asked for
    if (decltype(I)::value < steps) {
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((D - 2 - decltype(I)::value) * (WI + XI)) : "memory");
      multiply();
    }
  });
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // (fewer steps than the ring has: loads nobody reads end before the LDS is given away)

  // acc[t][q]: row 4 g + q of the wave's sixteen, row 16 t + r of A
  const bool wide = EPI == EPI_FLOAT ? rows_take_wide_stores(static_cast<const float*>(job.c), job.ldc) && job.part_stride % 4 == 0
                                     : rows_take_wide_stores(static_cast<const bf16_t*>(job.c), job.ldc);
  const int n = n0 + (GATED ? wave * 8 : wave * 16) + 4 * g;
#pragma unroll
  for (int t = 0; t < T; ++t) {
    const int m = t * 16 + r;
    float v[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      v[q] = acc[t][q];
      if (GATED) v[q] = gated_value(v[q], pair32(__float_as_uint(v[q])).b(), EPI - EPI_SILU, job.limit);      // lanes 0 .. 31 hold the gate's sums, 32 .. 63 up's
      if (EPI == EPI_BF16 && job.squared) v[q] = fmaxf(v[q], 0.f) * fmaxf(v[q], 0.f);
    }
    if (m >= job.M || n >= job.N || (GATED && g > 1)) continue;
    if (EPI == EPI_FLOAT)
      store_four<float>(static_cast<float*>(job.c) + part * job.part_stride + (size_t)m * job.ldc + n, v[0], v[1], v[2], v[3], job.N - n, wide);
    else
      store_four<bf16_t>(static_cast<bf16_t*>(job.c) + (size_t)m * job.ldc + n, v[0], v[1], v[2], v[3], job.N - n, wide);
  }
}

template <int T, int EPI>
int launch(Job job, hipStream_t stream) {
  constexpr int bytes = D * (kWeightRows + 16 * T) * kRow, OUT = EPI >= EPI_SILU ? kWeightRows / 2 : kWeightRows;
  static bool raised[64] = {};      // (the attribute belongs to a function on a device)
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return -1;
  if (!raised[dev]) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_flow_kernel<T, EPI>), hipFuncAttributeMaxDynamicSharedMemorySize,
                            bytes) != hipSuccess)
      return -1;
    raised[dev] = true;
  }
  job.tiles = (job.N + OUT - 1) / OUT;
  const long blocks = (long)job.tiles * job.parts;
  if (blocks > 0x7fffffffL) return -1;
  gemm_flow_kernel<T, EPI><<<(unsigned)blocks, 256, bytes, stream>>>(job);
  return launch_status();
}

template <int T>
int pick(int mode, const Job& job, hipStream_t stream) {
  switch (mode) {
    case EPI_BF16: return launch<T, EPI_BF16>(job, stream);
    case EPI_FLOAT: return launch<T, EPI_FLOAT>(job, stream);
    case EPI_SILU: return launch<T, EPI_SILU>(job, stream);
    case EPI_GELU: return launch<T, EPI_GELU>(job, stream);
    case EPI_CLAMPED: return launch<T, EPI_CLAMPED>(job, stream);
  }
  return -1;
}

}  // namespace

// mode 0: C[M, N] bfloat16 = A W^T (squared != 0: max(., 0)^2); mode 1: C float32 [parts][M, N], part_stride elements apart: the sums
// over `parts` shares of K; modes 2, 3, 4: W = [W_gate; W_up] of 2 N rows and C[M, N] bfloat16 = act(A W_gate^T) * (A W_up^T), act
// silu, the tanh form of gelu, or the gate whose halves are clamped at `limit`.  M <= 128, K a multiple of 128, rows of A and W 16-byte
// aligned.
TK_API int tk_gemm_flow(int mode, const void* A, const void* W, void* C, int M, int N, int K, long lda, long ldw, long ldc, int parts,
                        long part_stride, int squared, float limit, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (mode < EPI_BF16 || mode > EPI_CLAMPED || M > 128 || K < kStep || K % kStep != 0 || lda % 8 != 0 || ldw % 8 != 0) return -1;
  if (((uintptr_t)A | (uintptr_t)W) & 15) return -1;
  if (parts < 1 || parts > K / kStep || (mode != EPI_FLOAT && parts != 1) || (squared != 0 && mode != EPI_BF16)) return -1;
  // offsets within a block's rows are 32 bits
  if (lda < K || ldw < K || lda * 2 * 128 > 0xffffffffL || ldw * 2 * ((mode >= EPI_SILU ? (long)N : 0) + 128) > 0xffffffffL) return -1;
  const Job job{(const bf16_t*)A, (const bf16_t*)W, C, M, N, K, lda, ldw, ldc, part_stride, 0, parts, squared, limit};
#define TK_ROWS(T_) \
  case T_: return pick<T_>(mode, job, stream);
  switch ((M + 15) / 16) {
    TK_ROWS(1)
    TK_ROWS(2)
    TK_ROWS(3)
    TK_ROWS(4)
    TK_ROWS(5)
    TK_ROWS(6)
    TK_ROWS(7)
    TK_ROWS(8)
  }
#undef TK_ROWS
  return -1;
}

TK_SLOTS(tk_gemm_flow)
