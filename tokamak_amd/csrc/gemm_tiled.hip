// C[M,N] = A[M,K] * W[N,K]^T with float32 multiply-add and float32 accumulation
// for any M, N, K.  It is the true 32-bit matrix product of the float32 path
// (no reduced-precision matrix mode), and also accepts bf16 inputs.  Every
// output element is summed in one fixed order, whichever kernel below does it, so a row's
// result does not depend on which other rows are in the batch: k ascending within pieces of
// kPiece, whose sums are added to the total one after the other.  The two levels
// keep the rounding error of a sum over K terms near sqrt(kPiece) + sqrt(K / kPiece)
// units instead of sqrt(K) (K is 25,600 in the widest feed-forward).
#include "common.h"
#include "slots.h"

using namespace tk;

constexpr int BK = 16, PAD = 4;   // of gemm_tiled_kernel
constexpr int kPiece = 256;  // k values summed before they join the total (a multiple of BK)

// A block of 256 threads owns 64H x 64H outputs (H = 1 or 2); thread (ty, tx) of 16 x 16 owns
// rows ty*4.. (and 64 + ty*4..) and columns tx*4.. (and 64 + tx*4..): 4H x 4H outputs, per k
// 2H 16-byte LDS reads for 16 H^2 multiply-adds.  The next 16 k are fetched into registers while
// the current ones are multiplied.  H = 2 is the fast one (65 against 37 TFLOP/s on 2,048 rows);
// H = 1 has four times the blocks, for products too small to fill the GPU otherwise.
template <typename TI, typename TO, int H>
__global__ __launch_bounds__(256) void gemm_tiled_kernel(const TI* __restrict__ A,
                                                         const TI* __restrict__ W,
                                                         TO* __restrict__ C, int M, int N, int K,
                                                         long lda, long ldw, long ldc) {
  constexpr int BM = 64 * H, BN = 64 * H, R = 4 * H;
  __shared__ __attribute__((aligned(16))) float As[BK][BM + PAD];
  __shared__ __attribute__((aligned(16))) float Ws[BK][BN + PAD];
  const int tid = threadIdx.x;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  const int ty = tid / 16, tx = tid % 16;
  const int lrow = tid / 4, lk = (tid % 4) * 4;   // loader: rows lrow (and lrow + 64), four k from lk

  float acc[R][R], total[R][R];
#pragma unroll
  for (int i = 0; i < R; ++i)
#pragma unroll
    for (int j = 0; j < R; ++j) acc[i][j] = total[i][j] = 0.f;

  float ar[H][4], wr[H][4];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int h = 0; h < H; ++h) {
      const int m = m0 + lrow + 64 * h, n = n0 + lrow + 64 * h;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int k = k0 + lk + i;
        ar[h][i] = (m < M && k < K) ? Elem<TI>::load(A + (size_t)m * lda + k) : 0.f;
        wr[h][i] = (n < N && k < K) ? Elem<TI>::load(W + (size_t)n * ldw + k) : 0.f;
      }
    }
  };
  fetch(0);
  for (int k0 = 0; k0 < K; k0 += BK) {
    if (k0 > 0 && k0 % kPiece == 0) {
#pragma unroll
      for (int i = 0; i < R; ++i)
#pragma unroll
        for (int j = 0; j < R; ++j) {
          total[i][j] += acc[i][j];
          acc[i][j] = 0.f;
        }
    }
#pragma unroll
    for (int h = 0; h < H; ++h)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        As[lk + i][lrow + 64 * h] = ar[h][i];
        Ws[lk + i][lrow + 64 * h] = wr[h][i];
      }
    __syncthreads();
    if (k0 + BK < K) fetch(k0 + BK);
#pragma unroll
    for (int k = 0; k < BK; ++k) {
      float a[R], w[R];
#pragma unroll
      for (int h = 0; h < H; ++h) {
        *reinterpret_cast<float4*>(&a[4 * h]) = *reinterpret_cast<const float4*>(&As[k][64 * h + ty * 4]);
        *reinterpret_cast<float4*>(&w[4 * h]) = *reinterpret_cast<const float4*>(&Ws[k][64 * h + tx * 4]);
      }
#pragma unroll
      for (int i = 0; i < R; ++i)
#pragma unroll
        for (int j = 0; j < R; ++j) acc[i][j] = fmaf(a[i], w[j], acc[i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int m = m0 + (i / 4) * 64 + ty * 4 + i % 4;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const int n = n0 + (j / 4) * 64 + tx * 4 + j % 4;
      if (n < N) Elem<TO>::store(C + (size_t)m * ldc + n, total[i][j] + acc[i][j]);
    }
  }
}

// The same product on the matrix cores: v_mfma_f32_32x32x2_f32 multiplies and adds in full
// float32 and, for every output element, gives exactly the bits of fmaf over its two k in
// ascending order (measured against the chain on random operands: every output of every
// step equal), so a walk over k in steps of two is the chain of the kernels above and below,
// bit for bit, and the pieces of kPiece are kept as they are.  A block of four waves owns
// 64H x 64H outputs, a wave 32H x 32H of them (H x H tiles of 32 x 32, each 16 accumulators a
// lane and as many for the total).  A lane's operand of a step is one float, A[row lane % 32][k + lane / 32]: a row of
// a stage lies in LDS as its even k, then its odd k, so that one 16-byte read is four steps' operand.
// A wave's step is 64 cycles a pair of tiles, so a stage of 16 k of 64 x 64 outputs was over long before the next one's loads
// had come (47 TFLOP/s): stages hold 64 k there and 32 k of 128 x 128, two of them in LDS (one barrier a stage),
// loaded without a branch (1,000 rows: weights of 2,048 x 6,144 413 -> 267 us, 2,048 x 2,048 141 -> 92, 12,288 x 2,048 497 -> 439;
// 130 rows: 321 -> 153, 98 -> 55, 178 -> 143).
typedef float float16v __attribute__((ext_vector_type(16)));

template <typename TO, int H>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void gemm_tiled_mfma_kernel(const float* __restrict__ A,
                                                              const float* __restrict__ W,
                                                              TO* __restrict__ C, int M, int N, int K,
                                                              long lda, long ldw, long ldc) {
  typedef float float4v __attribute__((ext_vector_type(4)));
  constexpr int BM = 64 * H, BN = 64 * H, SK = H == 1 ? 64 : 32, PITCH = SK + 4;
  constexpr int LANES = SK / 4, ROWS = 256 / LANES, PASSES = BM / ROWS;   // the loader: lanes a row, rows a pass
  static_assert(kPiece % SK == 0, "a piece is whole stages");
  __shared__ __attribute__((aligned(16))) float As[2][BM][PITCH];
  __shared__ __attribute__((aligned(16))) float Ws[2][BN][PITCH];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 31, g = lane >> 5;
  const int wm = (wave & 1) * 32 * H, wn = (wave >> 1) * 32 * H;   // this wave's corner of the block's tile
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  const int lrow = tid / LANES, lk = (tid % LANES) * 4;
  // four k of a row are one 16-byte load; rows past the end are read at the last row and never stored, what lies past K is
  // read at the row's end and becomes zero.  Where rows do not lie on 16-byte borders, or K ends within a piece, a whole
  // piece is still one load of 16 bytes, on the border that its numbers have (1,000
  // rows, weights of 6,144 x 2,048, one operand off its border 293 us, by single numbers 394; K of 2,049 300 and 407; 4 rows 54, 66).
  const bool wide = K % 4 == 0 && K >= 4 && lda % 4 == 0 && ldw % 4 == 0 &&
                    (reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(W)) % 16 == 0;

  float16v acc[H][H], total[H][H];
#pragma unroll
  for (int i = 0; i < H; ++i)
#pragma unroll
    for (int j = 0; j < H; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = total[i][j][e] = 0.f;

  float4v ar[PASSES], wr[PASSES];
  const auto fetch = [&](int k0) {
    const int k = k0 + lk;
    if (wide) {
#pragma unroll
      for (int h = 0; h < PASSES; ++h) {
        ar[h] = *reinterpret_cast<const float4v*>(A + (size_t)min(m0 + lrow + ROWS * h, M - 1) * lda + min(k, K - 4));
        wr[h] = *reinterpret_cast<const float4v*>(W + (size_t)min(n0 + lrow + ROWS * h, N - 1) * ldw + min(k, K - 4));
      }
    } else if (k + 3 < K) {
#pragma unroll
      for (int h = 0; h < PASSES; ++h) {
        __builtin_memcpy(&ar[h], A + (size_t)min(m0 + lrow + ROWS * h, M - 1) * lda + k, 16);
        __builtin_memcpy(&wr[h], W + (size_t)min(n0 + lrow + ROWS * h, N - 1) * ldw + k, 16);
      }
    } else {
#pragma unroll
      for (int h = 0; h < PASSES; ++h) {
        const int m = m0 + lrow + ROWS * h, n = n0 + lrow + ROWS * h;
#pragma unroll
        for (int i = 0; i < 4; ++i) ar[h][i] = (m < M && k + i < K) ? A[(size_t)m * lda + k + i] : 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) wr[h][i] = (n < N && k + i < K) ? W[(size_t)n * ldw + k + i] : 0.f;
      }
    }
  };
  fetch(0);
  int buf = 0;
  for (int k0 = 0; k0 < K; k0 += SK, buf ^= 1) {
    if (k0 > 0 && k0 % kPiece == 0) {
#pragma unroll
      for (int i = 0; i < H; ++i)
#pragma unroll
        for (int j = 0; j < H; ++j) {
          total[i][j] += acc[i][j];
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
        }
    }
    const bool inside = k0 + lk < K;       // (K a multiple of four, or `fetch` has made the zeros)
#pragma unroll
    for (int h = 0; h < PASSES; ++h) {
      const float4v a = inside ? ar[h] : float4v{0.f, 0.f, 0.f, 0.f}, w = inside ? wr[h] : float4v{0.f, 0.f, 0.f, 0.f};
      float* const ap = &As[buf][lrow + ROWS * h][lk / 2];
      float* const wp = &Ws[buf][lrow + ROWS * h][lk / 2];
      *reinterpret_cast<float2*>(ap) = make_float2(a[0], a[2]);
      *reinterpret_cast<float2*>(ap + SK / 2) = make_float2(a[1], a[3]);
      *reinterpret_cast<float2*>(wp) = make_float2(w[0], w[2]);
      *reinterpret_cast<float2*>(wp + SK / 2) = make_float2(w[1], w[3]);
    }
    __syncthreads();      // (one a stage: this copy is written again behind the next stage's barrier)
    if (k0 + SK < K) fetch(k0 + SK);
#pragma unroll
    for (int kk = 0; kk < SK; kk += 8) {
      float4v a[H], w[H];
#pragma unroll
      for (int h = 0; h < H; ++h) {
        a[h] = *reinterpret_cast<const float4v*>(&As[buf][wm + 32 * h + r][g * (SK / 2) + kk / 2]);
        w[h] = *reinterpret_cast<const float4v*>(&Ws[buf][wn + 32 * h + r][g * (SK / 2) + kk / 2]);
      }
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int i = 0; i < H; ++i)
#pragma unroll
          for (int j = 0; j < H; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i][s], w[j][s], acc[i][j], 0, 0, 0);
    }
  }
  // acc[i][j][4 q + e] = C[m0 + wm + 32 i + 8 q + 4 g + e][n0 + wn + 32 j + r]
#pragma unroll
  for (int i = 0; i < H; ++i)
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int m = m0 + wm + 32 * i + 8 * q + 4 * g + e;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < H; ++j) {
          const int n = n0 + wn + 32 * j + r;
          if (n < N) Elem<TO>::store(C + (size_t)m * ldc + n, total[i][j][4 * q + e] + acc[i][j][4 * q + e]);
        }
      }
}

// Few rows (M <= 16, float32): the tiles above leave most of a block idle.  Here a wave owns 64 weight rows, a lane one of
// them, and walks them 32 k at a time; the activations are the same for every lane (the compiler reads them through
// the scalar path).  The order of the sum is the one of the tiled kernel, bit for bit: k ascending within a piece of
// kPiece, the pieces' sums added to the total one after the other; so a row's result is still the same whatever the batch holds.
// With `partial` a wave sums one piece only and writes it to partial[piece][M][N]; the second
// kernel adds the pieces in order (for matrices of too few rows to fill the GPU otherwise).
//
// Bound by the weights' bytes.  A tile of 64 rows by 32 k is loaded as whole cache lines (eight lanes a row's 128 bytes),
// two tiles ahead, and changes hands through the wave's own LDS (rows 36 floats apart: sixteen lanes' pieces lie in
// different banks).  Lanes that loaded from a row each touched 64 lines a load (4 rows:
// weights of 4,096 x 2,048 19.8 us, now 13.1, both kernels; 12,288 x 2,048 27.2, 23.0; 151,936 x 2,048 257, 235, and 425, 248 for 8 rows).
constexpr int kFewK = 32, kFewPitch = kFewK + 4;
template <int MT>
__global__ __launch_bounds__(64) void gemm_fewrows_kernel(const float* __restrict__ A,
                                                          const float* __restrict__ W,
                                                          float* __restrict__ C, float* __restrict__ partial,
                                                          int M, int N, int K, long lda, long ldw, long ldc) {
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  static_assert(kPiece % (2 * kFewK) == 0, "a piece is whole pairs of tiles");
  __shared__ __attribute__((aligned(16))) float tile[64 * kFewPitch];
  const int lane = threadIdx.x;
  const int n0 = blockIdx.x * 64, n = n0 + lane;
  const int pieces = (K + kPiece - 1) / kPiece;
  const int k_begin = (partial ? blockIdx.y : 0) * kPiece;
  const int k_end = min(K, (partial ? (int)blockIdx.y + 1 : pieces) * kPiece);
  // (rows past N are computed from a valid row and never stored; what lies past K is read at the row's end, not used)
  const float* from[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) from[i] = W + (size_t)min(n0 + 8 * i + lane / 8, N - 1) * ldw;
  const int col = lane % 8 * 4;
  f32x4 reg[2][8];
  const auto fetch = [&](f32x4 (&r)[8], int k0) {
    const int k = min(k0 + col, K - 4);
#pragma unroll
    for (int i = 0; i < 8; ++i) r[i] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(from[i] + k));
  };
  float acc[MT], total[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) acc[m] = total[m] = 0.f;
  const auto step = [&](int k, int at) {
    const f32x4 w = *reinterpret_cast<const f32x4*>(tile + lane * kFewPitch + at);
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const float4 a = *reinterpret_cast<const float4*>(A + (size_t)min(m, M - 1) * lda + k);
      acc[m] = fmaf(a.x, w[0], acc[m]);
      acc[m] = fmaf(a.y, w[1], acc[m]);
      acc[m] = fmaf(a.z, w[2], acc[m]);
      acc[m] = fmaf(a.w, w[3], acc[m]);
    }
  };
  fetch(reg[0], k_begin);
  if (k_begin + kFewK < k_end) fetch(reg[1], k_begin + kFewK);
  for (int k0 = k_begin; k0 < k_end; k0 += 2 * kFewK) {
    if (k0 > k_begin && k0 % kPiece == 0) {
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        total[m] += acc[m];
        acc[m] = 0.f;
      }
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int k = k0 + u * kFewK;
      if (k >= k_end) break;
#pragma unroll
      for (int i = 0; i < 8; ++i) *reinterpret_cast<f32x4*>(tile + (8 * i + lane / 8) * kFewPitch + col) = reg[u][i];
      if (k + 2 * kFewK < k_end) fetch(reg[u], k + 2 * kFewK);
      wave_lds_sync();
      if (k + kFewK <= k_end) {
#pragma unroll
        for (int at = 0; at < kFewK; at += 4) step(k + at, at);
      } else {
        for (int at = 0; k + at < k_end; at += 4) step(k + at, at);
      }
      wave_lds_sync();
    }
  }
  if (n >= N) return;
  if (partial) {
#pragma unroll
    for (int m = 0; m < MT; ++m)
      if (m < M) partial[((size_t)blockIdx.y * M + m) * N + n] = acc[m];
    return;
  }
#pragma unroll
  for (int m = 0; m < MT; ++m)
    if (m < M) C[(size_t)m * ldc + n] = total[m] + acc[m];
}

__global__ __launch_bounds__(256) void gemm_fewrows_add_kernel(const float* __restrict__ partial,
                                                               float* __restrict__ C, int M, int N,
                                                               int pieces, long ldc) {
  const int n = blockIdx.x * 256 + threadIdx.x, m = blockIdx.y;
  if (n >= N) return;
  float total = 0.f;
  for (int p = 0; p < pieces; ++p) total += partial[((size_t)p * M + m) * N + n];
  C[(size_t)m * ldc + n] = total;
}

// float32 in and out, M <= 16, K and the row strides multiples of 4, 16-byte aligned rows.
// partial: null, or room for ceil(K / 256) * M * N floats: then every piece of K has a wave of its own.
TK_API int tk_gemm_fewrows(const float* A, const float* W, float* C, float* partial, int M, int N, int K,
                           long lda, long ldw, long ldc, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (M > 16 || K < 4 || K % 4 != 0 || lda % 4 != 0 || ldw % 4 != 0) return -1;
  if (reinterpret_cast<uintptr_t>(A) % 16 != 0 || reinterpret_cast<uintptr_t>(W) % 16 != 0) return -1;
  const int pieces = (K + kPiece - 1) / kPiece;
  if (pieces > 65535) return -1;
  dim3 grid((N + 63) / 64, partial ? pieces : 1);
#define TK_FEW(MT_) gemm_fewrows_kernel<MT_><<<grid, 64, 0, stream>>>(A, W, C, partial, M, N, K, lda, ldw, ldc)
  if (M == 1) TK_FEW(1);
  else if (M == 2) TK_FEW(2);
  else if (M <= 4) TK_FEW(4);
  else if (M <= 8) TK_FEW(8);
  else TK_FEW(16);
#undef TK_FEW
  if (partial)
    gemm_fewrows_add_kernel<<<dim3((N + 255) / 256, M), 256, 0, stream>>>(partial, C, M, N, pieces, ldc);
  return launch_status();
}

// in_dtype / out_dtype: 0 = float32, 1 = bfloat16
TK_API int tk_gemm_tiled(int in_dtype, int out_dtype, const void* A, const void* W, void* C, int M,
                         int N, int K, long lda, long ldw, long ldc, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K < 0) return -1;
  // tiles of 128 x 128 if they give every CU a block, else of 64 x 64
  const long big = (long)((N + 127) / 128) * ((M + 127) / 128);
  const int H = big >= 256 ? 2 : 1;
  dim3 grid((N + 64 * H - 1) / (64 * H), (M + 64 * H - 1) / (64 * H));
  if (grid.y > 65535) return -1;
#define TK_TILED(TI_, TO_)                                                                         \
  {                                                                                                \
    if (H == 2)                                                                                    \
      gemm_tiled_kernel<TI_, TO_, 2><<<grid, 256, 0, stream>>>((const TI_*)A, (const TI_*)W,       \
                                                               (TO_*)C, M, N, K, lda, ldw, ldc);   \
    else                                                                                           \
      gemm_tiled_kernel<TI_, TO_, 1><<<grid, 256, 0, stream>>>((const TI_*)A, (const TI_*)W,       \
                                                               (TO_*)C, M, N, K, lda, ldw, ldc);   \
  }
  if (in_dtype == 0 && out_dtype == 0) {
    // float32 operands: the matrix-core form (the same bits)
    if (H == 2) gemm_tiled_mfma_kernel<float, 2><<<grid, 256, 0, stream>>>((const float*)A, (const float*)W, (float*)C, M, N, K, lda, ldw, ldc);
    else gemm_tiled_mfma_kernel<float, 1><<<grid, 256, 0, stream>>>((const float*)A, (const float*)W, (float*)C, M, N, K, lda, ldw, ldc);
  }
  else if (in_dtype == 1 && out_dtype == 1) TK_TILED(bf16_t, bf16_t)
  else if (in_dtype == 1 && out_dtype == 0) TK_TILED(bf16_t, float)
  else return -1;
#undef TK_TILED
  return launch_status();
}

// the same entry points in slot form (slots.h), for launch lists
TK_SLOTS(tk_gemm_tiled)
TK_SLOTS(tk_gemm_fewrows)
