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

// The same product on the matrix cores, for operands that gemm_float32.hip does not take (rows off 16-byte borders, K not a
// multiple of four) and a short K of many results (ops.float32_through_registers): v_mfma_f32_32x32x2_f32 multiplies and adds in full
// float32 and, for every output element, gives exactly the bits of fmaf over its two k in
// ascending order (measured against the chain on random operands: every output of every
// step equal), so a walk over k in steps of two is the chain of the kernels above and below,
// bit for bit, and the pieces of kPiece are kept as they are.  A block of four waves owns
// 64H x 64H outputs, a wave 32H x 32H of them (H x H tiles of 32 x 32, each 16 accumulators a
// lane and as many for the total).  A lane's operand of a step is one float, A[row lane % 32][k + lane / 32]: a row of
// a stage lies in LDS as its even k, then its odd k, so that one 16-byte read is four steps' operand.
// A wave's step is 64 cycles a pair of tiles, so a stage of 16 k of 64 x 64 outputs was over long before the next one's loads
// had come (47 TFLOP/s): stages hold 64 k there and 32 k of 128 x 128, two of them in LDS, one barrier a stage.  (1.1 to 2.1 times as
// fast so, measured on operands on their borders; what those off them take stands at the loads below.)
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
  // Four k of a row are one load of 16 bytes, on the border that its numbers have (1,000 rows, weights of 6,144 x 2,048, one operand off
  // its border 293 us, by single numbers 394; K of 2,049 300 and 407; 4 rows 54, 66); rows past the end are read at the last row
  // and never stored, what lies past K becomes zero.
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
    if (k + 3 < K) {
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
#pragma unroll
    for (int h = 0; h < PASSES; ++h) {
      const float4v a = ar[h], w = wr[h];
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

// Few rows (M <= 16, float32): the tiles above leave most of a block idle.  v_mfma_f32_16x16x4_f32 too gives the bits of
// fmaf over its four k in ascending order, so a wave that takes a piece of kPiece k four at a time forms the piece's sum as
// the tiled kernel does, and the pieces' sums are added to the total in their order, bit for bit; a row's result is still
// the same whatever the batch holds.
//
// Bound by the weights' bytes, and for small matrices by the trips to memory.  An operand's sixteen rows are J = 16 / TP
// pieces of K (a bundle) of TP weight rows, its columns the same pieces of TP rows of activations; the blocks on the
// result's diagonal are kept.  Groups of 4 or 8 rows give small matrices four and two times the blocks.  A block's waves
// take a bundle each a round; a round's sums meet in LDS, where one wave adds them in order.  Blocks walk over
// groups of rows, loads running ahead over their borders.  Weights come as 256 contiguous bytes of four rows a load, two
// or four stages of 64 k ahead, and change hands through the wave's own LDS (rows 68 floats apart: 64 banks); the activations'
// four numbers a lane become the four k of a step by swaps between the lanes of a column.
// DEALT: the bundles of a block's groups are dealt to its waves one after the other, over the groups' borders; else a group
// begins with a round, and where its bundles are not a multiple of the waves the last ones have none (10 pieces in rounds of
// four leave a sixth of the waves' time).  19,456 x 2,560 at one row 39.7 us in rounds, dealt 35.9;
// 14,000 x 2,560 31.5 and 28.5; 38,696 x 2,592 78.6 and 70.2; for smaller matrices, whose blocks have a group or two, rounds are as
// fast or a few percent faster (2,048 x 6,144 12.3, dealt 13.2).
// (Before, a lane owned a weight row and multiplied in the vector unit, 64 rows and a piece a wave, the pieces' sums
// through memory to a kernel of their own: us there and here, 4 rows, 2,048 x 2,048 12.1 and 6.7, 4,096 x 2,048 13.2 and 8.7,
// 2,048 x 6,144 19.3 and 13.1, 12,288 x 2,048 23.1 and 19.8, 151,936 x 2,048 240 and 202; at one row it was up to 8 % ahead for some
// matrices of 18,000 rows and more, 18,624 x 2,176 31.1 and 33.7, 26,048 x 4,224 74.5 and 80.8.)
template <int TP, int WAVES, int DEPTH, bool DEALT>
__global__ __launch_bounds__(WAVES * 64) __attribute__((amdgpu_waves_per_eu(2))) void gemm_fewrows_kernel(
    const float* __restrict__ A, const float* __restrict__ W, float* __restrict__ C, int M, int N, int K, long lda, long ldw,
    long ldc) {
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  constexpr int J = 16 / TP, STAGES = kPiece / 64, PITCH = 68, QUADS = TP / 4;
  static_assert(kPiece == 256 && (DEPTH == 2 || DEPTH == 4), "a piece is four stages of 64 k");
  __shared__ __attribute__((aligned(16))) float tile[WAVES][16 * PITCH];
  __shared__ __attribute__((aligned(16))) f32x4 sums[2][WAVES * J][TP * QUADS];   // of a round: [piece][row of activations, four weight rows]
  const int lane = threadIdx.x & 63, wave = DEALT ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : threadIdx.x >> 6;
  const int a = lane & 15, g = lane >> 4;
  const int pieces = (K + kPiece - 1) / kPiece, bundles = (pieces + J - 1) / J;
  const int rounds = (pieces + WAVES * J - 1) / (WAVES * J);      // of a group, not DEALT
  const int own_groups = ((N + TP - 1) / TP - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x;
  const int turns = own_groups * bundles;      // (group, bundle) pairs of this block
  const int visits = DEALT ? (turns + WAVES - 1) / WAVES : own_groups * rounds;

  // this lane's place: of the loads of weights row 4 i + lane / 16 of the operand, of those of activations column a
  const int wk = a * 4, own_m = min(a % TP, M - 1);
  const float* const arow = A + (size_t)own_m * lda;
  f32x4 wreg[DEPTH][4], areg[DEPTH][4];
  // `at`: a group's round, of which this wave has its own bundle (DEALT: the bundle).  A bundle past the last is never read (first
  // k >= K); rows past N are read at the last row and never stored, what lies past K is read at the row's end and becomes zero.
  const auto first_k = [&](int at, int share) { return ((DEALT ? at : at * WAVES + wave) * J + share) * kPiece; };
  const auto fetch = [&](int group, int at, int stage, int buf) {
    if (!DEALT && first_k(at, 0) >= K) return;      // (uniform)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = 4 * i + g;
      const int n = min(group * TP + row % TP, N - 1), k = min(first_k(at, row / TP) + 64 * stage + wk, K - 4);
      wreg[buf][i] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(W + (size_t)n * ldw + k));
    }
    const int k0 = first_k(at, a / TP) + 64 * stage + 4 * g;
#pragma unroll
    for (int j = 0; j < 4; ++j) areg[buf][j] = *reinterpret_cast<const f32x4*>(arow + min(k0 + 16 * j, K - 4));
  };

  int group = blockIdx.x, at = 0;
  if constexpr (DEALT) {
    group += wave / bundles * (int)gridDim.x;
    at = wave % bundles;
  }
  if (!DEALT || wave < turns) {
#pragma unroll
    for (int s = 0; s < DEPTH; ++s) fetch(group, at, s, s);
  }
  f32x4 total = {0.f, 0.f, 0.f, 0.f};
  for (int v = 0; v < visits; ++v) {
    bool turn, last;            // the group is done; this wave reads no more
    int next_at, next_group;
    if constexpr (DEALT) {
      next_at = at + WAVES % bundles;
      turn = next_at >= bundles;
      last = (v + 1) * WAVES + wave >= turns;
      next_group = group + (WAVES / bundles + (turn ? 1 : 0)) * (int)gridDim.x;
      next_at -= turn ? bundles : 0;
    } else {
      turn = at + 1 == rounds, last = v + 1 == visits;
      next_at = turn ? 0 : at + 1, next_group = turn ? group + (int)gridDim.x : group;
    }
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    if (DEALT ? v * WAVES + wave < turns : first_k(at, 0) < K) {
      const bool whole = first_k(at, J - 1) + kPiece <= K;
#pragma unroll
      for (int s = 0; s < STAGES; ++s) {
        const int buf = s % DEPTH;
        float* const mine = tile[wave];
        wave_lds_sync();      // (the stage before has been read)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          f32x4 w = wreg[buf][i];
          if (!whole && first_k(at, (4 * i + g) / TP) + 64 * s + wk >= K) w = f32x4{0.f, 0.f, 0.f, 0.f};
          *reinterpret_cast<f32x4*>(mine + (4 * i + g) * PITCH + wk) = w;
        }
        // areg[j][e] holds k = 16 j + 4 g + e; step[j][e] is to hold k = 16 j + 4 e + g
        uint32_t step[4][4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          f32x4 x = areg[buf][j];
          if (!whole && first_k(at, a / TP) + 64 * s + 16 * j + 4 * g >= K) x = f32x4{0.f, 0.f, 0.f, 0.f};
          const auto e02 = __builtin_amdgcn_permlane32_swap(__float_as_uint(x[0]), __float_as_uint(x[2]), false, false);
          const auto e13 = __builtin_amdgcn_permlane32_swap(__float_as_uint(x[1]), __float_as_uint(x[3]), false, false);
          const auto e01 = __builtin_amdgcn_permlane16_swap(e02[0], e13[0], false, false);
          const auto e23 = __builtin_amdgcn_permlane16_swap(e02[1], e13[1], false, false);
          step[j][0] = e01[0];
          step[j][1] = e01[1];
          step[j][2] = e23[0];
          step[j][3] = e23[1];
        }
        if (s + DEPTH < STAGES) fetch(group, at, s + DEPTH, buf);
        else if (!last) fetch(next_group, next_at, s + DEPTH - STAGES, buf);
        wave_lds_sync();
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(mine[a * PITCH + 16 * j + 4 * e + g], __uint_as_float(step[j][e]), acc, 0, 0, 0);
      }
    } else if (!DEALT && !last) {
#pragma unroll
      for (int s = 0; s < DEPTH; ++s) fetch(next_group, next_at, s, s);
    }
    // acc[e]: weight row 4 g + e of the operand against column a of the activations
    if (4 * g / TP == a / TP) sums[v & 1][wave * J + a / TP][a % TP * QUADS + g % QUADS] = acc;
    __syncthreads();      // (one a round: this copy is written again behind the next round's barrier)
    if (threadIdx.x < TP * QUADS) {      // (of wave 0, whose group and bundle are the round's first)
      const auto finish = [&](int at_group) {
        const int m = threadIdx.x / QUADS, n = at_group * TP + threadIdx.x % QUADS * 4;
        if (m < M && n < N) store_four<float>(C + (size_t)m * ldc + n, total[0], total[1], total[2], total[3], N - n, rows_take_wide_stores(C, ldc));
        total = f32x4{0.f, 0.f, 0.f, 0.f};
      };
      if constexpr (DEALT) {
        const int filled = min(WAVES, turns - v * WAVES);
        for (int w = 0, at_group = group, at_bundle = at; w < filled;) {
          const int run = min(filled - w, bundles - at_bundle), left = min(run * J, pieces - at_bundle * J);      // of one group
          for (int p = 0; p < left; ++p) total += sums[v & 1][w * J + p][threadIdx.x];
          w += run;
          if (at_bundle + run < bundles) break;      // (goes on in the next round)
          finish(at_group);
          at_bundle = 0;
          at_group += (int)gridDim.x;
        }
      } else {
        const int left = min(WAVES * J, pieces - at * WAVES * J);
        for (int p = 0; p < left; ++p) total += sums[v & 1][p][threadIdx.x];
        if (turn) finish(group);
      }
    }
    group = next_group;
    at = next_at;
  }
}

// float32 in and out, M <= 16, K and the row strides multiples of 4, 16-byte aligned rows.  rows: of a group, 4, 8 or 16, at
// least M; waves a block, 4, 6 or 8; depth: stages of 64 k asked for ahead, 2, or 4 for 16 rows and four waves; blocks: at most so many;
// dealt: as described above, for 8 or 16 rows and four waves.
TK_API int tk_gemm_fewrows(const float* A, const float* W, float* C, int M, int N, int K, long lda, long ldw, long ldc, int rows,
                           int waves, int depth, int blocks, int dealt, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (M > 16 || M > rows || K < 4 || K % 4 != 0 || lda % 4 != 0 || ldw % 4 != 0 || blocks < 1) return -1;
  if (reinterpret_cast<uintptr_t>(A) % 16 != 0 || reinterpret_cast<uintptr_t>(W) % 16 != 0) return -1;
  const int grid = min(blocks, (N + rows - 1) / rows);
#define TK_FEW(TP_, WAVES_, DEPTH_, DEALT_) \
  if (rows == TP_ && waves == WAVES_ && depth == DEPTH_ && (dealt != 0) == DEALT_) { \
    gemm_fewrows_kernel<TP_, WAVES_, DEPTH_, DEALT_><<<grid, WAVES_ * 64, 0, stream>>>(A, W, C, M, N, K, lda, ldw, ldc); \
    return launch_status(); \
  }
  TK_FEW(4, 4, 2, false)
  TK_FEW(4, 6, 2, false)
  TK_FEW(4, 8, 2, false)
  TK_FEW(8, 4, 2, false)
  TK_FEW(8, 6, 2, false)
  TK_FEW(8, 8, 2, false)
  TK_FEW(16, 4, 2, false)
  TK_FEW(16, 6, 2, false)
  TK_FEW(16, 8, 2, false)
  TK_FEW(16, 4, 4, false)
  TK_FEW(8, 4, 2, true)
  TK_FEW(16, 4, 2, true)
#undef TK_FEW
  return -1;
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
