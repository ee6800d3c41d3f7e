// bf16 products of few rows (M <= 16: decode steps of up to sixteen requests) whose weights go from memory
// straight into matrix operands.
//
// C[M,N] = A[M,K] W[N,K]^T.  Such a product's time is a few trips to memory (an empty kernel of a recorded step costs
// 1.6 us, a streaming read of 4 or 8 MB 2.3 or 3.0), so everything a wave reads is asked for at once and nothing
// stands between the loads and the products: no LDS, no barrier before the end.
// v_mfma_f32_16x16x32_bf16 multiplies sixteen rows by sixteen columns; with groups of TP = 4 or 8 rows the
// operands are cut into J = 16 / TP shares of k: lane (a, kb) holds of the TP weight rows row a % TP at
// k + ((a / TP) * 4 + kb) * 8, of the activations row a % TP at the same k, and of the result the shares'
// own blocks on the diagonal are kept (the others mix one share's weights with another's activations).  A
// load instruction of a wave is then TP pieces of 1024 / TP contiguous bytes, and each weight is multiplied once per
// tile of TP rows of activations (MT of them).  Groups of 16 rows (64-byte pieces) took up to twice the time.
//
// A block owns RG groups of TP columns, its waves split K in contiguous shares; the waves' and the shares'
// sums are added in LDS in a fixed order (the result is deterministic), and because a block holds complete
// sums the epilogue can finish the work of the kernels that would follow.  Small blocks are the point: 1,024
// columns are 256 blocks here and 64 in the form whose blocks hold 16 columns (gemm_wholek.hip).  Beside that form and the
// LDS-staged one (gemm_mfma.hip), in a recorded chain: 1,024 x 3,072 into the stream at one row 3.9 us against 5.7, at 16
// rows 7.0 against 7.6; 6,144 gated columns of 2,048 10.9 against 12.7; 4,096 x 2,048 with a row scale 5.7 against
// 7.2; 4,096 x 12,288 into the stream 18.3 against 21.5 with the norm's kernel; 4,096 x 4,096 to bfloat16 at one row 7.7
// against 22.0, at 16 rows 11.0 against 22.7.  From three rows on the activations' reads (as many
// bytes as the weights', over RG) show: 5.1 TB/s at 8 rows where one row reaches 6.1.
//
//   * scaled input: the activations may be given as a = bf16(x * gamma) of an RMSNorm whose row statistics are
//     not applied yet; the product is linear in a row's scale, so the block multiplies row m of its result by
//     rstd[m] = rsqrt(sum_s sumsq[s][m] / K + eps);
//   * GATED: C = act(A W_gate^T) * (A W_up^T);
//   * ADD: the result is added into the float32 residual stream; the block writes the new stream, bf16(new
//     stream * gamma_next) for the product that follows the next norm, and the sum of squares of its columns of
//     every row (sumsq[block][m]), from which that product takes its rstd.
//
// So a decode layer of few rows runs q/k/v product, attention, o product, gate/up product and down product
// with no kernel in between.
#include "common.h"
#include "gate.h"
#include "slots.h"

using namespace tk;

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));  // arrays of HIP's uint4 struct end up in scratch

union Frag8 {
  u32x4 u;
  bf16x8 v;
};

struct RowScale {        // the statistics of the norm before the product; sumsq == nullptr: none
  const float* sumsq;    // [slabs][M]: sums of squares of the rows over slabs of columns
  int slabs;
  float eps;
  int act;               // GATED: 0 silu, 1 the tanh form of gelu, 2 the clamped gate; STORE: 0 none, 3 the square of relu
  float limit;           // of the clamped gate
};

struct StreamSum {       // ADD
  float* resid;          // [M, N] float32, rows ld_resid elements apart
  long ld_resid;
  const float* gamma;    // [N]: weight of the norm that reads the stream next
  bf16_t* scaled;        // [M, N] bf16(resid * gamma), rows ld_scaled apart; or nullptr
  long ld_scaled;
  float* sumsq;          // [gridDim.x][M]
};

enum { EPI_STORE = 0, EPI_GATED = 1, EPI_ADD = 2 };

template <int TP, int MT, int RG, int EPI, typename TO, int WAVES>
__global__ __launch_bounds__(WAVES * 64) void gemm_direct_kernel(
    const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, TO* __restrict__ C, int M, int N, int K,
    long lda, long ldw, long ldc, RowScale scale, StreamSum sum) {
  constexpr int TILES = EPI == EPI_GATED ? 2 : 1;
  constexpr int J = 16 / TP, STEP = 32 * J, QUADS = TP / 4;
  constexpr int ROWS = TP * MT;                               // of activations
  constexpr int U = RG * TILES + MT > 4 ? 2 : 4;              // steps whose loads are in flight together
  constexpr int KEPT = 4 * TP;                                // lanes of a wave whose results are kept
  static_assert(RG * KEPT <= 64 && MT <= WAVES, "a wave finishes a tile of the block's result");
  __shared__ __attribute__((aligned(16))) float4v red[WAVES][MT][TILES][RG][KEPT];
  __shared__ float stat[WAVES][ROWS];
  // (the wave as a scalar: its steps are then kept by branches.  The matrix units take no notice of the lanes' mask, by which
  // a condition that could differ from lane to lane may be carried out: they would multiply what no load has filled)
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int a = lane & 15, kb = lane >> 4, own = a & (TP - 1), share = a / TP;
  const int n0 = blockIdx.x * (RG * TP);
  const int koff = (share * 4 + kb) * 8;

  const int steps = (K + STEP - 1) / STEP;
  const int per = (steps + WAVES - 1) / WAVES;
  const int s_begin = wave * per, s_end = min(steps, s_begin + per);

  // rows past N or M: a valid row, never stored
  const bf16_t* wrow[TILES][RG];
#pragma unroll
  for (int t = 0; t < TILES; ++t)
#pragma unroll
    for (int g = 0; g < RG; ++g) wrow[t][g] = W + ((size_t)t * N + min(n0 + g * TP + own, N - 1)) * ldw;
  const bf16_t* xrow[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) xrow[i] = A + (size_t)min(i * TP + own, M - 1) * lda;

  float4v acc[MT][TILES][RG];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int t = 0; t < TILES; ++t)
#pragma unroll
      for (int g = 0; g < RG; ++g) acc[i][t][g] = float4v{0.f, 0.f, 0.f, 0.f};
  const u32x4 zero = {0u, 0u, 0u, 0u};

  u32x4 wreg[U][TILES][RG], xreg[U][MT];
  // a piece past K is the row's last piece instead and becomes zeros (of both: an infinite weight is not to meet one)
  const auto fetch = [&](int s) {
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (s + u < s_end) {
        const int k = min((s + u) * STEP + koff, K - 8);
#pragma unroll
        for (int t = 0; t < TILES; ++t)
#pragma unroll
          for (int g = 0; g < RG; ++g)      // weights are read once: streaming loads
            wreg[u][t][g] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(wrow[t][g] + k));
#pragma unroll
        for (int i = 0; i < MT; ++i) xreg[u][i] = *reinterpret_cast<const u32x4*>(xrow[i] + k);
      }
  };
  fetch(s_begin);

  // what only the epilogue needs is asked for now, behind the first loads.  Lane l of wave i adds the waves' results of
  // tile i's row l % TP, group l / KEPT, share (l / (QUADS TP)) % J, columns 4 ((l / TP) % QUADS) ..; share 0's finish.
  const int m = wave * TP + (lane & (TP - 1));
  const int n = n0 + lane / KEPT * TP + lane / TP % QUADS * 4;
  const bool finishes = wave < MT && lane < RG * KEPT && lane / (QUADS * TP) % J == 0 && m < M && n < N;
  float4 old = make_float4(0.f, 0.f, 0.f, 0.f), gam = make_float4(0.f, 0.f, 0.f, 0.f);
  if constexpr (EPI == EPI_ADD) {
    if (finishes) {     // N is a multiple of 4: the four columns are inside together
      old = *reinterpret_cast<const float4*>(sum.resid + (size_t)m * sum.ld_resid + n);
      if (sum.scaled != nullptr) gam = *reinterpret_cast<const float4*>(sum.gamma + n);
    }
  }
  float ss = 0.f;
  if (EPI != EPI_ADD && scale.sumsq != nullptr && tid % ROWS < M) {
    constexpr int GROUPS = WAVES * 64 / ROWS;     // threads that share a row's slabs
    for (int sl = tid / ROWS; sl < scale.slabs; sl += 4 * GROUPS) {
      float part[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) part[u] = sl + u * GROUPS < scale.slabs ? scale.sumsq[(size_t)(sl + u * GROUPS) * M + tid % ROWS] : 0.f;
      ss += (part[0] + part[1]) + (part[2] + part[3]);
    }
  }

  for (int s = s_begin; s < s_end; s += U) {
    if (K % STEP != 0 && s + U >= steps) {
#pragma unroll
      for (int u = 0; u < U; ++u)
        if ((s + u) * STEP + koff >= K) {
#pragma unroll
          for (int i = 0; i < MT; ++i) xreg[u][i] = zero;
#pragma unroll
          for (int t = 0; t < TILES; ++t)
#pragma unroll
            for (int g = 0; g < RG; ++g) wreg[u][t][g] = zero;
        }
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (s + u < s_end) {
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          Frag8 xf;
          xf.u = xreg[u][i];
#pragma unroll
          for (int t = 0; t < TILES; ++t)
#pragma unroll
            for (int g = 0; g < RG; ++g) {
              Frag8 wf;
              wf.u = wreg[u][t][g];
              acc[i][t][g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf.v, xf.v, acc[i][t][g], 0, 0, 0);
            }
        }
      }
    if (s + U < s_end) fetch(s + U);
  }

  // acc[i][t][g][e]: row kb*4 + e of (share, weight row) against column a of (share, batch row)
  if (kb / QUADS == share) {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int t = 0; t < TILES; ++t)
#pragma unroll
        for (int g = 0; g < RG; ++g) red[wave][i][t][g][(share * QUADS + kb % QUADS) * TP + own] = acc[i][t][g];
  }
  if (EPI != EPI_ADD && scale.sumsq != nullptr) {
    ss = sum_lanes<ROWS, kWave>(ss);
    if (lane < ROWS) stat[wave][lane] = ss;
  }
  __syncthreads();
  if (wave >= MT) return;

  float4v total[TILES];
#pragma unroll
  for (int t = 0; t < TILES; ++t) {
    total[t] = float4v{0.f, 0.f, 0.f, 0.f};
    if (lane < RG * KEPT) {
#pragma unroll
      for (int w = 0; w < WAVES; ++w) total[t] += red[w][wave][t][lane / KEPT][lane % KEPT];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) total[t][e] = sum_lanes<QUADS * TP, KEPT>(total[t][e]);
  }

  if constexpr (EPI == EPI_ADD) {
    float sq = 0.f;
    if (finishes) {
      const float4 v = make_float4(old.x + total[0][0], old.y + total[0][1], old.z + total[0][2], old.w + total[0][3]);
      *reinterpret_cast<float4*>(sum.resid + (size_t)m * sum.ld_resid + n) = v;
      if (sum.scaled != nullptr)
        *reinterpret_cast<uint2*>(sum.scaled + (size_t)m * sum.ld_scaled + n) =
            make_uint2(pack_bf16x2(v.x * gam.x, v.y * gam.y), pack_bf16x2(v.z * gam.z, v.w * gam.w));
      sq = v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
    }
    // (lanes that finish nothing hold zeros)
    sq = sum_lanes<KEPT, RG * KEPT>(sum_lanes<TP, QUADS * TP>(sq));
    if (lane < TP && m < M) sum.sumsq[(size_t)blockIdx.x * M + m] = sq;
    return;
  }
  if (!finishes) return;
  float rstd = 1.f;
  if (scale.sumsq != nullptr) {
    float all = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) all += stat[w][m];
    rstd = rsqrtf(all / (float)K + scale.eps);
  }
  float res[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    res[e] = total[0][e] * rstd;
    if constexpr (EPI == EPI_GATED) {
      res[e] = gated_value(res[e], total[TILES - 1][e] * rstd, scale.act, scale.limit);
    } else if (scale.act == 3) {
      const float v = fmaxf(res[e], 0.f);
      res[e] = v * v;
    }
  }
  store_four<TO>(C + (size_t)m * ldc + n, res[0], res[1], res[2], res[3], N - n, rows_take_wide_stores(C, ldc));
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

struct Call {
  const void *A, *W;
  void* C;
  int M, N, K;
  long lda, ldw, ldc;
  RowScale scale;
  StreamSum sum;
  hipStream_t stream;
};

template <int TP, int MT, int RG, int EPI, typename TO>
int launch(int waves, const Call& c) {
  const unsigned blocks = (c.N + RG * TP - 1) / (RG * TP);
#define TK_GO(WAVES_)                                                                                                    \
  gemm_direct_kernel<TP, MT, RG, EPI, TO, WAVES_><<<blocks, WAVES_ * 64, 0, c.stream>>>(                                   \
      (const bf16_t*)c.A, (const bf16_t*)c.W, (TO*)c.C, c.M, c.N, c.K, c.lda, c.ldw, c.ldc, c.scale, c.sum)
  if (waves == 8) TK_GO(8);
  else if (waves == 4) TK_GO(4);
  else return -1;
#undef TK_GO
  return launch_status();
}

// rows: of a group, 4 or 8; groups: of columns a block
template <int EPI, typename TO>
int pick_shape(int rows, int groups, int waves, const Call& c) {
  const int tiles = (c.M + rows - 1) / rows;
#define TK_SHAPE(TP_, MT_, RG_) \
  if (rows == TP_ && tiles == MT_ && groups == RG_) return launch<TP_, MT_, RG_, EPI, TO>(waves, c)
  TK_SHAPE(4, 1, 1);
  TK_SHAPE(4, 1, 2);
  TK_SHAPE(4, 1, 4);
  TK_SHAPE(4, 2, 1);
  TK_SHAPE(8, 1, 1);
  TK_SHAPE(8, 1, 2);
  TK_SHAPE(8, 2, 1);
  TK_SHAPE(8, 2, 2);
#undef TK_SHAPE
  return -1;
}

bool operands_fit(const void* A, const void* W, int M, int K, long lda, long ldw) {
  return M <= 16 && K >= 8 && K % 8 == 0 && lda % 8 == 0 && ldw % 8 == 0 && aligned16(A) && aligned16(W);
}

}  // namespace

// C[M, N] = act((A W^T) * rstd), rstd[m] = rsqrt(sum_s sumsq[s][m] / K + eps), or 1 with sumsq == nullptr.
// out_dtype: 0 float32, 1 bfloat16.  gated == 1: W = [W_gate; W_up] of 2N rows and
// C = act(A W_gate^T * rstd) * (A W_up^T * rstd), bfloat16; act 0 silu, 1 the tanh form of gelu, 2 the gate whose halves are
// clamped at `limit`; without a gate 0 none, 3 the square of relu.  M <= 16; K a multiple of 8; rows
// 16-byte aligned.  rows (4 or 8) of a group, groups of as many columns and waves (4 or 8) a block: the forms of pick_shape.
TK_API int tk_gemm_direct(int out_dtype, int gated, const void* A, const void* W, void* C, int M, int N, int K,
                          long lda, long ldw, long ldc, const float* sumsq, int slabs, float eps, int act, float limit,
                          int rows, int groups, int waves, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (!operands_fit(A, W, M, K, lda, ldw) || (sumsq != nullptr && slabs < 1)) return -1;
  if (gated ? out_dtype != 1 || act < 0 || act > 2 : act != 0 && act != 3) return -1;
  const Call c{A, W, C, M, N, K, lda, ldw, ldc, RowScale{sumsq, slabs, eps, act, limit}, StreamSum{}, stream};
  if (gated) return pick_shape<EPI_GATED, bf16_t>(rows, groups, waves, c);
  if (out_dtype == 0) return pick_shape<EPI_STORE, float>(rows, groups, waves, c);
  if (out_dtype == 1) return pick_shape<EPI_STORE, bf16_t>(rows, groups, waves, c);
  return -1;
}

// resid[M, N] += A W^T (float32 stream); scaled[M, N] = bf16(resid * gamma) (skipped with scaled == nullptr);
// sumsq[b][m] = sum over block b's columns (groups * rows of them) of resid[m][.]^2.
// M <= 16; N a multiple of 4; rows 16-byte aligned.
TK_API int tk_gemm_direct_add(const void* A, const void* W, int M, int N, int K, long lda, long ldw, float* resid,
                              long ld_resid, const float* gamma, void* scaled, long ld_scaled, float* sumsq,
                              int rows, int groups, int waves, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (!operands_fit(A, W, M, K, lda, ldw)) return -1;
  if (N % 4 != 0 || ld_resid % 4 != 0 || !aligned16(resid) || resid == nullptr || sumsq == nullptr) return -1;
  if (scaled != nullptr && (gamma == nullptr || !aligned16(gamma) || ld_scaled % 4 != 0 ||
                            (reinterpret_cast<uintptr_t>(scaled) & 7) != 0))
    return -1;
  const Call c{A, W, nullptr, M, N, K, lda, ldw, 0, RowScale{}, StreamSum{resid, ld_resid, gamma, (bf16_t*)scaled, ld_scaled, sumsq}, stream};
  return pick_shape<EPI_ADD, float>(rows, groups, waves, c);
}

// the same entry points in slot form (slots.h), for launch lists
TK_SLOTS(tk_gemm_direct)
TK_SLOTS(tk_gemm_direct_add)
