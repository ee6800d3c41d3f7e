// The experts' products of a routed feed-forward for steps of few tokens (gfx950, bfloat16): a block an expert that the
// step meets and 16 output channels, the weights read once for all the expert's pairs.
//
// What bounds it: the weights' bytes (a pair's activations are a few KB).  The form with a block a (token, chosen
// expert) pair (moe.hip) reads an expert's weights again for each of its pairs, and for one or two tokens has too
// few blocks, all walking the same offsets of rows that lie a power of two apart: 8B-shaped experts (4,096 x 6,144),
// one token of two experts: 75 us for the first product's 201 MB and 99 for the second's 100, here 38 and 22; 8 tokens of
// 16 such experts (12 met) 270 + 154 -> 179 + 110 (the bytes at a streaming read's 6.3 TB/s: 192 + 96); 24 tokens of 16
// experts of 1,024 x 1,024 42 + 22 -> 18 + 12.
//
// As in gemm_wholek.hip: a block's waves deal the chunks of 256 k between them, starting at unlike chunks; a wave
// reads 512 bytes of a weight row with 32 lanes, parks its 16 rows (gate and up: 32) in a tile of its own in LDS,
// 16-byte pieces swizzled by row, and takes the matrix operands from there; activations come straight from L2.  No
// barrier in the walk; the waves' sums are added in wave order.
#include "common.h"
#include "slots.h"

using namespace tk;

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

union Frag8 {
  u32x4 u;
  bf16x8 v;
};

constexpr int kChunk = 256;                     // k of a chunk
constexpr int kTileBytes = 16 * kChunk * 2;
constexpr int kMaxPairs = 1024;                 // of a step (a block lists its expert's in LDS)

// With far more experts than pairs a block's number counts the experts that the step meets, in order of appearance (a
// wave's lanes hold the pairs; a step of that loop costs some 30 cycles); else it is the expert (a block of an expert
// that nobody chose leaves at once: with 32 tokens of 16 experts the loop took 20 us of 170).
__host__ __device__ inline bool counts_met(int P, int E) { return P <= kWave && E > 2 * P; }

// The pairs of the block's expert in `list` (ascending), their count; -1 where there are none.  All threads call.
__device__ __forceinline__ int list_pairs(const int* __restrict__ chosen, int P, int E, int slot, int* list, int* counts, int& expert) {
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave, waves = blockDim.x / kWave;
  if (counts_met(P, E)) {
    const int mine = lane < P ? chosen[lane] : -1;
    int at = 0;
    unsigned long long members = 0;
    for (int q = 0; q < P; ++q) {
      const unsigned long long same = __ballot(mine == __builtin_amdgcn_readlane(mine, q));
      if (__ffsll(same) - 1 != q) continue;      // (seen before)
      if (at++ == slot) {
        members = same;
        expert = __builtin_amdgcn_readlane(mine, q);
        break;
      }
    }
    if (members == 0) return -1;                 // (the whole block alike)
    if (wave == 0 && (members >> lane & 1)) list[__popcll(members & ((1ull << lane) - 1))] = lane;
    __syncthreads();
    return __popcll(members);
  }
  expert = slot;
  int count = 0;
  for (int base = 0; base < P; base += blockDim.x) {
    const int p = base + tid;
    const unsigned long long hit = __ballot(p < P && chosen[p] == slot);
    if (lane == 0) counts[wave] = __popcll(hit);
    __syncthreads();
    int before = count;
    for (int w = 0; w < waves; ++w) {
      if (w < wave) before += counts[w];
      count += counts[w];
    }
    if (hit >> lane & 1) list[before + __popcll(hit & ((1ull << lane) - 1))] = p;
    __syncthreads();
  }
  return count > 0 ? count : -1;
}

// GATED: weights [E][2 R][K], an expert's gate rows then its up rows; a pair's activations are its token's row of x [N][K];
//   out (bfloat16 [P][R]) = silu(w g) * (w u) with the pair's weight w (on_output: w * silu(g) * u).
// else: weights [E][R][K]; activations x [P][K] a row a pair; out (float32 [top][N][R]) takes pair (n, k)'s at [k][n].
// MT: tiles of 16 pairs whose products share what a wave has parked.
template <bool GATED, int WAVES, int MT>
__global__ __launch_bounds__(WAVES * 64) void moe_stream_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ weights,
                                                                const int* __restrict__ chosen, const float* __restrict__ pair_weight,
                                                                void* __restrict__ out, int N, int top, int E, int R, int K, int on_output) {
  constexpr int TILES = GATED ? 2 : 1;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  __shared__ int list[kMaxPairs], counts[WAVES];
  int expert = 0;
  const int count = list_pairs(chosen, N * top, E, blockIdx.y, list, counts, expert);
  if (count < 0) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = lane & 15, kb = lane >> 4;
  const int n0 = blockIdx.x * 16;
  unsigned char* const mine = lds + (size_t)wave * (TILES * kTileBytes);

  const int total_chunks = (K + kChunk - 1) / kChunk, per = (total_chunks + WAVES - 1) / WAVES;
  const int rot = (int)((blockIdx.x + blockIdx.y) % (unsigned)per);     // (blocks in step read unlike parts of their rows)
  const auto chunk_at = [&](int i) {
    const int j = i + rot;
    return wave + (j >= per ? j - per : j) * WAVES;     // (may lie past the last chunk: skipped)
  };
  // piece i of this lane: weight row 2 i + lane / 32, 16-byte column lane % 32
  const int w_piece = lane & 31, w_row0 = lane >> 5;
  const bf16_t* const base = weights + (size_t)expert * TILES * R * K;
  const bf16_t* wrow[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) wrow[i] = base + (size_t)min(n0 + 2 * i + w_row0, R - 1) * K;
  const size_t second = (size_t)R * K;

  for (int first = 0; first < count; first += 16 * MT) {
    const bf16_t* xrow[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const int p = list[min(first + 16 * t + r, count - 1)];
      xrow[t] = x + (size_t)(GATED ? p / top : p) * K;
    }
    float4v acc[TILES][MT];
#pragma unroll
    for (int i = 0; i < TILES; ++i)
#pragma unroll
      for (int t = 0; t < MT; ++t) acc[i][t] = float4v{0.f, 0.f, 0.f, 0.f};
    u32x4 wreg[TILES][8];
    // a weight piece past K is the row's last piece and meets zeros
    const auto fetch = [&](int c) {
      const int at = min(c * kChunk + w_piece * 8, K - 8);
#pragma unroll
      for (int i = 0; i < TILES; ++i)
#pragma unroll
        for (int p = 0; p < 8; ++p) wreg[i][p] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(wrow[p] + i * second + at));
    };
    int i = 0;
    while (i < per && chunk_at(i) >= total_chunks) ++i;
    if (i < per) fetch(chunk_at(i));
    while (i < per) {
      const int c = chunk_at(i);
#pragma unroll
      for (int j = 0; j < TILES; ++j)
#pragma unroll
        for (int p = 0; p < 8; ++p) {
          const int row = 2 * p + w_row0;
          *reinterpret_cast<u32x4*>(mine + j * kTileBytes + row * (kChunk * 2) + ((w_piece ^ row) & 31) * 16) = wreg[j][p];
        }
      int next = i + 1;
      while (next < per && chunk_at(next) >= total_chunks) ++next;
      if (next < per) fetch(chunk_at(next));
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        if (t == 0 || first + 16 * t < count) {
          Frag8 xf[8];
#pragma unroll
          for (int s = 0; s < 8; ++s) {
            const int k = c * kChunk + s * 32 + kb * 8;
            const u32x4 v = *reinterpret_cast<const u32x4*>(xrow[t] + min(k, K - 8));
            xf[s].u = k < K ? v : u32x4{0u, 0u, 0u, 0u};
          }
#pragma unroll
          for (int s = 0; s < 8; ++s)
#pragma unroll
            for (int j = 0; j < TILES; ++j) {
              Frag8 wf;
              wf.u = *reinterpret_cast<const u32x4*>(mine + j * kTileBytes + r * (kChunk * 2) + (((s * 4 + kb) ^ r) & 31) * 16);
              acc[j][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf.v, xf[s].v, acc[j][t], 0, 0, 0);
            }
        }
      }
      i = next;
    }
    // acc[j][t][q]: this wave's share of channel n0 + 4 kb + q for pair first + 16 t + r; left in the wave's own tile
    float* const sums = reinterpret_cast<float*>(mine);     // [MT][TILES][64 lanes][4]
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int j = 0; j < TILES; ++j) *reinterpret_cast<float4v*>(sums + ((t * TILES + j) * 64 + lane) * 4) = acc[j][t];
    __syncthreads();
    const int channel = n0 + kb * 4;
    for (int t = wave; t < MT; t += WAVES) {
      const int at = first + 16 * t + r;
      if (at >= count || channel >= R) continue;
      float4v total[TILES];
#pragma unroll
      for (int j = 0; j < TILES; ++j) total[j] = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < WAVES; ++w) {
        const float* theirs = reinterpret_cast<const float*>(lds + (size_t)w * (TILES * kTileBytes));
#pragma unroll
        for (int j = 0; j < TILES; ++j) total[j] += *reinterpret_cast<const float4v*>(theirs + ((t * TILES + j) * 64 + lane) * 4);
      }
      const int p = list[at];
      if (GATED) {
        const float w = pair_weight[p];
        float v[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float g = on_output ? total[0][q] : total[0][q] * w, u = total[TILES - 1][q] * w;
          v[q] = g / (1.f + expf(-g)) * u;
        }
        store_four<bf16_t>(reinterpret_cast<bf16_t*>(out) + (size_t)p * R + channel, v[0], v[1], v[2], v[3], R - channel, R % 4 == 0);
      } else {
        store_four<float>(reinterpret_cast<float*>(out) + ((size_t)(p % top) * N + p / top) * R + channel, total[0][0], total[0][1],
                          total[0][2], total[0][3], R - channel, R % 4 == 0);
      }
    }
    if (first + 16 * MT < count) __syncthreads();      // (the tiles take the next pairs' weights)
  }
}

template <bool GATED, int WAVES, int MT>
int launch(const void* x, const void* weights, const int* chosen, const float* pair_weight, void* out, int N, int top, int E, int R,
           int K, int on_output, hipStream_t stream) {
  constexpr size_t lds = (size_t)WAVES * (GATED ? 2 : 1) * kTileBytes;
  static bool raised = false;
  if (!raised) {
    const hipError_t err = hipFuncSetAttribute((const void*)moe_stream_kernel<GATED, WAVES, MT>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (err != hipSuccess) return (int)err;
    raised = true;
  }
  const int P = N * top;
  moe_stream_kernel<GATED, WAVES, MT><<<dim3((R + 15) / 16, counts_met(P, E) ? P : E), WAVES * 64, lds, stream>>>(
      (const bf16_t*)x, (const bf16_t*)weights, chosen, pair_weight, out, N, top, E, R, K, on_output);
  return launch_status();
}

}  // namespace

// gated, x, weights, pair_weight and out as in tk_moe_grouped (moe.hip; gated == 2: the weight acts on the expert's output);
// chosen [N, top].  K a multiple of 8, x and weights on 16-byte borders, up to 1,024 pairs.
TK_API int tk_moe_stream(int gated, const void* x, const void* weights, const int* chosen, const float* pair_weight, void* out,
                         int N, int top, int E, int R, int K, hipStream_t stream) {
  if (N <= 0) return 0;
  if (K % 8 != 0 || K < 8 || R < 1 || top < 1 || E < 1 || (long)N * top > kMaxPairs || (uintptr_t)x % 16 != 0 || (uintptr_t)weights % 16 != 0)
    return -1;
#define TK_STREAM(GATED_, WAVES_)                                                                                               \
  (N <= 16 ? launch<GATED_, WAVES_, 1>(x, weights, chosen, pair_weight, out, N, top, E, R, K, gated == 2, stream)               \
   : (long)N * top <= 16L * E ? launch<GATED_, WAVES_, 2>(x, weights, chosen, pair_weight, out, N, top, E, R, K, gated == 2, stream)             \
             : launch<GATED_, WAVES_, 4>(x, weights, chosen, pair_weight, out, N, top, E, R, K, gated == 2, stream))
  // (pairs an expert has on average: a pass over 32 pairs keeps two waves a SIMD, one over 64 keeps one and reads an
  // expert's weights half as often; a fuller expert takes another pass)
  if (gated) return TK_STREAM(true, 4);
  if (K > 4 * kChunk) return TK_STREAM(false, 8);
  return TK_STREAM(false, 4);
#undef TK_STREAM
}

TK_SLOTS(tk_moe_stream)
