// The experts' products of a routed feed-forward for steps of few tokens (gfx950, bfloat16): a block an expert that the
// step meets and 16 output channels, the weights read once for all the expert's pairs.
//
// What bounds it: the weights' bytes (a pair's activations are a few KB).  The form with a block a (token, chosen
// expert) pair (moe.hip) reads an expert's weights again for each of its pairs, and for one or two tokens has too
// few blocks, all walking the same offsets of rows that lie a power of two apart: 8B-shaped experts (4,096 x 6,144),
// one token of two experts: 75 us for the first product's 201 MB and 99 for the second's 100, here 38 and 22; 8 tokens of
// 16 such experts (12 met) 270 + 149 -> 198 + 103 (the bytes at a streaming read's 6.3 TB/s: 192 + 96); 24 tokens of 16
// experts of 1,024 x 1,024 42 + 22 -> 18 + 11.
//
// A block's waves deal the chunks of 256 k between them, starting at unlike chunks; no barrier in the walk, the waves'
// sums are added in wave order.
//
// For many tokens (moe_tiles): tiles of 128 pairs of one expert (the lists of moe_sort) by the channels of a block's
// waves.  The form that takes weights in rows (moe.hip) reads 64-byte pieces of 16 rows an instruction, which the vector
// memory path serves at a quarter of its rate; parked in LDS the weights' writes alone (a 16-byte write of a
// wave takes some 30 cycles) outlast the products.
//
// So both forms take the weights as the matrix operands want them, laid out once when a model is bound: of a matrix
// [R][K] blocks of 32 rows by 32 k, a block as [octet of k 4][row 32][8 k].  A wave's operand of 32 rows by 16 k
// (v_mfma_f32_32x32x16_bf16) is then one run of 1 KB, one of 16 rows by 32 k (16x16x32) four of 256 bytes, and
// neither passes through LDS.  R a multiple of 32, K of 64.
#include "common.h"
#include "slots.h"

#include <type_traits>

using namespace tk;

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

union Frag8 {
  u32x4 u;
  bf16x8 v;
};

typedef float float16v __attribute__((ext_vector_type(16)));

constexpr int kBlock = 32 * 32;                 // numbers of a block of the weights' layout
constexpr int kChunk = 256;                     // k of a chunk
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
  __shared__ __attribute__((aligned(16))) float sums[WAVES][MT * TILES * 256];
  __shared__ int list[kMaxPairs], counts[WAVES];
  int expert = 0;
  const int count = list_pairs(chosen, N * top, E, blockIdx.y, list, counts, expert);
  if (count < 0) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = lane & 15, kb = lane >> 4;
  const int n0 = blockIdx.x * 16;

  const int total_chunks = (K + kChunk - 1) / kChunk, per = (total_chunks + WAVES - 1) / WAVES;
  // (blocks in step read unlike parts of their rows; by the expert and not by the block's number, which may follow the order
  // in which the step meets its experts: a pair's sums run in one order whoever stands before it)
  const int rot = (int)((blockIdx.x + (unsigned)expert) % (unsigned)per);
  const auto chunk_at = [&](int i) {
    const int j = i + rot;
    return wave + (j >= per ? j - per : j) * WAVES;     // (may lie past the last chunk: skipped)
  };
  // the 16 rows from n0 on: half of a block of 32
  const size_t second = (size_t)R * K;
  const bf16_t* const rows = weights + (size_t)expert * TILES * second + (size_t)(n0 / 32) * 32 * K + kb * 256 + (n0 & 16) * 8 + r * 8;
  const int blocks = K / 32;      // of 32 k

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
    // (blocks past K are the last one again and meet zeros)
    const auto fetch = [&](int c) {
#pragma unroll
      for (int i = 0; i < TILES; ++i)
#pragma unroll
        for (int s = 0; s < 8; ++s)
          wreg[i][s] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(rows + i * second + (size_t)min(c * 8 + s, blocks - 1) * kBlock));
    };
    int i = 0;
    while (i < per && chunk_at(i) >= total_chunks) ++i;
    if (i < per) fetch(chunk_at(i));
    while (i < per) {
      const int c = chunk_at(i);
      u32x4 now[TILES][8];
#pragma unroll
      for (int j = 0; j < TILES; ++j)
#pragma unroll
        for (int s = 0; s < 8; ++s) now[j][s] = wreg[j][s];
      int next = i + 1;
      while (next < per && chunk_at(next) >= total_chunks) ++next;
      if (next < per) fetch(chunk_at(next));
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        if (t == 0 || first + 16 * t < count) {
          Frag8 xf[8];
#pragma unroll
          for (int s = 0; s < 8; ++s) {
            const int b = c * 8 + s;
            const u32x4 v = *reinterpret_cast<const u32x4*>(xrow[t] + (size_t)min(b, blocks - 1) * 32 + kb * 8);
            xf[s].u = b < blocks ? v : u32x4{0u, 0u, 0u, 0u};
          }
#pragma unroll
          for (int s = 0; s < 8; ++s)
#pragma unroll
            for (int j = 0; j < TILES; ++j) {
              Frag8 wf;
              wf.u = now[j][s];
              acc[j][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf.v, xf[s].v, acc[j][t], 0, 0, 0);
            }
        }
      }
      i = next;
    }
    // acc[j][t][q]: this wave's share of channel n0 + 4 kb + q for pair first + 16 t + r
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int j = 0; j < TILES; ++j) *reinterpret_cast<float4v*>(&sums[wave][((t * TILES + j) * 64 + lane) * 4]) = acc[j][t];
    __syncthreads();
    const int channel = n0 + kb * 4;
    for (int t = wave; t < MT; t += WAVES) {
      const int at = first + 16 * t + r;
      if (at >= count) continue;
      float4v total[TILES];
#pragma unroll
      for (int j = 0; j < TILES; ++j) total[j] = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < WAVES; ++w) {
#pragma unroll
        for (int j = 0; j < TILES; ++j) total[j] += *reinterpret_cast<const float4v*>(&sums[w][((t * TILES + j) * 64 + lane) * 4]);
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
        store_four<bf16_t>(reinterpret_cast<bf16_t*>(out) + (size_t)p * R + channel, v[0], v[1], v[2], v[3], 4, true);
      } else {
        store_four<float>(reinterpret_cast<float*>(out) + ((size_t)(p % top) * N + p / top) * R + channel, total[0][0], total[0][1],
                          total[0][2], total[0][3], 4, true);
      }
    }
    if (first + 16 * MT < count) __syncthreads();      // (the next pairs' sums take their place)
  }
}

constexpr int kXcds = 8;        // dies of the GPU, each with an L2 of its own; blocks go to them in turn
constexpr int kTile = 128;      // pairs of a tile
constexpr int kStep = 64;       // k of a step
constexpr int kTileWaves = 4;
__device__ __align__(16) const bf16_t kZeros[32 * kStep] = {};      // a step of 32 rows' weights

// A block: a tile and the channels of its waves: with a gate a wave has 32 channels' gate and up rows, else 64 rows.  The
// tile's activations go through LDS (two copies, 64 k each, rows' 16-byte pieces swizzled so that sixteen rows' reads of
// one piece meet all banks), the weights come straight from memory: an operand's registers take their next step but one as
// soon as it has been multiplied, so that twice a step's loads are under way, and a step's reads of LDS run ahead of its
// products.  Four waves and two blocks a CU, which wait for barriers of their own; eight waves that share a tile's
// activations were slower.  The tiles of an expert at the same channels run side by side on one die, and beside them the
// die's other channels of the same tiles, so that a tile's activations too come from memory once a die (a channel block
// after the other read them again for each: 2,000 tokens 561 + 316 us where this order takes 501 + 288).
// 16 experts of 4,096 x 6,144, tokens of two, us before (loads one step ahead, a branch for every 32 pairs) and now: 300 tokens
// 304 + 202, 292 + 153; 2,000 544 + 333, 501 + 288; 4,000 894 + 507, 817 + 446 (0.99 PFLOP/s); 16 of 1,024 x 1,024, 300 tokens 23.8 +
// 20.6, 19.4 + 14.2.  Up to some 32 pairs an expert the weights' bytes bound it (1,610 MB in 292 us, 5.5 TB/s), beyond that bytes and
// products in turn: half of the tiles are filled in part.
// ODD: K is an odd number of steps, walked in pairs.
template <bool GATED, bool ODD>
__global__ __launch_bounds__(kTileWaves * 64) __attribute__((amdgpu_waves_per_eu(2, 2))) void moe_tiles_kernel(
    const bf16_t* __restrict__ x, const bf16_t* __restrict__ weights, const int* __restrict__ order,
    const int* __restrict__ tile_expert, const int* __restrict__ tile_start, const int* __restrict__ tile_count,
    const int* __restrict__ num_tiles, const float* __restrict__ pair_weight, void* __restrict__ out, int N, int top, int R, int K,
    int max_tiles, int channel_blocks, int on_output) {
  constexpr int kThreads = kTileWaves * 64, kPieces = kTile * kStep / 8 / kThreads;   // 16-byte pieces of a step a thread copies
  __shared__ __attribute__((aligned(16))) unsigned char xs[2][kTile * kStep * 2];
  const int per_die = gridDim.x / kXcds, work = (blockIdx.x % kXcds) * per_die + blockIdx.x / kXcds;
  if (work >= max_tiles * channel_blocks) return;
  // channel blocks in groups, of which a die has one where there are enough; in a group a tile's channel blocks, then the next tile's
  const int group_blocks = max(1, channel_blocks / kXcds), group = work / (max_tiles * group_blocks), in_group = work - group * max_tiles * group_blocks;
  const int here = min(group_blocks, channel_blocks - group * group_blocks);
  const int tile = in_group / here, channels = group * group_blocks + in_group % here;
  if (tile >= *num_tiles) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), col = lane & 31, g = lane >> 5;
  const int start = tile_start[tile], count = tile_count[tile];
  const int groups = (count + 31) / 32;                  // of 32 pairs that exist
  const int unit = channels * kTileWaves + wave;              // the wave's 32 channels (gated) or 64 rows
  const int row_blocks = R / 32;
  const bool active = GATED ? unit < row_blocks : 2 * unit < row_blocks;      // (a wave past the last still copies activations)
  const int first_block = GATED ? min(unit, row_blocks - 1) : min(2 * unit, row_blocks - 1);
  const int second_block = GATED ? first_block + row_blocks : min(first_block + 1, row_blocks - 1);
  const bf16_t* const base = weights + (size_t)tile_expert[tile] * (GATED ? 2 : 1) * R * K;      // (the same in all lanes)
  const bf16_t* const wp[2] = {base + (size_t)first_block * 32 * K, base + (size_t)second_block * 32 * K};
  const bf16_t* xp[kPieces];
  const int part = tid & 7, swizzle = (tid >> 4) & 7;      // (row >> 1, whose low three bits are the same in all rows of a thread)
  const int xat = (tid >> 3) * (kStep * 2) + (part ^ swizzle) * 16;
  static_assert(kThreads / 8 % 16 == 0, "a thread's rows share their swizzle");
#pragma unroll
  for (int i = 0; i < kPieces; ++i) {
    const int p = order[start + min(i * (kThreads / 8) + (tid >> 3), count - 1)];
    xp[i] = x + (size_t)(GATED ? p / top : p) * K + part * 8;
  }
  float16v acc[2][4];
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int q = 0; q < 16; ++q) acc[b][j][q] = 0.f;
  Frag8 w[2][2][4];
  u32x4 xr[kPieces];
  // Past the end nothing is used but where an odd number of steps is walked in pairs: zeros are (never a repeated step, whose
  // infinities would meet them).
  const auto weights_at = [&](int b, int k0) {
    if (ODD) return k0 < K ? wp[b] + (size_t)k0 * 32 : kZeros;
    return wp[b] + (size_t)min(k0, K - kStep) * 32;
  };
  const auto fetch_weights = [&](int k0, Frag8 (&to)[2][4]) {
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const bf16_t* const from = weights_at(b, k0);
#pragma unroll
      for (int s = 0; s < 4; ++s) to[b][s].u = *reinterpret_cast<const u32x4*>(from + s * 512 + lane * 8);
    }
  };
  const auto fetch_rows = [&](int k0) {
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
      if (ODD) {
        xr[i] = *reinterpret_cast<const u32x4*>(k0 < K ? xp[i] + k0 : kZeros);
      } else {
        if (k0 > 0 && k0 < K) xp[i] += kStep;
        xr[i] = *reinterpret_cast<const u32x4*>(xp[i]);
      }
    }
  };
  const auto park_rows = [&](int copy) {
#pragma unroll
    for (int i = 0; i < kPieces; ++i) *reinterpret_cast<u32x4*>(&xs[copy][xat + i * (kThreads / 8 * kStep * 2)]) = xr[i];
  };
  fetch_weights(0, w[0]);
  fetch_weights(kStep, w[1]);
  fetch_rows(0);
  park_rows(0);
  // GROUPS: of 32 pairs that the products take, known to the compiler: a step without branches, whose reads of LDS run ahead
  const auto walk = [&](auto groups_taken) {
    constexpr int GROUPS = groups_taken;
    const auto step = [&](int k0, int copy) {
      __syncthreads();      // this copy is written, the other one read
      fetch_rows(k0 + kStep);
      __builtin_amdgcn_sched_barrier(0);
      const int ahead = k0 + 2 * kStep;
      const bf16_t* const from[2] = {weights_at(0, ahead), weights_at(1, ahead)};
      Frag8 xf[GROUPS];
      const auto read = [&](int s, int j) {
        xf[j].u = *reinterpret_cast<const u32x4*>(&xs[copy][j * (32 * kStep * 2) + col * (kStep * 2) + (((2 * s + g) ^ (col >> 1)) & 7) * 16]);
      };
#pragma unroll
      for (int j = 0; j < GROUPS; ++j) read(0, j);
#pragma unroll
      for (int s = 0; s < 4; ++s) {
#pragma unroll
        for (int j = 0; j < GROUPS; ++j) {
          acc[0][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[copy][0][s].v, xf[j].v, acc[0][j], 0, 0, 0);
          acc[1][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[copy][1][s].v, xf[j].v, acc[1][j], 0, 0, 0);
          if (s < 3) read(s + 1, j);
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int b = 0; b < 2; ++b) w[copy][b][s].u = *reinterpret_cast<const u32x4*>(from[b] + s * 512 + lane * 8);
        __builtin_amdgcn_sched_barrier(0);
      }
      park_rows(copy ^ 1);
    };
    for (int k0 = 0; k0 < K; k0 += 2 * kStep) {
      step(k0, 0);
      step(k0 + kStep, 1);
    }
  };
  if (groups > 2) walk(std::integral_constant<int, 4>{});
  else walk(std::integral_constant<int, 2>{});
  if (!active) return;
  // acc[b][j][4 i + q]: row 8 i + 4 g + q of the wave's block b, pair 32 j + col
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (32 * j + col >= count) continue;
    const int p = order[start + 32 * j + col];
    if (GATED) {
      const float weight = pair_weight[p];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float v[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float a = on_output ? acc[0][j][4 * i + q] : acc[0][j][4 * i + q] * weight, u = acc[1][j][4 * i + q] * weight;
          v[q] = a / (1.f + expf(-a)) * u;
        }
        store_four<bf16_t>(reinterpret_cast<bf16_t*>(out) + (size_t)p * R + unit * 32 + 8 * i + 4 * g, v[0], v[1], v[2], v[3], 4, true);
      }
    } else {
      float* const dst = reinterpret_cast<float*>(out) + ((size_t)(p % top) * N + p / top) * R + unit * 64 + 4 * g;
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (unit * 64 + 32 * b < R)
            store_four<float>(dst + 32 * b + 8 * i, acc[b][j][4 * i], acc[b][j][4 * i + 1], acc[b][j][4 * i + 2], acc[b][j][4 * i + 3], 4, true);
        }
    }
  }
}

bool sizes_fit(int R, int K, const void* x, const void* weights) {
  return R >= 32 && R % 32 == 0 && K >= 64 && K % 64 == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)weights % 16 == 0;
}

template <bool GATED, int WAVES, int MT>
int launch(const void* x, const void* weights, const int* chosen, const float* pair_weight, void* out, int N, int top, int E, int R,
           int K, int on_output, hipStream_t stream) {
  const int P = N * top;
  moe_stream_kernel<GATED, WAVES, MT><<<dim3(R / 16, counts_met(P, E) ? P : E), WAVES * 64, 0, stream>>>(
      (const bf16_t*)x, (const bf16_t*)weights, chosen, pair_weight, out, N, top, E, R, K, on_output);
  return launch_status();
}

}  // namespace

// gated, x, pair_weight and out as in tk_moe_grouped (moe.hip; gated == 2: the weight acts on the expert's output); chosen
// [N, top]; an expert's weights (gate rows, then up rows) in the order above.  Up to 1,024 pairs.
TK_API int tk_moe_stream(int gated, const void* x, const void* weights, const int* chosen, const float* pair_weight, void* out,
                         int N, int top, int E, int R, int K, hipStream_t stream) {
  if (N <= 0) return 0;
  if (!sizes_fit(R, K, x, weights) || top < 1 || E < 1 || (long)N * top > kMaxPairs) return -1;
#define TK_STREAM(GATED_, WAVES_)                                                                                               \
  (N <= 16 ? launch<GATED_, WAVES_, 1>(x, weights, chosen, pair_weight, out, N, top, E, R, K, gated == 2, stream)               \
   : (long)N * top <= 16L * E ? launch<GATED_, WAVES_, 2>(x, weights, chosen, pair_weight, out, N, top, E, R, K, gated == 2, stream) \
             : launch<GATED_, WAVES_, 4>(x, weights, chosen, pair_weight, out, N, top, E, R, K, gated == 2, stream))
  // (pairs an expert has on average: a pass over 32 pairs keeps two waves a SIMD, one over 64 keeps one and reads an
  // expert's weights half as often; a fuller expert takes another pass)
  if (K > 4 * kChunk) return gated ? TK_STREAM(true, 8) : TK_STREAM(false, 8);
  return gated ? TK_STREAM(true, 4) : TK_STREAM(false, 4);
#undef TK_STREAM
}

// The same products over the tiles of moe_sort (tile_pairs 128); lists as in tk_moe_grouped.
TK_API int tk_moe_tiles(int gated, const void* x, const void* weights, const int* order, const int* tile_expert,
                        const int* tile_start, const int* tile_count, const int* num_tiles, const float* pair_weight, void* out,
                        int N, int top, int R, int K, int max_tiles, int tile_pairs, hipStream_t stream) {
  if (N <= 0 || max_tiles <= 0) return 0;
  if (!sizes_fit(R, K, x, weights) || top < 1 || tile_pairs != kTile) return -1;
  const int channels = (gated ? 32 : 64) * kTileWaves;
  const int channel_blocks = (R + channels - 1) / channels;
  const long total = (long)max_tiles * channel_blocks;
  if (total > 0x7ffffff0L) return -1;
  const dim3 grid((unsigned)((total + kXcds - 1) / kXcds * kXcds));
  const bool odd = K / kStep % 2 != 0;
  const auto kernel = gated ? odd ? moe_tiles_kernel<true, true> : moe_tiles_kernel<true, false>
                            : odd ? moe_tiles_kernel<false, true> : moe_tiles_kernel<false, false>;
  kernel<<<grid, kTileWaves * 64, 0, stream>>>((const bf16_t*)x, (const bf16_t*)weights, order, tile_expert, tile_start, tile_count,
                                               num_tiles, pair_weight, out, N, top, R, K, max_tiles, channel_blocks, gated == 2);
  return launch_status();
}

TK_SLOTS(tk_moe_stream)
TK_SLOTS(tk_moe_tiles)
