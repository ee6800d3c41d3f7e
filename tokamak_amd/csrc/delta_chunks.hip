// The gated delta rule with a decay a key channel, in chunks of 16 tokens on the matrix cores (gfx950): the form of portions
// for the scan of delta.hip, from the rows that delta_inputs leaves there.
//
// The walk's u_i = beta_i (v_i - (diag(a_i) S_(i-1))^T k_i) asks for the u of every token before; over a chunk with start
// state S, with P_i = prod_(l <= i) a_l and M_ij = sum_c k_ic k_jc prod_(j < l <= i) a_lc, that is a system of 16 unknowns:
//   u_i + beta_i sum_(j < i) M_ij u_j = beta_i (v_i - (k_i * P_i)^T S)
//   u = U - W S with U = T V, W = T K', T = (1 + diag(beta) M)^-1 diag(beta), K'_i = k_i * P_i
//   o_i = (q_i * P_i)^T S + sum_(j <= i) A_ij u_j,                         A_ij = sum_c q_ic k_jc prod_(j < l <= i) a_lc
//   S'  = diag(P_16) S + sum_j (k_j * prod_(l > j) a_l) u_j^T
// No product of decays is divided by another: M and A are found in rounds, one for each bit in which i and j differ first (see
// scan_chunks.hip).  T, which no state enters, is found in 64 bits, a column a lane, and rounded once.
//
//   delta_operands: a block a (chunk, head), a wave 64 channels, a lane one channel of 16 tokens.  All chunks side by side.
//   delta_walk: a block a (head, 16 value columns, request), the chunks in order, the state in the waves' accumulators (a
//     wave a quarter of the key channels).
//
// Where the state ends up with numbers that are not finite, the walk repeats the request a token at a time: products of whole tiles
// carry a token's infinity to tokens before it, which no decay may undo.
//
// Requests of `least` tokens and more; shorter ones are the walk's (delta.hip), whoever stands beside them.  Everything is float32.
//
// Walked, a token is a chain of some 430 clocks whatever else the GPU does.  2,048 tokens of 128 x 128: 32 heads 357 us ->
// 75 + 139, 8 heads 349 -> 25 + 128.  The walk in chunks is still its chain: 2,260 clocks a chunk, of which 25 matrix
// instructions of 32 are 800, their results' way back to the vector unit another 300 and the shares' way through LDS 500; u as
// T (V - K' S) had two more steps in it (154), loads that waited for one another at a branch 184.  The operands are bound by
// memory (67 MB in, 140 out) and by the vector unit in like parts; three waves a SIMD spill (85 us), value columns asked for
// behind the stores wait for those (87).
// Against 64 bits: decays as softplus leaves them, 160 to 600 tokens, state 0.60 to 0.78 of the walk's distance, outputs 0.87
// to 1.10 (0.97 on average of eight); without decays 0.4 to 0.7 of both.
#include "common.h"
#include "request_tiles.h"
#include "slots.h"

using namespace tk;

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kTokens = 16;       // tokens of a chunk
constexpr int kMaxDim = 128;
constexpr int kTiles = 2;         // of 16 key channels that a wave of the walk holds (the last of them may not exist)

struct Shape {
  int R, heads, kv, dim, vdim, least;
  // a token's row: [q: kv dim | k: kv dim | v: heads vdim | decay: heads dim | beta: heads], whole 16-byte pieces
  __host__ __device__ int v_at() const { return 2 * kv * dim; }
  __host__ __device__ int g_at() const { return v_at() + heads * vdim; }
  __host__ __device__ int b_at() const { return g_at() + heads * dim; }
  __host__ __device__ int row() const { return (b_at() + heads + 3) / 4 * 4; }
  // per (chunk, head): q * P [16][dim], W [16][dim], k times the decays behind it [dim][16], the chunk's decay [dim], A [j][i],
  // U [vdim][16].  The 16 tokens of W, of the third and of U lie as [token & 3][token >> 2]: a lane's 16 bytes are its operands
  // of four steps, the oldest tokens' first, and u comes out of the matrix unit in the order in which it goes back in.
  __host__ __device__ size_t floats() const { return (size_t)49 * dim + 256 + (size_t)16 * vdim; }
};

__global__ __launch_bounds__(2 * kWave) __attribute__((amdgpu_waves_per_eu(2))) void delta_operands_kernel(const float* __restrict__ in, const int* __restrict__ q_start,
                                                             float* __restrict__ operands, Shape sh) {
  constexpr int kPitch = 64 + 4, kTriPitch = 16 + 4;
  static_assert(kPitch * kTokens >= 512 && kPitch >= kTriPitch, "what follows the rounds lies where they had their rows");
  __shared__ __align__(16) float rows[2][3][kTokens * kPitch];      // [wave][q, then the wave's M and A; k, then T; K']
  RequestTile rt;
  if (!find_request_tile(q_start, sh.R, kTokens, blockIdx.x, rt, sh.least)) return;
  const int head = blockIdx.y, lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int c = threadIdx.x, first = q_start[rt.req] + rt.index * kTokens, n = min(kTokens, q_start[rt.req + 1] - first);
  const bool live = c < sh.dim;
  const int at = min(c, sh.dim - 1), kvh = head / (sh.heads / sh.kv), row = sh.row();
  const float* const x0 = in + (size_t)first * row;
  float* const mine = operands + ((size_t)blockIdx.x * sh.heads + head) * sh.floats();
  float q[kTokens], k[kTokens], a[kTokens];
#pragma unroll
  for (int t = 0; t < kTokens; ++t) {         // (rows past the n-th are the n-th's: all loads in flight together)
    const float* of = x0 + (size_t)min(t, n - 1) * row;
    q[t] = of[kvh * sh.dim + at];
    k[t] = of[(sh.kv + kvh) * sh.dim + at];
    a[t] = of[sh.g_at() + head * sh.dim + at];
  }
  const int x = lane & 15, g = lane >> 4;
  const float beta_of_lane = x < n ? x0[(size_t)x * row + sh.b_at() + head] : 0.f;
  f32x4 v[kMaxDim / 32];           // this wave's tiles of 16 value columns (asked for here: a wait for a load waits for the stores before it, too)
#pragma unroll
  for (int s = 0; s < kMaxDim / 32; ++s) {
    const int v0 = min(16 * (wave + 2 * s), sh.vdim - 16);
#pragma unroll
    for (int r = 0; r < 4; ++r) v[s][r] = x0[(size_t)min(4 * g + r, n - 1) * row + sh.v_at() + head * sh.vdim + v0 + x];
  }
#pragma unroll
  for (int t = 0; t < kTokens; ++t) {         // (tokens past the request's end: nothing enters, nothing decays)
    q[t] = live && t < n ? q[t] : 0.f;
    k[t] = live && t < n ? k[t] : 0.f;
    a[t] = t < n ? a[t] : 1.f;
  }
  float* const ql = rows[wave][0];
  float* const kl = rows[wave][1];
  float* const decayed = rows[wave][2];      // (channels that do not exist are in no product)
  if (live) {
    double p = 1.0;      // (products of decays rounded once: a state lives on)
#pragma unroll
    for (int t = 0; t < kTokens; ++t) {
      p *= a[t];
      mine[t * sh.dim + c] = (float)(q[t] * p);
      decayed[t * kPitch + lane] = (float)(k[t] * p);
    }
    mine[48 * sh.dim + c] = (float)p;
    float* const kt = mine + 32 * sh.dim + (size_t)c * kTokens;
    float s[kTokens];
    p = 1.0;
#pragma unroll
    for (int t = kTokens - 1; t >= 0; --t) {
      s[t] = (float)(k[t] * p);
      p *= a[t];
    }
#pragma unroll
    for (int g = 0; g < 4; ++g) *reinterpret_cast<f32x4*>(kt + 4 * g) = f32x4{s[g], s[g + 4], s[g + 8], s[g + 12]};
  }
  // M and A: lane (i = lane & 15 as a row, j = lane & 15 as a column); D holds column j = lane & 15, rows 4 (lane >> 4) + r
  f32x4 m = {0.f, 0.f, 0.f, 0.f}, av = {0.f, 0.f, 0.f, 0.f};
  const int steps = min(4, sh.dim / 16 - 4 * wave);
#pragma unroll
  for (int round = 0; round < 5; ++round) {
    const int half = round < 4 ? 8 >> round : 0;
#pragma unroll
    for (int t = 0; t < kTokens; ++t) asm volatile("" : "+v"(a[t]));      // (products kept from round to round are more registers than there are)
    // rows of the upper halves get the decays from the middle to themselves, rows of the lower halves those to the middle
#pragma unroll
    for (int t = 0; t < kTokens; ++t) {
      float p = 1.f;
      if (half != 0 && (t & half)) {
#pragma unroll
        for (int l = t & ~(half - 1); l <= t; ++l) p *= a[l];
      } else if (half != 0) {
#pragma unroll
        for (int l = t + 1; l < ((t & ~(half - 1)) + half); ++l) p *= a[l];
      }
      if (half == 0 || (t & half)) ql[t * kPitch + lane] = q[t] * p;       // (lower rows: as they are, their products are dropped)
      kl[t * kPitch + lane] = k[t] * p;
    }
    wave_lds_sync();
    f32x4 acc_a = {0.f, 0.f, 0.f, 0.f}, acc_m = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int s = 0; s < steps; ++s) {       // (sums of eight channels each, then these: no more roundings than the walk's)
      const f32x4 qv = *reinterpret_cast<const f32x4*>(ql + x * kPitch + 16 * s + 4 * g);
      const f32x4 kv = *reinterpret_cast<const f32x4*>(kl + x * kPitch + 16 * s + 4 * g);
      f32x4 sum_a[2], sum_m[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) sum_a[h] = sum_m[h] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        sum_a[r & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(qv[r], kv[r], sum_a[r & 1], 0, 0, 0);
        if (half != 0) sum_m[r & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[r], kv[r], sum_m[r & 1], 0, 0, 0);
      }
      acc_a += sum_a[0] + sum_a[1];
      acc_m += sum_m[0] + sum_m[1];
    }
    wave_lds_sync();
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = 4 * g + r, j = x, bits = i ^ j;
      const bool here = half == 0 ? i == j : (i > j && bits >= half && bits < 2 * half);
      if (here) av[r] = acc_a[r];
      if (here && half != 0) m[r] = acc_m[r];
    }
  }
  *reinterpret_cast<f32x4*>(ql + 4 * lane) = m;
  *reinterpret_cast<f32x4*>(ql + 256 + 4 * lane) = av;
  __syncthreads();
  m = *reinterpret_cast<const f32x4*>(rows[0][0] + 4 * lane) + *reinterpret_cast<const f32x4*>(rows[1][0] + 4 * lane);
  av = *reinterpret_cast<const f32x4*>(rows[0][0] + 256 + 4 * lane) + *reinterpret_cast<const f32x4*>(rows[1][0] + 256 + 4 * lane);
  if (wave == 0) *reinterpret_cast<f32x4*>(mine + 49 * sh.dim + x * 16 + 4 * g) = av;
  // either wave finds T, column x a lane (its four groups of lanes the same), from above
  float* const tr = kl;
#pragma unroll
  for (int r = 0; r < 4; ++r) tr[(4 * g + r) * kTriPitch + x] = m[r];
  wave_lds_sync();
  double t[kTokens];
  f32x4 line[2][4];      // a row of M, the next one on its way (all at once are more registers than there are)
#pragma unroll
  for (int i = 0; i < kTokens; ++i) {
    if (i + 1 < kTokens) {
#pragma unroll
      for (int l = 0; l <= i; l += 4) line[(i + 1) & 1][l / 4] = *reinterpret_cast<const f32x4*>(tr + (i + 1) * kTriPitch + l);
    }
    __builtin_amdgcn_sched_barrier(0);
    double sum = i == x ? 1.0 : 0.0;
#pragma unroll
    for (int l = 0; l < i; ++l) sum -= (double)line[i & 1][l / 4][l % 4] * t[l];
    t[i] = (double)__shfl(beta_of_lane, i, kWave) * sum;
  }
  wave_lds_sync();
#pragma unroll
  for (int i = 0; i < kTokens; ++i)
    if ((i & 3) == g) tr[(4 * (i & 3) + (i >> 2)) * kTriPitch + x] = (float)t[i];
  wave_lds_sync();
  const f32x4 tv = *reinterpret_cast<const f32x4*>(tr + x * kTriPitch + 4 * g);      // row x, columns 4 g + step
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    if (s >= steps) continue;
    f32x4 w = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 4; ++r) w = __builtin_amdgcn_mfma_f32_16x16x4f32(tv[r], decayed[(4 * g + r) * kPitch + 16 * s + x], w, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 4; ++r) mine[(16 + 4 * g + r) * sh.dim + wave * kWave + 16 * s + x] = w[r];
  }
#pragma unroll
  for (int s = 0; s < kMaxDim / 32; ++s) {
    const int v0 = 16 * (wave + 2 * s);
    if (v0 >= sh.vdim) continue;
    f32x4 u = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 4; ++r) u = __builtin_amdgcn_mfma_f32_16x16x4f32(tv[r], v[s][r], u, 0, 0, 0);
    *reinterpret_cast<f32x4*>(mine + 49 * sh.dim + 256 + (size_t)(v0 + x) * kTokens + 4 * g) = u;
  }
}

struct WalkIn {        // a chunk's operands as a lane of the walk holds them
  f32x4 q[kTiles], w[kTiles], k[kTiles], d[kTiles], u;
  float a;
};

// Four waves; wave w holds the tiles w and w + 4 of 16 key channels of the block's 16 value columns: S[i][r] is
// channel 16 tile + 4 (lane >> 4) + r of column lane & 15.  One barrier a chunk: the waves' shares of W S meet behind it, their
// shares of the outputs behind the next chunk's.  Operands are asked for kAhead chunks ahead, without a branch around any load.
constexpr int kAhead = 4;
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void delta_walk_kernel(const float* __restrict__ in, const float* __restrict__ operands,
                                                         float* __restrict__ state, const int* __restrict__ q_start,
                                                         const int* __restrict__ state_slots, float* __restrict__ y, Shape sh) {
  __shared__ __align__(16) float seen[2][4][256];     // shares of W S
  __shared__ __align__(16) float outs[2][4][256];     // shares of the outputs
  const int head = blockIdx.x, v0 = blockIdx.y * 16, req = blockIdx.z;
  const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), x = lane & 15, g = lane >> 4;
  const int first = q_start[req], end = q_start[req + 1], chunks = request_tiles(q_start, req, kTokens, sh.least);
  if (chunks == 0) return;
  const int before = tiles_before(q_start, req, kTokens, sh.least);
  const float* op = operands + ((size_t)before * sh.heads + head) * sh.floats();
  const size_t pitch = sh.heads * sh.floats();
  float* const S = state + (((size_t)state_slots[req] * sh.heads + head) * sh.vdim + v0 + x) * sh.dim;
  bool have[kTiles];
  int channel[kTiles];       // the first of a tile's channels (of a tile that exists: loads need no branch)
  f32x4 s[kTiles];
#pragma unroll
  for (int i = 0; i < kTiles; ++i) {
    have[i] = 16 * (wave + 4 * i) < sh.dim;
    channel[i] = have[i] ? 16 * (wave + 4 * i) : 0;
    s[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (have[i]) s[i] = *reinterpret_cast<const f32x4*>(S + channel[i] + 4 * g);
  }
  // (a chunk's numbers from a scalar address on, at 32-bit offsets a lane keeps: no address arithmetic in the walk)
  uint32_t row_at[kTiles], key_at[kTiles], decay_at[kTiles];
#pragma unroll
  for (int i = 0; i < kTiles; ++i) {
    row_at[i] = (x * sh.dim + channel[i] + 4 * g) * 4;
    key_at[i] = ((channel[i] + x) * kTokens + 4 * g) * 4;
    decay_at[i] = (channel[i] + 4 * g) * 4;
  }
  uint32_t a_at = threadIdx.x * 4, u_at = ((v0 + x) * kTokens + 4 * g) * 4;
  const auto at = [](const char* base, uint32_t& offset) {
    asm volatile("" : "+v"(offset));      // (widened here, where the load can take a scalar base and a 32-bit offset)
    return base + offset;
  };
  const auto fetch = [&](int ci, WalkIn& in) {
    const char* const o = reinterpret_cast<const char*>(op + (size_t)min(ci, chunks - 1) * pitch);
    const uint32_t rows = 64 * sh.dim;      // bytes of 16 rows of channels
#pragma unroll
    for (int i = 0; i < kTiles; ++i) in.w[i] = *reinterpret_cast<const f32x4*>(at(o + rows, row_at[i]));
#pragma unroll
    for (int i = 0; i < kTiles; ++i) in.q[i] = *reinterpret_cast<const f32x4*>(at(o, row_at[i]));
    in.u = *reinterpret_cast<const f32x4*>(at(o + 3 * rows + 4 * sh.dim + 1024, u_at));
#pragma unroll
    for (int i = 0; i < kTiles; ++i) in.k[i] = *reinterpret_cast<const f32x4*>(at(o + 2 * rows, key_at[i]));
#pragma unroll
    for (int i = 0; i < kTiles; ++i) in.d[i] = *reinterpret_cast<const f32x4*>(at(o + 3 * rows, decay_at[i]));
    in.a = *reinterpret_cast<const float*>(at(o + 3 * rows + 4 * sh.dim, a_at));
  };
  const auto sum_of = [&](int half) {      // token 4 wave + g of a chunk: register g of lanes 16 wave ..
    const float* p = &outs[half][0][(wave * 16 + x) * 4 + g];
    return ((p[0] + p[256]) + p[512]) + p[768];
  };
  const int mine_at = 4 * wave + g, tokens = end - first, VW = sh.heads * sh.vdim;
  float* const y_first = y + (size_t)first * VW + head * sh.vdim;
  uint32_t y_at = (mine_at * VW + v0 + x) * 4;
  const auto put = [&](int ci, float sum) {
    if (ci >= 0 && ci * kTokens + mine_at < tokens) {
      asm volatile("" : "+v"(y_at));
      *reinterpret_cast<float*>(reinterpret_cast<char*>(y_first + (size_t)ci * kTokens * VW) + y_at) = sum;
    }
  };
  constexpr int kSums = 4 / kTiles;
  const bool odd = threadIdx.x & kWave, upper = threadIdx.x & (2 * kWave);      // (of the wave's number, as lane masks: no branches)
  WalkIn ahead[kAhead];
#pragma unroll
  for (int u = 0; u < kAhead; ++u) {
    fetch(u, ahead[u]);
    __builtin_amdgcn_sched_barrier(0);      // (in this order: what the loop's first chunk waits for is then the oldest)
  }
  int c0 = 0;
  do {      // (there is a chunk: without a branch ahead of the loop the loads above stay in their order)
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      // (no branch around a chunk: the loads in flight would be waited for there.  One past the last leaves nothing behind)
      const int ci = c0 + u;
      const WalkIn& now = ahead[u];
      f32x4 ks[4], o[4];      // (sums of eight channels each, then a tree: no more roundings than the walk's)
#pragma unroll
      for (int i = 0; i < 4; ++i) ks[i] = o[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int i = 0; i < kTiles; ++i) {
          f32x4& sum = ks[i * kSums + r % kSums];
          sum = __builtin_amdgcn_mfma_f32_16x16x4f32(now.w[i][r], s[i][r], sum, 0, 0, 0);
        }
      *reinterpret_cast<f32x4*>(&seen[u & 1][wave][4 * lane]) = (ks[0] + ks[1]) + (ks[2] + ks[3]);
      __syncthreads();      // (one a chunk: either copy is written again behind the next chunk's barrier)
      f32x4 rest[4];
#pragma unroll
      for (int w = 0; w < 4; ++w) rest[w] = *reinterpret_cast<const f32x4*>(&seen[u & 1][w][4 * lane]);
      const float sum = sum_of((u & 1) ^ 1);
      __builtin_amdgcn_sched_barrier(0);
      // (q' S while the shares come from LDS)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int i = 0; i < kTiles; ++i) {
          f32x4& sum = o[i * kSums + r % kSums];
          sum = __builtin_amdgcn_mfma_f32_16x16x4f32(now.q[i][r], s[i][r], sum, 0, 0, 0);
        }
      const f32x4 un = now.u - ((rest[0] + rest[1]) + (rest[2] + rest[3]));      // u of token 4 r + g in register r
      put(ci < chunks + 1 ? ci - 1 : -1, sum);
      f32x4 own[kTiles];
#pragma unroll
      for (int i = 0; i < kTiles; ++i) own[i] = f32x4{0.f, 0.f, 0.f, 0.f};
      // the chunk's tokens by themselves, oldest first, then the decayed state: one rounding of the state a chunk
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int i = 0; i < kTiles; ++i) own[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(now.k[i][r], un[r], own[i], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < kTiles; ++i) {
#pragma unroll
        for (int r = 0; r < 4; ++r) own[i][r] = fmaf(now.d[i][r], s[i][r], own[i][r]);
      }
      const float low = odd ? un[1] : un[0], high = odd ? un[3] : un[2], mine = upper ? high : low;
      const f32x4 far = (o[0] + o[1]) + (o[2] + o[3]);
      *reinterpret_cast<f32x4*>(&outs[u & 1][wave][4 * lane]) = __builtin_amdgcn_mfma_f32_16x16x4f32(now.a, mine, far, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      fetch(ci + kAhead, ahead[u]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < kTiles; ++i) {
        const uint32_t moves = have[i] && ci < chunks ? ~0u : 0u;      // (bits, not a condition: no branch)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          s[i][r] = __uint_as_float((__float_as_uint(own[i][r]) & moves) | (__float_as_uint(s[i][r]) & ~moves));
      }
    }
    c0 += kAhead;
  } while (c0 < chunks);
  __syncthreads();
  if (chunks % kAhead == 0) put(chunks - 1, sum_of((chunks - 1) & 1));      // (else a turn past the last chunk has put them)
  // A number that is not finite has met the zeros of T, A and the rows past the end above, and made tokens before its own NaN.  It
  // stays in the state: the request again, then, a token at a time, from the state as it was.
  bool lost = false;
#pragma unroll
  for (int i = 0; i < kTiles; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) lost |= !(fabsf(s[i][r]) < INFINITY);
  if (__syncthreads_or(lost)) {
#pragma unroll
    for (int i = 0; i < kTiles; ++i)
      if (have[i]) s[i] = *reinterpret_cast<const f32x4*>(S + channel[i] + 4 * g);
    const int kvh = head / (sh.heads / sh.kv);
    const float* row = in + (size_t)first * sh.row();
    for (int t = 0; t < tokens; ++t, row += sh.row()) {
      const float v = row[sh.v_at() + head * sh.vdim + v0 + x], beta = row[sh.b_at() + head];
      f32x4 k[kTiles], q[kTiles];
      float sum = 0.f;
#pragma unroll
      for (int i = 0; i < kTiles; ++i) {
        if (!have[i]) continue;
        q[i] = *reinterpret_cast<const f32x4*>(row + kvh * sh.dim + channel[i] + 4 * g);
        k[i] = *reinterpret_cast<const f32x4*>(row + (sh.kv + kvh) * sh.dim + channel[i] + 4 * g);
        s[i] *= *reinterpret_cast<const f32x4*>(row + sh.g_at() + head * sh.dim + channel[i] + 4 * g);
#pragma unroll
        for (int r = 0; r < 4; ++r) sum = fmaf(k[i][r], s[i][r], sum);
      }
      sum = sum32(sum16(sum));
      if (g == 0) seen[t & 1][wave][x] = sum;
      __syncthreads();      // (either copy is written again behind the next token's barriers)
      const float* const before_u = &seen[t & 1][0][x];
      const float u = beta * (v - (((before_u[0] + before_u[256]) + before_u[512]) + before_u[768]));
      sum = 0.f;
#pragma unroll
      for (int i = 0; i < kTiles; ++i) {
        if (!have[i]) continue;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          s[i][r] = fmaf(k[i][r], u, s[i][r]);
          sum = fmaf(q[i][r], s[i][r], sum);
        }
      }
      sum = sum32(sum16(sum));
      if (g == 0) outs[t & 1][wave][x] = sum;
      __syncthreads();
      // (by the thread that has put this token's output above)
      const float* const all = &outs[t & 1][0][x];
      if ((t & (kTokens - 1)) == mine_at) y_first[(size_t)t * VW + v0 + x] = ((all[0] + all[256]) + all[512]) + all[768];
    }
  }
#pragma unroll
  for (int i = 0; i < kTiles; ++i)
    if (have[i]) *reinterpret_cast<f32x4*>(S + channel[i] + 4 * g) = s[i];
}

}  // namespace

// in, state, y as in tk_delta_scan (delta.hip); dim (80 to 128) and vdim (up to 128) multiples of 16, in and state on 16-byte borders.  least:
// requests of fewer tokens are left alone; chunks: at least the chunks of 16 tokens that the others have together; operands
// (float32 [chunks, heads, 49 dim + 16 vdim + 256], on a 16-byte border) is scratch.
TK_API int tk_delta_chunks(const float* in, float* state, const int* q_start, const int* state_slots, float* y, float* operands,
                           int R, int least, int chunks, int heads, int kv, int dim, int vdim, hipStream_t stream) {
  if (R <= 0) return 0;
  if (heads < 1 || heads > 65535 || kv < 1 || heads % kv || dim <= kWave || dim > kMaxDim || dim % 16 || vdim < 16 || vdim > kMaxDim ||
      vdim % 16 || least < 1 || chunks < 1 || R > 65535 || operands == nullptr || (uintptr_t)in % 16 || (uintptr_t)state % 16 ||
      (uintptr_t)operands % 16)
    return -1;
  const Shape sh{R, heads, kv, dim, vdim, least};
  delta_operands_kernel<<<dim3(chunks, heads), 2 * kWave, 0, stream>>>(in, q_start, operands, sh);
  // (heads the fastest index: the value columns' blocks of a head, which read the same operands, then share an XCD's L2
  // where the heads are a multiple of eight)
  const dim3 walks(heads, vdim / 16, R);
  delta_walk_kernel<<<walks, 256, 0, stream>>>(in, operands, state, q_start, state_slots, y, sh);
  return launch_status();
}

TK_SLOTS(tk_delta_chunks)
