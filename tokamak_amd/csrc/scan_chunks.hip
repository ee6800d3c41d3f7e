// Linear recurrences with a decay a key channel, in chunks of 16 tokens on the matrix cores (gfx950): the form of
// portions for the two scans of recurrent.hip, bfloat16 storage.
//
//   gla:  S <- diag(a_t) S + k_t v_t^T,  o_t = S^T (q_t * q_scale)                 a_t = sigmoid(z_t + bias)^(1/tau)
//   wkv:  o_t = (S + diag(u) k_t v_t^T)^T r_t,  S <- diag(a_t) S + k_t v_t^T       a_t = exp(-exp(d_t + w0))
//
// A chunk with start state S (gla; for wkv the products over l run to i - 1 and the diagonal is r u k):
//   o_i = (q_i * prod_(l <= i) a_l)^T S + sum_(j <= i) M_ij v_j,    M_ij = sum_c q_ic k_jc prod_(j < l <= i) a_lc
//   S'  = diag(prod a_l) S + sum_j (k_j * prod_(l > j) a_l) v_j^T
// No product of decays is ever divided by another: M is found in five rounds, one for each bit in which i and j
// differ first and one for i = j: the product over j < l <= i is cut at the middle of the block that parts them, so both
// factors are products of decays, at most one, and each round is a plain matrix product of scaled rows.
//
// Requests of `least` tokens and more; shorter ones are the walk's (recurrent.hip), whoever stands beside them.
//
//   chunk_operands: a block a (chunk, head), a wave 64 channels, a lane one channel of 16 tokens: decays, the scaled
//     rows q' and k', the whole chunk's decay, M.  All chunks side by side.
//   chunk_walk: a block a (head, 16 value columns, request), the chunks in order, the state in the waves' accumulators
//     (a wave a quarter of the key channels), outputs before the norm, float32.
//   chunk_finish: norm, gain, gate.
//
// Walked a token at a time a token costs a chain of some 0.5 to 0.7 us; a chunk of 16 costs a chain of two short matrix
// products and a barrier.  2,048 tokens: gla, 32 heads of 128 x 128, 1.45 ms -> 68 + 111 + 23 us; wkv, 64 heads of 64 x
// 64, 1.10 ms -> 61 + 70 + 23.  The operands kernel of gla is bound by the vector unit (85 % of its time busy: logarithms and
// exponentials), of wkv by neither (45 %; in 33 MB, out 105); the walk by its chain (0.9 us a chunk of 128 x 16 state a
// block: 17 matrix instructions of 32 cycles a wave, LDS, barrier; matrix units 29 % busy, vector 20 %).  Everything
// is float32, the products are those of the float32 matrix instruction (16 x 16 x 4); its k index may name any four
// channels as long as both operands agree, so index g of step r is channel 4 g + r: a lane's operands are then
// the parts of one 16-byte load, and the state's accumulators are an operand as they are.
// The state's distance from 64 bits is the walk's or less (0.90 to 1.00 with decays of a half and more a token): a chunk
// rounds it five times, not 16, products of decays are rounded once, and tokens enter in their order, so that what is rounded before
// the newest, which weigh most, is small.  (The state as the accumulator of all 16 tokens, products of decays rounded at each
// factor: 1.03 to 1.24.  Where nothing outlives a token the walk rounds once and a chunk up to twice: to 1.16 of 2.4e-8.)
#include "common.h"
#include "request_tiles.h"
#include "slots.h"

using namespace tk;

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kTokens = 16;       // tokens of a chunk
constexpr int kMaxDim = 128;

struct In {                       // an operand [N, width]: T, or float32, or float32 partial sums of a split product
  const void* p;
  int f32, parts;
  long stride;
};

__device__ __forceinline__ float load(const In& in, size_t idx) {
  if (!in.f32) return Elem<bf16_t>::load(reinterpret_cast<const bf16_t*>(in.p) + idx);
  const float* f = reinterpret_cast<const float*>(in.p) + idx;
  float s = f[0];
  for (int i = 1; i < in.parts; ++i) s += f[(size_t)i * in.stride];
  return s;
}

// Column `col` of the 16 rows of a chunk, all loads in flight together (a load behind a branch of its own is waited for
// there); rows past the n-th are the n-th's.
__device__ __forceinline__ void load_column(const In& in, size_t first, int n, size_t ld, size_t col, float (&x)[kTokens]) {
  if (!in.f32) {
    const bf16_t* p = reinterpret_cast<const bf16_t*>(in.p) + first * ld + col;
#pragma unroll
    for (int t = 0; t < kTokens; ++t) x[t] = Elem<bf16_t>::load(p + min(t, n - 1) * ld);
    return;
  }
  const float* p = reinterpret_cast<const float*>(in.p) + first * ld + col;
#pragma unroll
  for (int t = 0; t < kTokens; ++t) x[t] = p[min(t, n - 1) * ld];
  for (int i = 1; i < in.parts; ++i) {
#pragma unroll
    for (int t = 0; t < kTokens; ++t) x[t] += p[(size_t)i * in.stride + min(t, n - 1) * ld];
  }
}

struct Shape {
  int R, heads, dim, vdim, least;
  // per (chunk, head): q' [16][dim], k' [dim][16], the chunk's decay [dim], M (see chunk_operands), v [vdim][16]; the 16
  // tokens of k' and v lie as [token & 3][token >> 2], so that a lane's 16 bytes are its operands of four steps, the oldest
  // tokens' first
  __host__ __device__ size_t floats() const { return (size_t)33 * dim + 256 + (size_t)16 * vdim; }
};

// WKV: the state is read before a token enters it, and the token's own term has its weights u
template <bool WKV>
__global__ __launch_bounds__(128) void chunk_operands_kernel(In q_in, In k_in, In v_in, In d_in, const float* __restrict__ bias,
                                                             const float* __restrict__ u, const int* __restrict__ q_start,
                                                             float* __restrict__ operands, Shape sh, float q_scale, float inv_tau) {
  constexpr int kPitch = 64 + 4;
  __shared__ __align__(16) float rows[2][2][kTokens * kPitch];      // [wave][q', k']
  __shared__ float other[256];
  RequestTile rt;
  if (!find_request_tile(q_start, sh.R, kTokens, blockIdx.x, rt, sh.least)) return;
  const int head = blockIdx.y, lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const int c = threadIdx.x, first = q_start[rt.req] + rt.index * kTokens, n = min(kTokens, q_start[rt.req + 1] - first);
  const bool live = c < sh.dim;
  const int col = head * sh.dim + min(c, sh.dim - 1);
  const size_t KW = (size_t)sh.heads * sh.dim;
  float* const mine = operands + ((size_t)blockIdx.x * sh.heads + head) * sh.floats();
  if (c < sh.vdim) {
    float v[kTokens];
    load_column(v_in, first, n, (size_t)sh.heads * sh.vdim, head * sh.vdim + c, v);
    float* const vt = mine + 33 * sh.dim + 256 + (size_t)c * kTokens;
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<f32x4*>(vt + 4 * g) = f32x4{g < n ? v[g] : 0.f, g + 4 < n ? v[g + 4] : 0.f, g + 8 < n ? v[g + 8] : 0.f, g + 12 < n ? v[g + 12] : 0.f};
  }
  float q[kTokens], k[kTokens], a[kTokens];
  load_column(q_in, first, n, KW, col, q);
  load_column(k_in, first, n, KW, col, k);
  load_column(d_in, first, n, KW, col, a);
#pragma unroll
  for (int t = 0; t < kTokens; ++t) {
    q[t] = live && t < n ? q[t] : 0.f;
    k[t] = live && t < n ? k[t] : 0.f;
  }
  const float b = live ? bias[col] : 0.f, own = WKV && live ? u[col] : 1.f;
#pragma unroll
  for (int t = 0; t < kTokens; ++t) {
    if (!WKV) q[t] *= q_scale;
    const float x = a[t] + b;
    // (tokens past the request's end: nothing enters, nothing decays)
    const float d = WKV ? expf(-expf(x)) : expf(-(fmaxf(-x, 0.f) + log1pf(expf(-fabsf(x)))) * inv_tau);
    a[t] = t < n ? d : 1.f;
  }
  if (live) {
    double p = 1.0;      // (products of decays rounded once: a state lives on, see chunk_walk)
#pragma unroll
    for (int t = 0; t < kTokens; ++t) {
      if (!WKV) p *= a[t];
      mine[t * sh.dim + c] = (float)(q[t] * p);
      if (WKV) p *= a[t];
    }
    mine[32 * sh.dim + c] = (float)p;
    float* const kt = mine + 16 * sh.dim + (size_t)c * kTokens;
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
  // M: lane (i = lane & 15 as a row, j = lane & 15 as a column); D holds column j = lane & 15, rows 4 (lane >> 4) + r
  float* const ql = rows[wave][0];
  float* const kl = rows[wave][1];
  const int x = lane & 15, g = lane >> 4;
  f32x4 m = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int round = 0; round < 5; ++round) {
    const int half = round < 4 ? 8 >> round : 0;
    // rows of the upper halves get the decays from the middle to themselves, rows of the lower halves those to the middle
#pragma unroll
    for (int t = 0; t < kTokens; ++t) {
      if (half == 0) {
        ql[t * kPitch + lane] = q[t];
        kl[t * kPitch + lane] = k[t] * own;
      } else if (t & half) {
        float p = 1.f;
#pragma unroll
        for (int l = t & ~(half - 1); l < t + (WKV ? 0 : 1); ++l) p *= a[l];
        ql[t * kPitch + lane] = q[t] * p;
      } else {
        float p = 1.f;
#pragma unroll
        for (int l = t + 1; l < ((t & ~(half - 1)) + half); ++l) p *= a[l];
        kl[t * kPitch + lane] = k[t] * p;
      }
    }
    wave_lds_sync();
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    const int steps = max(0, min(4, (sh.dim - wave * kWave + 15) / 16));
    for (int s = 0; s < steps; ++s) {
      const f32x4 av = *reinterpret_cast<const f32x4*>(ql + x * kPitch + 16 * s + 4 * g);
      const f32x4 bv = *reinterpret_cast<const f32x4*>(kl + x * kPitch + 16 * s + 4 * g);
#pragma unroll
      for (int r = 0; r < 4; ++r) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(av[r], bv[r], acc, 0, 0, 0);
    }
    wave_lds_sync();
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = 4 * g + r, j = x, part = i ^ j;
      if (half == 0 ? i == j : (i > j && part >= half && part < 2 * half)) m[r] = acc[r];
    }
  }
  if (wave == 1) {
#pragma unroll
    for (int r = 0; r < 4; ++r) other[(4 * g + r) * 16 + x] = m[r];
  }
  __syncthreads();
  if (wave == 0) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = 4 * g + r;
      if (blockDim.x > kWave) m[r] += other[i * 16 + x];
      // [j >> 2][j & 3][i]: step j >> 2 of the walk's product reads 64 numbers in its lanes' order
      mine[33 * sh.dim + x * 16 + i] = m[r];
    }
  }
}

template <int TILES>
struct WalkIn {        // a chunk's operands as a lane of the walk holds them
  f32x4 q[TILES], k[TILES], d[TILES], v;
  float m;
};

// Four waves; wave w holds the tiles w and (TILES 2) w + 4 of 16 key channels of the block's 16 value columns: S[i][r] is
// channel 16 tile + 4 (lane >> 4) + r of column lane & 15.  A wave has a SIMD to itself and a chunk is some 600 cycles of
// work, less than a load takes: the operands are asked for kAhead chunks ahead, without a branch around any load
// (one chunk ahead and values behind branches: 2 us a chunk).
constexpr int kAhead = 4;
template <int TILES>
__global__ __launch_bounds__(256) void chunk_walk_kernel(const float* __restrict__ operands, float* __restrict__ state,
                                                         const int* __restrict__ q_start, const int* __restrict__ state_slots,
                                                         float* __restrict__ raw, Shape sh) {
  __shared__ float part[2][4][256];
  const int head = blockIdx.x, v0 = blockIdx.y * 16, req = blockIdx.z;
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave, x = lane & 15, g = lane >> 4;
  const int first = q_start[req], end = q_start[req + 1], chunks = request_tiles(q_start, req, kTokens, sh.least);
  if (chunks == 0) return;
  const int before = tiles_before(q_start, req, kTokens, sh.least);
  const float* op = operands + ((size_t)before * sh.heads + head) * sh.floats();
  const size_t pitch = sh.heads * sh.floats();
  const int VW = sh.heads * sh.vdim;
  float* const S = state + ((size_t)state_slots[req] * sh.heads + head) * sh.dim * sh.vdim + v0 + x;
  bool have[TILES];
  int channel[TILES];       // the first of a tile's channels (of a tile that exists: loads need no branch)
  f32x4 s[TILES];
#pragma unroll
  for (int i = 0; i < TILES; ++i) {
    have[i] = 16 * (wave + 4 * i) < sh.dim;
    channel[i] = have[i] ? 16 * (wave + 4 * i) : 0;
#pragma unroll
    for (int r = 0; r < 4; ++r) s[i][r] = have[i] ? S[(size_t)(channel[i] + 4 * g + r) * sh.vdim] : 0.f;
  }
  const auto fetch = [&](int ci, WalkIn<TILES>& w) {
    const float* o = op + (size_t)min(ci, chunks - 1) * pitch;
#pragma unroll
    for (int i = 0; i < TILES; ++i) {
      w.q[i] = *reinterpret_cast<const f32x4*>(o + x * sh.dim + channel[i] + 4 * g);
      w.k[i] = *reinterpret_cast<const f32x4*>(o + 16 * sh.dim + (size_t)(channel[i] + x) * kTokens + 4 * g);
      w.d[i] = *reinterpret_cast<const f32x4*>(o + 32 * sh.dim + channel[i] + 4 * g);
    }
    w.m = o[33 * sh.dim + wave * 64 + lane];
    w.v = *reinterpret_cast<const f32x4*>(o + 33 * sh.dim + 256 + (size_t)(v0 + x) * kTokens + 4 * g);
  };
  WalkIn<TILES> in[kAhead];
#pragma unroll
  for (int u = 0; u < kAhead; ++u) fetch(u, in[u]);
  for (int c0 = 0; c0 < chunks; c0 += kAhead) {
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      const int ci = c0 + u;
      if (ci >= chunks) break;          // (the whole block alike)
      const WalkIn<TILES> now = in[u];
      // outputs: this wave's channels of q' S, and its step of M v
      f32x4 o[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int i = 0; i < TILES; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) o[i & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(now.q[i][r], s[i][r], o[i & 1], 0, 0, 0);
      const float mv = wave == 0 ? now.v[0] : wave == 1 ? now.v[1] : wave == 2 ? now.v[2] : now.v[3];
      o[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(now.m, mv, o[1], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < TILES; ++i) {
        if (have[i]) {
          // twelve tokens by themselves, then the decayed state joins, then the newest four, which weigh most
          f32x4 own = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int r = 0; r < 3; ++r) own = __builtin_amdgcn_mfma_f32_16x16x4f32(now.k[i][r], now.v[r], own, 0, 0, 0);
#pragma unroll
          for (int r = 0; r < 4; ++r) own[r] = fmaf(now.d[i][r], s[i][r], own[r]);
          s[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(now.k[i][3], now.v[3], own, 0, 0, 0);
        }
      }
      fetch(ci + kAhead, in[u]);
      float* const p = part[u & 1][wave];
#pragma unroll
      for (int r = 0; r < 4; ++r) p[(4 * g + r) * 16 + x] = o[0][r] + o[1][r];
      __syncthreads();      // (one a chunk: this copy is written again behind the next chunk's barrier)
      const int t = first + ci * kTokens + (int)threadIdx.x / 16;
      const float* sum = &part[u & 1][0][threadIdx.x];
      const float y = ((sum[0] + sum[256]) + sum[512]) + sum[768];
      if (t < end) raw[(size_t)t * VW + head * sh.vdim + v0 + (threadIdx.x & 15)] = y;
    }
  }
#pragma unroll
  for (int i = 0; i < TILES; ++i)
    if (have[i])
#pragma unroll
      for (int r = 0; r < 4; ++r) S[(size_t)(channel[i] + 4 * g + r) * sh.vdim] = s[i][r];
}

// out = o / rms(o) * gain * silu(gate) per (token, head) of a chunk: `lanes` lanes a head, four channels each (bound by its
// bytes)
__global__ __launch_bounds__(256) void chunk_finish_kernel(const float* __restrict__ raw, In g_in, const float* __restrict__ gain,
                                                           const int* __restrict__ q_start, bf16_t* __restrict__ out, Shape sh,
                                                           int gain_heads, int lanes, float eps) {
  RequestTile rt;
  if (!find_request_tile(q_start, sh.R, kTokens, blockIdx.x, rt, sh.least)) return;
  const int first = q_start[rt.req] + rt.index * kTokens, n = min(kTokens, q_start[rt.req + 1] - first), vdim = sh.vdim;
  const int at_lane = threadIdx.x % lanes, c = 4 * at_lane;
  const int pair = blockIdx.y * (blockDim.x / lanes) + threadIdx.x / lanes;      // (token of the chunk) * heads + head
  const bool live = pair < n * sh.heads && c < vdim;
  const size_t at = ((size_t)first * sh.heads + pair) * vdim + c;
  f32x4 o = {0.f, 0.f, 0.f, 0.f};
  if (live) o = *reinterpret_cast<const f32x4*>(raw + at);
  float sq = o[0] * o[0] + o[1] * o[1] + o[2] * o[2] + o[3] * o[3];
  for (int m = lanes / 2; m >= 1; m >>= 1) sq += __shfl_xor(sq, m, kWave);
  if (!live) return;
  const float rstd = 1.f / sqrtf(sq / (float)vdim + eps);
  const f32x4 gn = *reinterpret_cast<const f32x4*>(gain + (pair % sh.heads % gain_heads) * vdim + c);
  float y[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float g = load(g_in, at + r);
    y[r] = o[r] * rstd * gn[r] * (g / (1.f + expf(-g)));
  }
  *reinterpret_cast<uint2*>(out + at) = make_uint2(pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3]));
}

int launch(bool wkv, In q, In k, In v, In g, In d, const float* bias, const float* u, const float* gain, int gain_heads, float* state,
           const int* q_start, const int* slots, void* out, float* operands, float* raw, int N, int chunks, Shape sh, float q_scale,
           float inv_tau, float eps, hipStream_t stream) {
  if (sh.R <= 0 || N <= 0) return 0;
  if (sh.heads < 1 || sh.heads > 65535 || sh.dim < 16 || sh.dim > kMaxDim || sh.dim % 16 || sh.vdim < 16 || sh.vdim > kMaxDim ||
      sh.vdim % 16 || sh.least < 1 || chunks < 1 || operands == nullptr || raw == nullptr)
    return -2;
  const dim3 per_chunk(chunks, sh.heads);
  const int threads = (max(sh.dim, sh.vdim) + kWave - 1) / kWave * kWave;
  if (wkv) chunk_operands_kernel<true><<<per_chunk, threads, 0, stream>>>(q, k, v, d, bias, u, q_start, operands, sh, q_scale, inv_tau);
  else chunk_operands_kernel<false><<<per_chunk, threads, 0, stream>>>(q, k, v, d, bias, u, q_start, operands, sh, q_scale, inv_tau);
  // (heads the fastest index: the value columns' blocks of a head, which read the same operands, then share an XCD's L2
  // where the heads are a multiple of eight)
  const dim3 walks(sh.heads, sh.vdim / 16, sh.R);
  if (sh.dim <= 64) chunk_walk_kernel<1><<<walks, 256, 0, stream>>>(operands, state, q_start, slots, raw, sh);
  else chunk_walk_kernel<2><<<walks, 256, 0, stream>>>(operands, state, q_start, slots, raw, sh);
  int lanes = 4;
  while (4 * lanes < sh.vdim) lanes *= 2;
  const int per = 256 / lanes;
  chunk_finish_kernel<<<dim3(chunks, (kTokens * sh.heads + per - 1) / per), 256, 0, stream>>>(raw, g, gain, q_start, (bf16_t*)out, sh, gain_heads,
                                                                                            lanes, eps);
  return launch_status();
}

}  // namespace

// Operands, state and output as in tk_gla_scan / tk_wkv_scan (recurrent.hip), bfloat16 storage; dim and vdim multiples of
// 16 up to 128.  least: requests of fewer tokens are left alone; chunks: at least the chunks of 16 tokens that the others
// have together; operands (float32 [chunks, heads, 33 dim + 16 vdim + 256]) and raw (float32 [N, heads * vdim]) are
// scratch on 16-byte borders.
TK_API int tk_gla_chunks(const void* q, int q_f32, int q_parts, long q_stride, const void* k, int k_f32, int k_parts,
                         long k_stride, const void* v, int v_f32, int v_parts, long v_stride, const void* g, int g_f32,
                         int g_parts, long g_stride, const void* z, int z_f32, int z_parts, long z_stride, const float* bias,
                         const float* gain, float* state, const int* q_start, const int* state_slots, void* out,
                         float* operands, float* raw, int N, int R, int least, int chunks, int heads, int dim, int vdim, float q_scale,
                         float inv_tau, float eps, hipStream_t stream) {
  return launch(false, In{q, q_f32, q_parts, q_stride}, In{k, k_f32, k_parts, k_stride}, In{v, v_f32, v_parts, v_stride},
                In{g, g_f32, g_parts, g_stride}, In{z, z_f32, z_parts, z_stride}, bias, nullptr, gain, 1, state, q_start, state_slots,
                out, operands, raw, N, chunks, Shape{R, heads, dim, vdim, least}, q_scale, inv_tau, eps, stream);
}

TK_API int tk_wkv_chunks(const void* r, int r_f32, int r_parts, long r_stride, const void* k, int k_f32, int k_parts,
                         long k_stride, const void* v, int v_f32, int v_parts, long v_stride, const void* g, int g_f32,
                         int g_parts, long g_stride, const void* d, int d_f32, int d_parts, long d_stride, const float* w0,
                         const float* u, const float* gain, float* state, const int* q_start, const int* state_slots, void* out,
                         float* operands, float* raw, int N, int R, int least, int chunks, int heads, int dim, float eps, hipStream_t stream) {
  return launch(true, In{r, r_f32, r_parts, r_stride}, In{k, k_f32, k_parts, k_stride}, In{v, v_f32, v_parts, v_stride},
                In{g, g_f32, g_parts, g_stride}, In{d, d_f32, d_parts, d_stride}, w0, u, gain, heads, state, q_start, state_slots, out,
                operands, raw, N, chunks, Shape{R, heads, dim, dim, least}, 1.f, 1.f, eps, stream);
}

TK_SLOTS(tk_gla_chunks)
TK_SLOTS(tk_wkv_chunks)
