// Attention over a sliding window plus pooled blocks behind it, with mixing of the heads'
// softmax weights, on the matrix cores (gfx950; bfloat16 storage).  What is computed stands in
// attention_pooled.hip.
//
// What bounds the other form there: every raw score goes to memory, comes back to be normalised and mixed,
// goes out and comes back again, eight rows share what a block loads, and the values are applied by the
// vector unit (2,048 rows over 1,024 keys and up to 130 blocks, 32 / 8 heads of 128: 0.65 ms of
// scores, 0.5 of mixing, 1.2 of values; the three kernels here together 0.40).  The mixing needs every head's
// NORMALISED weight of an entry, so a single walk with a running maximum cannot do it; but scores are cheap
// on the matrix cores, so they are formed twice instead of being kept:
//   stats:    per (16 rows of one request, four heads, share of the entries) the maximum and the sum of exponentials;
//   weights:  per (16 rows, run of entries) the scores of ALL heads again, their normalised weights, and the
//             mixed ones, sum_g talk[h, g] w_g, as a matrix product over the heads;
//   values:   per (16 rows, four heads, share of the entries) the product of mixed weights and values.
// Weights, the mixing matrix and the block means are float32 and stay so: as operands each is split into three
// bfloat16, a piece of what the pieces before it leave (24 bits of mantissa; of two splits the products below 2^-24 of
// the largest are dropped).  Sums are float32, and so are the mixed weights in memory.  (Two pieces, 16 bits, and a
// mixed weight as such a pair hid behind the bfloat16 output, but not where heads are mixed with opposite signs.)
//
// Entries: a row sees tokens (tiles of 16 that begin at a multiple of 16, so that a tile lies in one page:
// pages of a multiple of 16) and block means (tiles of 16, padded to chunks of 32); a chunk is
// either all tokens or all means.  Tiles never cross a request, so blocks find theirs by counting the requests' tiles.
#include "common.h"
#include "request_tiles.h"
#include "slots.h"

using namespace tk;

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

union Frag {
  u32x4_t u;
  bf16x8_t v;
};

constexpr int kRows = 16;      // rows of a tile
constexpr int kChunk = 32;     // entries of a chunk
constexpr int kMaxShares = 16; // shares of a tile's entries
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLowest = -1e30f;   // a maximum of nothing (finite: differences of two stay numbers)

struct Args {
  const bf16_t* q;
  const bf16_t* k_cache;
  const bf16_t* v_cache;
  const float* k_pool;
  const float* v_pool;
  bf16_t* out;
  const int* positions;
  const int* q_start;
  const int* tables;
  const float* talk;
  float* weights;      // mixed: a tile's [Cmax][H][its rows][32 entries] at its first row's place
  float* part_m;       // [tiles][H][16][S], in powers of two
  float* part_l;
  float* part_o;       // [S][N][H * vdim]
  int table_width, N, R, H, G, size, pool, page_size, KE, VE, S, Cmax;
  float scale2;        // the scores' scale times log2(e)
};

struct Tile {
  int row, tq, i0, NB, j0, ja, i_last, PC, chunks;   // (ja: j0 rounded down to a tile's start; PC: chunks of block means)
  const int* table;
};

__device__ __forceinline__ bool find_tile(const Args& a, int at, Tile& t) {
  RequestTile rt;
  if (!find_request_tile(a.q_start, a.R, kRows, at, rt)) return false;
  t.row = a.q_start[rt.req] + rt.index * kRows;
  t.tq = min(kRows, a.q_start[rt.req + 1] - t.row);
  t.i0 = __builtin_amdgcn_readfirstlane(a.positions[t.row]);
  t.i_last = t.i0 + t.tq - 1;
  const int behind = t.i_last - a.size - (a.pool - 1);
  t.NB = behind >= 0 ? behind / a.pool + 1 : 0;
  t.j0 = max(0, t.i0 - a.size + 1);
  t.ja = t.j0 & ~15;
  t.PC = (t.NB + kChunk - 1) / kChunk;
  t.chunks = t.PC + (t.i_last - t.ja + kChunk) / kChunk;
  t.table = a.tables + (size_t)rt.req * a.table_width;
  return true;
}

// a float's leading bfloat16 pieces: two numbers at a time, each piece packed
__device__ __forceinline__ void split3(float x, float y, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
  hi = pack_bf16x2(x, y);
  const float x1 = x - __uint_as_float(hi << 16), y1 = y - __uint_as_float(hi & 0xffff0000u);
  mid = pack_bf16x2(x1, y1);
  lo = pack_bf16x2(x1 - __uint_as_float(mid << 16), y1 - __uint_as_float(mid & 0xffff0000u));
}
__device__ __forceinline__ void split_eight(const float (&f)[8], Frag& hi, Frag& mid, Frag& lo) {
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    uint32_t h0, m0, l0;
    split3(f[2 * x], f[2 * x + 1], h0, m0, l0);
    hi.u[x] = h0;
    mid.u[x] = m0;
    lo.u[x] = l0;
  }
}
// (low halves, high halves) of two words
__device__ __forceinline__ uint32_t low_halves(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x05040100u); }
__device__ __forceinline__ uint32_t high_halves(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); }

__device__ __forceinline__ f32x4_t mfma16(const Frag& a, const Frag& b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v, b.v, c, 0, 0, 0);
}

__device__ __forceinline__ f32x16_t mfma32(const Frag& a, const Frag& b, f32x16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.v, b.v, c, 0, 0, 0);
}

// The queries of four heads as the second operand: lane (row = lane & 15, k group = lane >> 4).
template <int KS>
__device__ __forceinline__ void load_queries(const Args& a, const Tile& t, int quad, Frag (&qf)[4][KS]) {
  const int lane = threadIdx.x & (kWave - 1);
  const int row = t.row + min(lane & 15, t.tq - 1);
#pragma unroll
  for (int h = 0; h < 4; ++h)
#pragma unroll
    for (int s = 0; s < KS; ++s)
      qf[h][s].u = *reinterpret_cast<const u32x4_t*>(a.q + ((size_t)row * a.H + quad * 4 + h) * (32 * KS) + 32 * s + 8 * (lane >> 4));
}

// Scores (times scale2) of 16 entries (tile `et`) for the quad's four heads: sc[h][i] belongs to entry
// 4 (lane >> 4) + i of the tile and row lane & 15; entries the row does not see are -inf.
template <int KS, int KVQ>
__device__ __forceinline__ void tile_scores(const Args& a, const Tile& t, int et, int quad, const Frag (&qf)[4][KS], f32x4_t (&sc)[4]) {
  const int lane = threadIdx.x & (kWave - 1), g = lane >> 4, my_i = t.i0 + (lane & 15);
  constexpr int dim = 32 * KS, per = 4 / KVQ;      // per: heads of the quad a kv head has
  const int kv0 = quad * 4 / (a.H / a.G);
  const int KW = a.G * dim;
#pragma unroll
  for (int h = 0; h < 4; ++h) sc[h] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  if (et < 2 * t.PC) {
    const int b = min(et * 16 + (lane & 15), t.NB - 1);
    const unsigned per_page = (unsigned)a.page_size * a.KE;
#pragma unroll
    for (int kv = 0; kv < KVQ; ++kv) {
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const unsigned flat = (unsigned)b * KW + (kv0 + kv) * dim + 32 * s + 8 * g;     // (eight numbers lie in one page)
        const float* p = a.k_pool + (size_t)t.table[flat / per_page] * per_page + flat % per_page;
        const float4 x = *reinterpret_cast<const float4*>(p), y = *reinterpret_cast<const float4*>(p + 4);
        Frag hi, mid, lo;
        uint32_t h0, m0, l0;
        split3(x.x, x.y, h0, m0, l0); hi.u[0] = h0; mid.u[0] = m0; lo.u[0] = l0;
        split3(x.z, x.w, h0, m0, l0); hi.u[1] = h0; mid.u[1] = m0; lo.u[1] = l0;
        split3(y.x, y.y, h0, m0, l0); hi.u[2] = h0; mid.u[2] = m0; lo.u[2] = l0;
        split3(y.z, y.w, h0, m0, l0); hi.u[3] = h0; mid.u[3] = m0; lo.u[3] = l0;
#pragma unroll
        for (int h = 0; h < per; ++h) {
          f32x4_t& c = sc[kv * per + h];
          c = mfma16(lo, qf[kv * per + h][s], c);
          c = mfma16(mid, qf[kv * per + h][s], c);
          c = mfma16(hi, qf[kv * per + h][s], c);
        }
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int e = et * 16 + 4 * g + i;
      const bool seen = e < t.NB && e * a.pool + a.pool - 1 <= my_i - a.size;
#pragma unroll
      for (int h = 0; h < 4; ++h) sc[h][i] = seen ? sc[h][i] * a.scale2 : -INFINITY;
    }
  } else {
    const int p0 = t.ja + (et - 2 * t.PC) * 16;
    if (p0 <= t.i_last) {
      const size_t slot = (size_t)t.table[p0 / a.page_size] * a.page_size + p0 % a.page_size + (lane & 15);
#pragma unroll
      for (int kv = 0; kv < KVQ; ++kv) {
        const bf16_t* rowp = a.k_cache + slot * KW + (size_t)(kv0 + kv) * dim + 8 * g;
        Frag kf[KS];
#pragma unroll
        for (int s = 0; s < KS; ++s) kf[s].u = *reinterpret_cast<const u32x4_t*>(rowp + 32 * s);
#pragma unroll
        for (int s = 0; s < KS; ++s)
#pragma unroll
          for (int h = 0; h < per; ++h) sc[kv * per + h] = mfma16(kf[s], qf[kv * per + h][s], sc[kv * per + h]);
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int j = p0 + 4 * g + i;
      const bool seen = j <= my_i && my_i - j < a.size;      // (a row past the tile's last sees what it likes: it is not kept)
#pragma unroll
      for (int h = 0; h < 4; ++h) sc[h][i] = seen ? sc[h][i] * a.scale2 : -INFINITY;
    }
  }
}

// Four waves take a share's tiles of 16 entries in turn.  A key tile is read once for four heads and sixteen rows.
// The vector unit most (60 % of the time busy: an exponential, a mask and a maximum a score; the matrix units 16 %): 82 us
// at 2,048 rows of 32 / 8 heads of 128.
template <int KS, int KVQ>
__global__ __launch_bounds__(256) void portion_stats_kernel(Args a) {
  __shared__ float red[4][4][kRows][2];
  Tile t;
  if (!find_tile(a, blockIdx.x, t)) return;
  const int quad = blockIdx.y, split = blockIdx.z;
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  Frag qf[4][KS];
  load_queries<KS>(a, t, quad, qf);
  float m[4], l[4];
#pragma unroll
  for (int h = 0; h < 4; ++h) {
    m[h] = kLowest;
    l[h] = 0.f;
  }
  const int tiles = 2 * t.chunks, lo = (int)((long)tiles * split / a.S), hi = (int)((long)tiles * (split + 1) / a.S);
  for (int et = lo + wave; et < hi; et += 4) {
    f32x4_t sc[4];
    tile_scores<KS, KVQ>(a, t, et, quad, qf, sc);
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      const float top = fmaxf(fmaxf(fmaxf(sc[h][0], sc[h][1]), fmaxf(sc[h][2], sc[h][3])), m[h]);
      float sum = l[h] * __builtin_amdgcn_exp2f(m[h] - top);
#pragma unroll
      for (int i = 0; i < 4; ++i) sum += __builtin_amdgcn_exp2f(sc[h][i] - top);
      l[h] = sum;
      m[h] = top;
    }
  }
#pragma unroll
  for (int h = 0; h < 4; ++h) {
#pragma unroll
    for (int x = 16; x < kWave; x <<= 1) {
      const float om = __shfl_xor(m[h], x, kWave), ol = __shfl_xor(l[h], x, kWave), top = fmaxf(m[h], om);
      l[h] = l[h] * __builtin_amdgcn_exp2f(m[h] - top) + ol * __builtin_amdgcn_exp2f(om - top);
      m[h] = top;
    }
    if (lane < kRows) {
      red[wave][h][lane][0] = m[h];
      red[wave][h][lane][1] = l[h];
    }
  }
  __syncthreads();
  if (threadIdx.x < 4 * kRows) {
    const int h = threadIdx.x / kRows, row = threadIdx.x % kRows;
    float top = kLowest, sum = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) top = fmaxf(top, red[w][h][row][0]);
#pragma unroll
    for (int w = 0; w < 4; ++w) sum += red[w][h][row][1] * __builtin_amdgcn_exp2f(red[w][h][row][0] - top);
    const size_t at = (((size_t)blockIdx.x * a.H + quad * 4 + h) * kRows + row) * a.S + split;
    a.part_m[at] = top;
    a.part_l[at] = sum;
  }
}

// H / 4 waves, a wave four heads.  A chunk: every wave's normalised weights of 16 rows by 32 entries, float32, into LDS
// [row][entry][head] (two copies, one barrier a chunk), then a wave mixes whole rows: D = talk (32 heads by H) times
// the row's weights (H by 32 entries), whose pieces are split as they are read.  154 us for 2,048 rows of 32 heads of
// 128 over 1,024 tokens and up to 130 blocks (147 with two pieces a weight): vector units 44 % busy (an exponential and a
// split of every weight), matrix units 17 %, a quarter of the waves' time waits, 300 MB of weights written.
template <int KS, int KVQ, int H>
__global__ __launch_bounds__(16 * H) void portion_weights_kernel(Args a) {
  constexpr int kWaves = H / 4, kMix = H / 16;
  constexpr int kPitch = kChunk * H + 4;     // (a row's start moved by four banks: the 16 rows' writes spread)
  // pieces of 16 bytes (four heads) swizzled by the entry: the reads walk entries 4 H bytes apart, and sixteen of them
  // meet all banks
  constexpr int kPieces = H / 4, kSwizzle = H == 32 ? 1 : 2;
  __shared__ __align__(16) float lds[2][kRows * kPitch];
  Tile t;
  if (!find_tile(a, blockIdx.x, t)) return;
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave, quad = wave;
  const int lo = (int)((long)t.chunks * blockIdx.y / gridDim.y), hi = (int)((long)t.chunks * (blockIdx.y + 1) / gridDim.y);
  if (lo >= hi) return;
  Frag qf[4][KS];
  load_queries<KS>(a, t, quad, qf);
  float m[4], il[4];
#pragma unroll
  for (int h = 0; h < 4; ++h) {
    const size_t at = (((size_t)blockIdx.x * H + quad * 4 + h) * kRows + (lane & 15)) * a.S;
    // the four lanes of a row take a quarter of the shares each, all loads in flight (one after the other a
    // step of single tokens, 16 shares, took 55 us; 20)
    float pm[kMaxShares / 4], pl[kMaxShares / 4], top = kLowest, sum = 0.f;
#pragma unroll
    for (int x = 0; x < kMaxShares / 4; ++x) {
      const int s = min(4 * x + (lane >> 4), a.S - 1);
      pm[x] = a.part_m[at + s];
      pl[x] = a.part_l[at + s];
    }
#pragma unroll
    for (int x = 0; x < kMaxShares / 4; ++x) top = fmaxf(top, pm[x]);
    top = max16(top);
    top = max32(top);
#pragma unroll
    for (int x = 0; x < kMaxShares / 4; ++x)
      if (4 * x + (lane >> 4) < a.S) sum += pl[x] * __builtin_amdgcn_exp2f(pm[x] - top);
    sum = sum16(sum);
    sum = sum32(sum);
    m[h] = top;
    il[h] = 1.f / sum;
  }
  // the mixing matrix as the first operand: lane (head = lane & 31, heads 16 s + 8 (lane >> 5) .. + 8)
  Frag th[kMix], tm[kMix], tl[kMix];
#pragma unroll
  for (int s = 0; s < kMix; ++s) {
    const int to = lane & 31, from = 16 * s + 8 * (lane >> 5);
    float f[8];
#pragma unroll
    for (int x = 0; x < 8; ++x) f[x] = to < H ? a.talk[to * H + from + x] : 0.f;
    split_eight(f, th[s], tm[s], tl[s]);
  }
  for (int c = lo; c < hi; ++c) {
    float* const copy = lds[c & 1];
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      f32x4_t sc[4];
      tile_scores<KS, KVQ>(a, t, 2 * c + half, quad, qf, sc);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float w[4];
#pragma unroll
        for (int h = 0; h < 4; ++h) w[h] = __builtin_amdgcn_exp2f(sc[h][i] - m[h]) * il[h];
        const int entry = 16 * half + 4 * (lane >> 4) + i, piece = (quad ^ (entry >> kSwizzle)) & (kPieces - 1);
        *reinterpret_cast<float4*>(copy + (lane & 15) * kPitch + entry * H + piece * 4) = make_float4(w[0], w[1], w[2], w[3]);
      }
    }
    __syncthreads();
    const int entry = lane & 31;
    for (int row = wave; row < t.tq; row += kWaves) {
      f32x16_t acc;
#pragma unroll
      for (int x = 0; x < 16; ++x) acc[x] = 0.f;
#pragma unroll
      for (int s = 0; s < kMix; ++s) {
        float f[8];
#pragma unroll
        for (int x = 0; x < 2; ++x) {
          const int piece = ((4 * s + 2 * (lane >> 5) + x) ^ (entry >> kSwizzle)) & (kPieces - 1);
          const float4 w = *reinterpret_cast<const float4*>(copy + row * kPitch + entry * H + piece * 4);
          f[4 * x] = w.x;
          f[4 * x + 1] = w.y;
          f[4 * x + 2] = w.z;
          f[4 * x + 3] = w.w;
        }
        Frag bh, bm, bl;
        split_eight(f, bh, bm, bl);
        acc = mfma32(tl[s], bh, acc);
        acc = mfma32(tm[s], bm, acc);
        acc = mfma32(th[s], bl, acc);
        acc = mfma32(tm[s], bh, acc);
        acc = mfma32(th[s], bm, acc);
        acc = mfma32(th[s], bh, acc);
      }
      float* out = a.weights + ((size_t)t.row * a.Cmax * H + (size_t)c * H * t.tq + row) * kChunk + entry;
#pragma unroll
      for (int x = 0; x < 16; ++x) {
        const int h = 8 * (x >> 2) + 4 * (lane >> 5) + (x & 3);
        if (H == 32 || x < 8) out[(size_t)h * t.tq * kChunk] = acc[x];
      }
    }
    // (one barrier a chunk: a wave writes this copy again only after the next chunk's barrier, which every wave
    // reaches behind its reads here)
  }
}

// Four waves take a share's chunks in turn: D = mixed weights (16 rows by 32 entries) times values (32 entries by
// channels), four heads.  A lane reads VT neighbouring channels of eight entries, which are the VT channel tiles' operands
// once their halves are paired (column n of tile c is channel VT n + c), so values need no LDS.  169 us at the same
// sizes (157 with two pieces a weight): one wave a SIMD, vector units 39 % and matrix units 18 % busy, 300 MB of weights
// read once and the values by every tile from L2; on the vector unit it was 1.2 ms.
template <int VT, int KVQ>
__global__ __launch_bounds__(256) void portion_values_kernel(Args a) {
  constexpr int vdim = 16 * VT, per = 4 / KVQ;
  __shared__ float red[2][4][kRows][vdim];
  Tile t;
  if (!find_tile(a, blockIdx.x, t)) return;
  const int quad = blockIdx.y, split = blockIdx.z;
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave, n = lane & 15, g = lane >> 4;
  const int kv0 = quad * 4 / (a.H / a.G), VW = a.G * vdim;
  f32x4_t acc[4][VT];
#pragma unroll
  for (int h = 0; h < 4; ++h)
#pragma unroll
    for (int c = 0; c < VT; ++c) acc[h][c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int lo = (int)((long)t.chunks * split / a.S), hi = (int)((long)t.chunks * (split + 1) / a.S);
  for (int c = lo + wave; c < hi; c += 4) {
    Frag wh[4], wm[4], wl[4];
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      const float* p = a.weights + ((size_t)t.row * a.Cmax * a.H + ((size_t)c * a.H + quad * 4 + h) * t.tq + min(n, t.tq - 1)) * kChunk + 8 * g;
      const float4 x = *reinterpret_cast<const float4*>(p), y = *reinterpret_cast<const float4*>(p + 4);
      const float f[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
      split_eight(f, wh[h], wm[h], wl[h]);
    }
    if (c < t.PC) {
      const int b0 = c * kChunk + 8 * g;
      const unsigned per_page = (unsigned)a.page_size * a.VE;
#pragma unroll
      for (int kv = 0; kv < KVQ; ++kv) {
        const float* from[8];       // (VT numbers lie in one page)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const unsigned flat = (unsigned)max(0, min(b0 + e, t.NB - 1)) * VW + (kv0 + kv) * vdim + VT * n;
          from[e] = a.v_pool + (size_t)t.table[flat / per_page] * per_page + flat % per_page;
        }
#pragma unroll
        for (int cc = 0; cc < VT; cc += 2) {
          float2 f[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            f[e] = *reinterpret_cast<const float2*>(from[e] + cc);
            if (b0 + e >= t.NB) f[e] = make_float2(0.f, 0.f);
          }
#pragma unroll
          for (int y = 0; y < 2; ++y) {
            Frag vh, vm, vl;
#pragma unroll
            for (int x = 0; x < 4; ++x) {
              uint32_t h0, m0, l0;
              split3(y ? f[2 * x].y : f[2 * x].x, y ? f[2 * x + 1].y : f[2 * x + 1].x, h0, m0, l0);
              vh.u[x] = h0;
              vm.u[x] = m0;
              vl.u[x] = l0;
            }
#pragma unroll
            for (int h = 0; h < per; ++h) {
              f32x4_t& o = acc[kv * per + h][cc + y];
              o = mfma16(wh[kv * per + h], vl, o);
              o = mfma16(wm[kv * per + h], vm, o);
              o = mfma16(wl[kv * per + h], vh, o);
              o = mfma16(wh[kv * per + h], vm, o);
              o = mfma16(wm[kv * per + h], vh, o);
              o = mfma16(wh[kv * per + h], vh, o);
            }
          }
        }
      }
    } else {
      const int p0 = t.ja + (c - t.PC) * kChunk + 8 * g;     // (eight entries that begin at a multiple of 8: one page)
      const size_t slot = p0 <= t.i_last ? (size_t)t.table[p0 / a.page_size] * a.page_size + p0 % a.page_size : 0;
#pragma unroll
      for (int kv = 0; kv < KVQ; ++kv) {
        uint32_t v[8][VT / 2];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const bf16_t* p = a.v_cache + (slot + e) * VW + (size_t)(kv0 + kv) * vdim + VT * n;
          // what no row of the tile sees is taken as zero: its weight is, and zero times a number nobody wrote may not be
          const bool there = p0 + e >= t.j0 && p0 + e <= t.i_last;
          if (VT == 8) {
            const u32x4_t x = there ? *reinterpret_cast<const u32x4_t*>(p) : u32x4_t{0, 0, 0, 0};
#pragma unroll
            for (int d = 0; d < VT / 2; ++d) v[e][d] = x[d];
          } else {
            const uint2 x = there ? *reinterpret_cast<const uint2*>(p) : make_uint2(0, 0);
            v[e][0] = x.x;
            v[e][1] = x.y;
          }
        }
#pragma unroll
        for (int cc = 0; cc < VT; ++cc) {
          Frag vf;
#pragma unroll
          for (int x = 0; x < 4; ++x)
            vf.u[x] = cc & 1 ? high_halves(v[2 * x][cc / 2], v[2 * x + 1][cc / 2]) : low_halves(v[2 * x][cc / 2], v[2 * x + 1][cc / 2]);
#pragma unroll
          for (int h = 0; h < per; ++h) {
            f32x4_t& o = acc[kv * per + h][cc];
            o = mfma16(wl[kv * per + h], vf, o);
            o = mfma16(wm[kv * per + h], vf, o);
            o = mfma16(wh[kv * per + h], vf, o);
          }
        }
      }
    }
  }
  // the waves' sums: 2 + 3 onto 0 + 1, then 1 onto 0
#pragma unroll
  for (int step = 2; step >= 1; step >>= 1) {
    if (wave >= step && wave < 2 * step) {
#pragma unroll
      for (int h = 0; h < 4; ++h)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int c = 0; c < VT; ++c) red[wave - step][h][4 * g + i][VT * n + c] = acc[h][c][i];
    }
    __syncthreads();
    if (wave < step) {
#pragma unroll
      for (int h = 0; h < 4; ++h)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int c = 0; c < VT; ++c) acc[h][c][i] += red[wave][h][4 * g + i][VT * n + c];
    }
    __syncthreads();
  }
  if (wave != 0) return;
#pragma unroll
  for (int h = 0; h < 4; ++h) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = 4 * g + i;
      if (row >= t.tq) continue;
      const size_t at = ((size_t)(t.row + row) * a.H + quad * 4 + h) * vdim + VT * n;
      if (a.S == 1) {
        uint32_t w[VT / 2];
#pragma unroll
        for (int c = 0; c < VT / 2; ++c) w[c] = pack_bf16x2(acc[h][2 * c][i], acc[h][2 * c + 1][i]);
        if (VT == 8) *reinterpret_cast<uint4*>(a.out + at) = make_uint4(w[0], w[1], w[VT / 2 - 2], w[VT / 2 - 1]);
        else *reinterpret_cast<uint2*>(a.out + at) = make_uint2(w[0], w[1]);
      } else {
        float* p = a.part_o + (size_t)split * a.N * a.H * vdim + at;
#pragma unroll
        for (int c = 0; c < VT; c += 4)
          *reinterpret_cast<float4*>(p + c) = make_float4(acc[h][c][i], acc[h][c + 1][i], acc[h][c + 2][i], acc[h][c + 3][i]);
      }
    }
  }
}

// the shares' partial outputs added in their order, four channels a thread
__global__ __launch_bounds__(256) void portion_merge_kernel(const float* __restrict__ part_o, bf16_t* __restrict__ out, int S, size_t total) {
  const size_t at = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (at >= total) return;
  float4 sum = *reinterpret_cast<const float4*>(part_o + at);
#pragma unroll 4
  for (int s = 1; s < S; ++s) {
    const float4 x = *reinterpret_cast<const float4*>(part_o + (size_t)s * total + at);
    sum.x += x.x;
    sum.y += x.y;
    sum.z += x.z;
    sum.w += x.w;
  }
  *reinterpret_cast<uint2*>(out + at) = make_uint2(pack_bf16x2(sum.x, sum.y), pack_bf16x2(sum.z, sum.w));
}

template <int KS, int KVQ>
void launch_scores(const Args& a, int tiles, int runs, hipStream_t stream) {
  portion_stats_kernel<KS, KVQ><<<dim3(tiles, a.H / 4, a.S), 256, 0, stream>>>(a);
  if (a.H == 32) portion_weights_kernel<KS, KVQ, 32><<<dim3(tiles, runs), 512, 0, stream>>>(a);
  else portion_weights_kernel<KS, KVQ, 16><<<dim3(tiles, runs), 256, 0, stream>>>(a);
}

}  // namespace

// Sizes: H 16 or 32; H / G of 1, 2 or a multiple of 4; dim and vdim 64 or 128; pages of a multiple of 16
// tokens; every array on a 16-byte border.  tiles: at least the tiles of 16 rows all requests have together;
// Cmax: at least the chunks any of them sees; runs: pieces the weights kernel cuts a tile's chunks into.
TK_API int tk_pooled_window_portions(const void* q, const void* k_cache, const void* v_cache, const float* k_pool,
                                     const float* v_pool, int KE, int VE, void* out, const int* positions,
                                     const int* q_start, const int* tables, int table_width, const float* talk,
                                     float* weights, float* part_m, float* part_l, float* part_o, int N, int R, int H,
                                     int G, int dim, int vdim, int size, int pool, int page_size, int tiles, int S,
                                     int Cmax, int runs, float scale, hipStream_t stream) {
  if (N <= 0) return 0;
  if (R < 1 || (H != 16 && H != 32) || G < 1 || H % G || (dim != 64 && dim != 128) || (vdim != 64 && vdim != 128) ||
      size < 1 || pool < 1 || page_size < 16 || page_size % 16 || tiles < 1 || S < 1 || S > kMaxShares || Cmax < 1 || runs < 1 ||
      (long)KE * pool < (long)G * dim || (long)VE * pool < (long)G * vdim ||
      (long)table_width * page_size * max(KE, VE) > 0x7fffffffL)     // (places among a request's means in 32 bits)
    return -2;
  const int group = H / G, kvq = group >= 4 ? 1 : 4 / group;
  if (group > 2 && group % 4) return -2;
  Args a{(const bf16_t*)q, (const bf16_t*)k_cache, (const bf16_t*)v_cache, k_pool, v_pool, (bf16_t*)out, positions,
         q_start, tables, talk, weights, part_m, part_l, part_o, table_width, N, R, H, G, size, pool, page_size, KE, VE, S,
         Cmax, scale * kLog2e};
  if (dim == 128) {
    if (kvq == 1) launch_scores<4, 1>(a, tiles, runs, stream);
    else if (kvq == 2) launch_scores<4, 2>(a, tiles, runs, stream);
    else launch_scores<4, 4>(a, tiles, runs, stream);
  } else {
    if (kvq == 1) launch_scores<2, 1>(a, tiles, runs, stream);
    else if (kvq == 2) launch_scores<2, 2>(a, tiles, runs, stream);
    else launch_scores<2, 4>(a, tiles, runs, stream);
  }
  const dim3 grid(tiles, H / 4, S);
  if (vdim == 128) {
    if (kvq == 1) portion_values_kernel<8, 1><<<grid, 256, 0, stream>>>(a);
    else if (kvq == 2) portion_values_kernel<8, 2><<<grid, 256, 0, stream>>>(a);
    else portion_values_kernel<8, 4><<<grid, 256, 0, stream>>>(a);
  } else {
    if (kvq == 1) portion_values_kernel<4, 1><<<grid, 256, 0, stream>>>(a);
    else if (kvq == 2) portion_values_kernel<4, 2><<<grid, 256, 0, stream>>>(a);
    else portion_values_kernel<4, 4><<<grid, 256, 0, stream>>>(a);
  }
  if (S > 1) {
    const size_t total = (size_t)N * H * vdim;
    portion_merge_kernel<<<(unsigned)((total / 4 + 255) / 256), 256, 0, stream>>>(part_o, (bf16_t*)out, S, total);
  }
  return launch_status();
}

TK_SLOTS(tk_pooled_window_portions)
