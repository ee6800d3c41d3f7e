// Paged causal attention for any head size (multiple of 16, up to 512), any
// number of heads and groups, any page size that is a multiple of 8, in float32
// or bf16 storage with float32 arithmetic throughout.  It serves prompt portions
// and decode tokens alike: every query token walks its own request's block table
// from the first visible position to its own position.
//
// A block of kWaves waves takes up to QT queries that walk the same keys and values and
// share every one they load: consecutive tokens of one request at one query head (a piece
// of a 16-token tile of a prompt portion), or the query heads of one kv head's group at one
// token (a token that runs alone, a decode token).  Keys are taken 64 at a time, one key per lane;
// the round that starts at key 64 i goes to wave i % kWaves, which keeps a running maximum,
// a running sum and an output of its own in float32 for every query (online softmax); at
// the end the waves' results are merged in wave order.  Which wave takes which keys, and
// the order of every sum, follow from the query's own position alone: the result does not
// depend on how the request was cut into steps, on what else is in the batch, or on
// whether the token ran alone or in a tile (equal bits).
//
// Keys and values may differ in size (hd and vd).  What a query sees besides causality is given
// by `span`: 0 everything before it, W > 0 the last W positions, -C < 0 the positions of its own
// chunk of C (chunks counted from position 0 of the sequence).  With a window, `keep` > 0 leaves the
// first `keep` positions of the sequence visible as well, whatever the distance (they keep their places:
// a round of 64 keys still goes to the wave its index names).
//
// Cache pages: K [nkv][hd/8][ps][8], V [nkv][vd/16][ps/4][16][4] (see elementwise.hip).
#include "common.h"
#include "lds_copy.h"
#include "slots.h"

using namespace tk;

constexpr int kMaxHd = 512;
constexpr int kWaves = 8;  // waves of a block; kWaves * 64 threads cover every dimension of the widest head
static_assert(kWaves * kWave >= kMaxHd, "the merge gives every dimension a thread");
constexpr int kTileTokens = 16;  // tokens of a tile in the work list
constexpr int kQueries = 8;      // queries a block of the tile kernel takes

// four consecutive elements (four keys of one dimension in a V page) as one load
__device__ __forceinline__ void load_four(const float* p, float (&v)[4]) {
  const float4 x = *reinterpret_cast<const float4*>(p);
  v[0] = x.x; v[1] = x.y; v[2] = x.z; v[3] = x.w;
}
__device__ __forceinline__ void load_four(const bf16_t* p, float (&v)[4]) {
  const uint2 x = *reinterpret_cast<const uint2*>(p);
  v[0] = __uint_as_float(x.x << 16); v[1] = __uint_as_float(x.x & 0xffff0000u);
  v[2] = __uint_as_float(x.y << 16); v[3] = __uint_as_float(x.y & 0xffff0000u);
}

// eight consecutive elements (a key's piece of a K page)
__device__ __forceinline__ void load_eight(const float* p, float (&v)[8]) {
  const float4 a = *reinterpret_cast<const float4*>(p), b = *reinterpret_cast<const float4*>(p + 4);
  v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}
__device__ __forceinline__ void load_eight(const bf16_t* p, float (&v)[8]) {
  const uint4 x = *reinterpret_cast<const uint4*>(p);
  const uint32_t w[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    v[2 * i] = __uint_as_float(w[i] << 16);
    v[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
  }
}

// The same as they lie in memory, for a query alone: a round's loads are held until they are used.
typedef float f32x4 __attribute__((ext_vector_type(4)));     // (arrays of HIP's own vectors end up in scratch)
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
template <typename T> struct Held;
template <> struct Held<float> {
  struct Eight { f32x4 a, b; };
  typedef f32x4 Four;
  static __device__ __forceinline__ Eight eight(const float* p) { return {*reinterpret_cast<const f32x4*>(p), *reinterpret_cast<const f32x4*>(p + 4)}; }
  static __device__ __forceinline__ Four four(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
  static __device__ __forceinline__ float at(const Eight& x, int e) { return e < 4 ? x.a[e] : x.b[e - 4]; }
  static __device__ __forceinline__ float at(const Four& x, int e) { return x[e]; }
};
template <> struct Held<bf16_t> {
  typedef u32x4 Eight;
  typedef u32x2 Four;
  static __device__ __forceinline__ Eight eight(const bf16_t* p) { return *reinterpret_cast<const u32x4*>(p); }
  static __device__ __forceinline__ Four four(const bf16_t* p) { return *reinterpret_cast<const u32x2*>(p); }
  static __device__ __forceinline__ float half(uint32_t w, int e) { return __uint_as_float(e & 1 ? w & 0xffff0000u : w << 16); }
  static __device__ __forceinline__ float at(const Eight& x, int e) { return half(x[e / 2], e); }
  static __device__ __forceinline__ float at(const Four& x, int e) { return half(x[e / 2], e); }
};

// pieces of a key (8 dimensions each) asked for together where heads share it: few where eight queries do and the
// multiply-adds fill the time (and the registers)
template <int QT> constexpr int key_pieces() { return QT <= 4 ? 4 : 2; }
constexpr int kValuePieces = 4;      // of four values, that a lane asks for together there

// What all lanes hold alike, as a scalar (conditions on it are then scalar work, not the vector unit's masks).
__device__ __forceinline__ int scalar(int v) { return __builtin_amdgcn_readfirstlane(v); }

struct GenericItems {
  const int* single;      // token rows that run alone (null: every token of the step does)
  const int* tile_first;  // first token row of each tile
  const int* tile_count;  // tokens in it (1..kTileTokens), consecutive positions of one request
};

// QT: queries of a block; HEADS: they are heads of one group at one token (blockIdx.y is the kv
// head, blockIdx.z the piece of the group), else tokens of one tile at one head (blockIdx.y).
// SLOTS: value dimensions a lane owns (vd <= 64 * SLOTS).
// MANY, of queries alone: more blocks than CUs, of which one then holds two (half of the registers a wave).
template <typename T, int QT, bool HEADS, int SLOTS, bool MANY = false>
__global__ __launch_bounds__(kWaves * kWave) __attribute__((amdgpu_waves_per_eu(MANY ? 4 : 2))) void paged_attention_generic_kernel(
    const T* __restrict__ q, const T* __restrict__ k_cache, const T* __restrict__ v_cache,
    const int* __restrict__ block_tables, const int* __restrict__ positions,
    const int* __restrict__ req_of_token, GenericItems items, T* __restrict__ out, int nh, int nkv,
    int hd, int vd, int ps, int max_pages, float scale, int span, int keep, const float* __restrict__ sinks, float cap) {
  __shared__ __attribute__((aligned(16))) float q_s[QT][kMaxHd];
  __shared__ __attribute__((aligned(16))) float p_s[kWaves][kWave][QT];
  __shared__ long base_s[kWaves][kWave];  // where a key's values lie (a quad's, for heads that share a block), or -1
  __shared__ float m_s[kWaves], l_s[kWaves];
  __shared__ float acc_s[kWaves][kMaxHd];

  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1), wave = scalar(tid / kWave);
  const int group = nh / nkv;
  int n0, cnt, head0, kvh;
  if (HEADS) {
    n0 = items.single ? scalar(items.single[blockIdx.x]) : (int)blockIdx.x;
    kvh = blockIdx.y;
    head0 = kvh * group + blockIdx.z * QT;
    cnt = min(QT, group - (int)blockIdx.z * QT);
  } else {
    n0 = scalar(items.tile_first[blockIdx.x]) + blockIdx.z * QT;
    cnt = min(QT, scalar(items.tile_count[blockIdx.x]) - (int)blockIdx.z * QT);
    head0 = blockIdx.y;
    kvh = head0 / group;
  }
  if (cnt <= 0) return;
  const int* table = block_tables + (size_t)scalar(req_of_token[n0]) * max_pages;
  // query t: its row of q and out, its position and the first key it sees
  size_t row[QT];
  int pos[QT], first[QT];
#pragma unroll
  for (int t = 0; t < QT; ++t) {
    const int u = min(t, cnt - 1);
    row[t] = HEADS ? (size_t)n0 * nh + head0 + u : (size_t)(n0 + u) * nh + head0;
    pos[t] = scalar(positions[HEADS ? n0 : n0 + u]);
    first[t] = span > 0 ? (pos[t] - span + 1 > 0 ? pos[t] - span + 1 : 0) : span < 0 ? pos[t] - pos[t] % (-span) : 0;
  }
  const int lo = first[0], hi = pos[QT - 1];  // positions ascend within a tile
  const size_t page_elems = (size_t)nkv * hd * ps, v_page_elems = (size_t)nkv * vd * ps;
  const size_t head_off = (size_t)kvh * hd * ps, v_head_off = (size_t)kvh * vd * ps;

#pragma unroll
  for (int t = 0; t < QT; ++t) {
    const T* qrow = q + row[t] * hd;
    for (int d = tid; d < hd; d += kWaves * kWave) q_s[t][d] = Elem<T>::load(qrow + d) * scale;
  }
  __syncthreads();

  float m[QT], l[QT], acc[SLOTS][QT];
#pragma unroll
  for (int t = 0; t < QT; ++t) {
    m[t] = -INFINITY;
    l[t] = 0.f;
#pragma unroll
    for (int i = 0; i < SLOTS; ++i) acc[i][t] = 0.f;
  }

  // this wave's rounds: those whose index is wave modulo kWaves, from the one that holds lo
  // (with kept first positions the walk starts at round 0 and passes over the rounds between them and lo)
  const int round0 = keep > 0 ? 0 : lo / kWave;
  for (int rd = round0 + (wave - round0 % kWaves + kWaves) % kWaves; rd * kWave <= hi; rd += kWaves) {
    const int c0 = rd * kWave, c = c0 + lane;
    if (c0 >= keep && c0 + kWave - 1 < lo) continue;     // (the same for every lane of the wave)
    const bool loaded = (c >= lo || c < keep) && c <= hi;
    float dot[QT];
#pragma unroll
    for (int t = 0; t < QT; ++t) dot[t] = 0.f;
    // A query alone is a chain of trips to memory: a round's keys (of float32 half of them) and the values of its first dimensions are asked
    // for together, the values of the next ones behind the keys' products, and only then comes the softmax (four requests of up to 600 keys, heads of 128, float32
    // 20.9 -> 14.1 us, bfloat16 20.2 -> 13.4; of 2,048 keys 51 -> 34, 48 -> 31).
    constexpr bool ALONE = HEADS && QT == 1;
    constexpr int BUFFERS = MANY ? 1 : 2;
    typename Held<T>::Four held_v[ALONE ? BUFFERS : 1][kWave / 4];
    unsigned long quad = 0, seen = 0;      // where the values of this lane's key and its three neighbours lie; the round's keys that are seen
    const auto ask_values = [&](int slot, int buffer) {
      const int d = min(lane + slot * kWave, vd - 1);      // (a dimension past the head's is another one's, and not used)
      const uint32_t v_dim_off = (uint32_t)(d >> 4) * (ps >> 2) * 64 + (d & 15) * 4;
#pragma unroll
      for (int u = 0; u < kWave / 4; ++u) {      // (the same for all lanes: scalars)
        const uint32_t low = __builtin_amdgcn_readlane((uint32_t)quad, 4 * u), high = __builtin_amdgcn_readlane((uint32_t)(quad >> 32), 4 * u);
        held_v[buffer][u] = Held<T>::four(v_cache + (((unsigned long)high << 32) | low) + v_dim_off);
      }
    };
    if constexpr (ALONE) {
      constexpr int kHeldPieces = 32 / sizeof(T) / (MANY ? 2 : 1);      // of a key, eight dimensions each: 64 registers (MANY 32)
      // (a lane whose key and its three neighbours nobody sees, whose page may be another's, takes the last key and does not use it)
      const int there = c <= hi && ((c | 3) >= lo || c < keep) ? c : hi, page = table[there / ps];
      const T* const kp = k_cache + (size_t)page * page_elems + head_off + (size_t)(there % ps) * 8;
      seen = __ballot(loaded);
      quad = (size_t)page * v_page_elems + v_head_off + (size_t)((there % ps) >> 2) * 64;
      const int pieces = hd / 8;
      for (int j0 = 0; j0 < pieces; j0 += kHeldPieces) {
        typename Held<T>::Eight held_k[kHeldPieces];
#pragma unroll
        for (int u = 0; u < kHeldPieces; ++u) held_k[u] = Held<T>::eight(kp + (size_t)min(j0 + u, pieces - 1) * ps * 8);
        if (!MANY && j0 == 0) ask_values(0, 0);
#pragma unroll
        for (int u = 0; u < kHeldPieces; ++u)
          if (j0 + u < pieces) {
#pragma unroll
            for (int e = 0; e < 8; ++e) dot[0] = fmaf(q_s[0][(j0 + u) * 8 + e], Held<T>::at(held_k[u], e), dot[0]);
          }
      }
      __builtin_amdgcn_sched_barrier(0);      // (the registers of the keys)
      if (MANY) ask_values(0, 0);
      else if (SLOTS > 1 && kWave < vd) ask_values(1, 1);
    }
    // Heads that share a block at a token (decode of many) are bound by round trips to memory, too: they
    // ask for several pieces of a key at once and for the values of four keys in one piece (four
    // such pieces at once).  Tiles of a prompt portion, eight queries to a key, are bound by
    // their multiply-adds and keep the plain loops.  The order of every sum is the same.
    constexpr bool BATCHED = HEADS;
    long vbase = -1;
    if (BATCHED && !ALONE && (lane & 3) == 0 && c <= hi && (c + 3 >= lo || c < keep)) {
      // the values of four consecutive keys of a dimension are one piece of a page
      const int page = table[c / ps];
      vbase = (long)((size_t)page * v_page_elems + v_head_off + (size_t)((c % ps) >> 2) * 64);
    }
    if (!ALONE && loaded) {
      const int page = table[c / ps];
      const int off = c % ps;
      const T* kp = k_cache + (size_t)page * page_elems + head_off;
      if constexpr (BATCHED) {
        constexpr int kKeyPieces = key_pieces<QT>();
        for (int j0 = 0; j0 < hd / 8; j0 += kKeyPieces) {
          float k8[kKeyPieces][8];
#pragma unroll
          for (int u = 0; u < kKeyPieces; ++u) {
            const int j = min(j0 + u, hd / 8 - 1);      // (a piece past the head is loaded again and not used)
            load_eight(kp + ((size_t)j * ps + off) * 8, k8[u]);
          }
#pragma unroll
          for (int u = 0; u < kKeyPieces; ++u) {
            if (j0 + u < hd / 8) {
#pragma unroll
              for (int t = 0; t < QT; ++t) {
#pragma unroll
                for (int e = 0; e < 8; ++e) dot[t] = fmaf(q_s[t][(j0 + u) * 8 + e], k8[u][e], dot[t]);
              }
            }
          }
        }
      } else {
        for (int j = 0; j < hd / 8; ++j) {
          float k8[8];
          load_eight(kp + ((size_t)j * ps + off) * 8, k8);
#pragma unroll
          for (int t = 0; t < QT; ++t) {
#pragma unroll
            for (int e = 0; e < 8; ++e) dot[t] = fmaf(q_s[t][j * 8 + e], k8[e], dot[t]);
          }
        }
        vbase = (long)((size_t)page * v_page_elems + v_head_off + (size_t)(off >> 2) * 64 + (off & 3));
      }
    }
    float alpha[QT], p[QT];
#pragma unroll
    for (int t = 0; t < QT; ++t) {
      // a round that holds none of query t's keys leaves its sums as they are
      const bool takes = c0 <= pos[t] && (c0 + kWave - 1 >= first[t] || c0 < keep);
      alpha[t] = 1.f;
      p[t] = 0.f;
      if (takes) {
        const bool valid = (c >= first[t] || c < keep) && c <= pos[t];
        const float sc = valid ? (cap > 0.f ? cap * tanhf(dot[t] / cap) : dot[t]) : -INFINITY;
        const float m_new = fmaxf(m[t], wave_max(sc));
        p[t] = valid ? expf(sc - m_new) : 0.f;
        alpha[t] = expf(m[t] - m_new);  // m = -inf on the first round: alpha = 0
        l[t] = l[t] * alpha[t] + wave_sum(p[t]);
        m[t] = m_new;
      }
    }
    wave_lds_sync();   // the wave has read the probabilities of the 64 keys before
#pragma unroll
    for (int t = 0; t < QT; ++t) p_s[wave][lane][t] = p[t];
    if (!BATCHED) base_s[wave][lane] = vbase;
    else if (!ALONE && (lane & 3) == 0) base_s[wave][lane >> 2] = vbase;
    wave_lds_sync();
    const int count = (hi - c0 + 1 < kWave) ? hi - c0 + 1 : kWave;
#pragma unroll
    for (int i = 0; i < SLOTS; ++i) {
      const int d = lane + i * kWave;
      if (d < vd) {
        const size_t v_dim_off = (size_t)(d >> 4) * (ps >> 2) * 64 + (d & 15) * 4;
        float a[QT];
#pragma unroll
        for (int t = 0; t < QT; ++t) a[t] = acc[i][t] * alpha[t];
        if constexpr (ALONE) {
          // (bit k of `seen`: key k of the round is one that somebody sees; it is asked for in scalars)
          const auto add = [&](auto ALL) {
#pragma unroll
            for (int u = 0; u < kWave / 4; ++u) {
              const f32x4 p4 = *reinterpret_cast<const f32x4*>(&p_s[wave][4 * u][0]);
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                const float v = Held<T>::at(held_v[i % BUFFERS][u], e);
                a[0] = fmaf(p4[e], decltype(ALL)::value || (seen >> (4 * u + e) & 1) ? v : 0.f, a[0]);
              }
            }
          };
          if (seen == ~0ul) add(std::true_type{});
          else add(std::false_type{});
        } else if constexpr (BATCHED) {
          // four keys a load (16 bytes of float32) and four such loads asked for together, added
          // key by key in ascending order: the same sums as one key at a time.  A key out of
          // range adds a probability times 0.
          constexpr int kPieces = kValuePieces;
          for (int quad0 = 0; quad0 * 4 < count; quad0 += kPieces) {
            float v4[kPieces][4];
            bool there[kPieces];
#pragma unroll
            for (int u = 0; u < kPieces; ++u) {
              const long b = base_s[wave][quad0 + u];
              there[u] = (quad0 + u) * 4 < count && b >= 0;
              load_four(v_cache + (there[u] ? b : 0) + v_dim_off, v4[u]);   // (absent: the cache's first page, not used)
            }
#pragma unroll
            for (int u = 0; u < kPieces; ++u) {
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                const int key = (quad0 + u) * 4 + e;
                const bool in = there[u] && (c0 + key >= lo || c0 + key < keep) && c0 + key <= hi;
                const float v = in ? v4[u][e] : 0.f;   // (the probabilities of such a key are finite: 0 * p adds nothing)
#pragma unroll
                for (int t = 0; t < QT; ++t) a[t] = fmaf(p_s[wave][key][t], v, a[t]);
              }
            }
          }
        } else {
          for (int key = 0; key < count; ++key) {
            const long b = base_s[wave][key];
            if (b >= 0) {
              const float v = Elem<T>::load(v_cache + b + v_dim_off);
#pragma unroll
              for (int t = 0; t < QT; ++t) a[t] = fmaf(p_s[wave][key][t], v, a[t]);
            }
          }
        }
#pragma unroll
        for (int t = 0; t < QT; ++t) acc[i][t] = a[t];
      }
      if (ALONE && i + BUFFERS < SLOTS && (i + BUFFERS) * kWave < vd) ask_values(i + BUFFERS, i % BUFFERS);
    }
  }
  // merge, one query after the other: a wave that had no round of the query's brings
  // m = -inf, l = 0 and zeros, which weigh nothing
#pragma unroll
  for (int t = 0; t < QT; ++t) {
    if (t >= cnt) break;
    __syncthreads();   // the last query's merge has read the waves' results
    if (lane == 0) {
      m_s[wave] = m[t];
      l_s[wave] = l[t];
    }
#pragma unroll
    for (int i = 0; i < SLOTS; ++i) {
      const int d = lane + i * kWave;
      if (d < vd) acc_s[wave][d] = acc[i][t];
    }
    __syncthreads();
    if (tid < vd) {
      float top = m_s[0];
#pragma unroll
      for (int w = 1; w < kWaves; ++w) top = fmaxf(top, m_s[w]);
      // a sink is one more term exp(sink) of the head's denominator: no key, no value, not scaled
      const float sink = sinks ? sinks[HEADS ? head0 + t : head0] : -INFINITY;
      top = fmaxf(top, sink);
      float sum = 0.f, o = 0.f;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        const float e = expf(m_s[w] - top);
        sum = fmaf(l_s[w], e, sum);
        o = fmaf(acc_s[w][tid], e, o);
      }
      if (sinks) sum += expf(sink - top);
      Elem<T>::store(out + row[t] * vd + tid, o / sum);
    }
  }
}

// Tiles of a float32 prompt portion on the matrix cores (heads of 64 or 128, pages of whole 16s of keys): the sums of the kernel above in the
// same order, bit for bit, by
// v_mfma_f32_16x16x4_f32, which gives the bits of fmaf over its four k in ascending order.  A wave multiplies its round's 64 keys by
// the tile's 16 tokens at H heads of a group (scores: rows keys, columns tokens; output: rows dimensions), so a number loaded from a
// page meets H times 16 queries, where the kernel above has eight multiply-adds for it.  The matrix unit waits for every vector
// instruction of the wave, so operands come as they are multiplied, at scalar addresses and a lane's fixed place.  16 query heads over 8 kv
// heads of 128, us: 1,053 tokens of four requests 236 -> 88, one prompt of 1,024 316 -> 108, of 2,048 865 -> 296, 1,024 behind 1,024
// 652 -> 198 (with keys as 4-byte loads of operands 236 -> 126, 874 -> 548).  What is left: the waves of a block have unlike numbers
// of rounds, and a block has its CU to itself.
template <int HD, int H>
__global__ __launch_bounds__(kWaves * kWave) void attention_float32_tiles_kernel(
    const float* __restrict__ q, const float* __restrict__ k_cache, const float* __restrict__ v_cache, const int* __restrict__ block_tables,
    const int* __restrict__ positions, const int* __restrict__ req_of_token, GenericItems items, float* __restrict__ out, int nh, int nkv,
    int ps, int max_pages, float scale, int span, int keep, const float* __restrict__ sinks, float cap) {
  constexpr int STEPS = HD / 4, DIMS = HD / 16, KEYS = kWave / 16;      // products of a score, 16s of dimensions and of a round's keys
  constexpr int OWN = kWave * 32, SUMS = kWaves * kTileTokens * (HD + 4);
  static_assert(H * kTileTokens <= 32, "the probabilities take no more room than the keys");
  __shared__ __attribute__((aligned(16))) float shared_s[kWaves * OWN > SUMS ? kWaves * OWN : SUMS];
  __shared__ float q_s[H * STEPS * kWave], m_s[kWaves][kTileTokens], l_s[kWaves][kTileTokens];
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave), a = lane & 15, g = lane >> 4;
  const int tile = (int)gridDim.x - 1 - (int)blockIdx.x;      // (the list is shortest walk first)
  const int n0 = scalar(items.tile_first[tile]), cnt = min(kTileTokens, scalar(items.tile_count[tile]));
  if (cnt <= 0) return;
  const int head0 = blockIdx.y * H, kvh = head0 / (nh / nkv);
  const int* const table = block_tables + (size_t)scalar(req_of_token[n0]) * max_pages;
  // this lane's token: its position and the first key it sees (tokens of a tile are consecutive)
  const int pos0 = scalar(positions[n0]), pos = pos0 + min(a, cnt - 1), hi = pos0 + cnt - 1;
  const auto first_of = [&](int at) { return span > 0 ? (at - span + 1 > 0 ? at - span + 1 : 0) : span < 0 ? at - at % (-span) : 0; };
  const int first = first_of(pos), lo = first_of(pos0);
  const size_t page_elems = (size_t)nkv * HD * ps;
  const float* const k_head = k_cache + (size_t)kvh * HD * ps;
  const float* const v_head = v_cache + (size_t)kvh * HD * ps;

  // the queries as an operand, [head][step of four dimensions s][lane]: column a, dimension 4 s + g
  for (int at = tid; at < H * STEPS * kWave; at += kWaves * kWave) {
    const int column = at & 15, d = at / kWave % STEPS * 4 + (at >> 4 & 3), h = at / (kWave * STEPS);
    q_s[at] = q[((size_t)(n0 + min(column, cnt - 1)) * nh + head0 + h) * HD + d] * scale;
  }
  __syncthreads();
  float m[H], l[H];
  float4v acc[H][DIMS];      // [.][i][e]: dimension 16 i + 4 g + e of column a
#pragma unroll
  for (int h = 0; h < H; ++h) {
    m[h] = -INFINITY;
    l[h] = 0.f;
#pragma unroll
    for (int i = 0; i < DIMS; ++i) acc[h][i] = float4v{0.f, 0.f, 0.f, 0.f};
  }
  // a wave's own: 32 dimensions of a round's keys, then the round's probabilities
  float* const mine = shared_s + wave * OWN;
  const uint32_t key_place = (uint32_t)(lane >> 5) * ps * 8 + (lane & 31) * 4;

  const int round0 = keep > 0 ? 0 : lo / kWave;
  for (int rd = round0 + (wave - round0 % kWaves + kWaves) % kWaves; rd * kWave <= hi; rd += kWaves) {
    const int c0 = rd * kWave;
    if (c0 >= keep && c0 + kWave - 1 < lo) continue;
    int page[KEYS], off[KEYS];      // of each 16 keys (of 16 that nobody sees, whose page may be another's: the last key's)
#pragma unroll
    for (int t = 0; t < KEYS; ++t) {
      const int at = c0 + 16 * t, c = at <= hi && (at + 15 >= lo || at < keep) ? at : hi & ~15;
      page[t] = scalar(table[c / ps]);
      off[t] = c % ps;
    }
    // Operands, asked for while the ones before are multiplied: 32 dimensions of the round's keys, 16 bytes a lane (what an
    // operand takes, 16 of 32 bytes of every key, the vector memory path serves at a quarter of its rate) and through the wave's own LDS, then
    // 16 keys of all dimensions of the values, 256 bytes a load.
    constexpr int GROUPS = HD / 32;
    static_assert(GROUPS % 2 == 0 && DIMS <= 8, "values take the first of two sets of registers; 16 keys of a head are a set");
    float4v held[2][8];
    const auto ask_keys = [&](int group) {
#pragma unroll
      for (int t = 0; t < KEYS; ++t) {
        const float* const base = k_head + (size_t)page[t] * page_elems + (size_t)off[t] * 8;
#pragma unroll
        for (int j = 0; j < 2; ++j) held[group & 1][2 * t + j] = *reinterpret_cast<const float4v*>(base + (size_t)(4 * group + 2 * j) * ps * 8 + key_place);
      }
    };
    const auto ask_values = [&](int t) {
      const float* const base = v_head + (size_t)page[t] * page_elems + (size_t)(off[t] >> 2) * 64;
#pragma unroll
      for (int i = 0; i < DIMS; ++i)
#pragma unroll
        for (int s = 0; s < 4; ++s) held[t & 1][i][s] = base[(size_t)i * (ps >> 2) * 64 + s * 64 + (uint32_t)(a * 4 + g)];
    };
    float4v sc[H][KEYS];      // [.][t][e]: key 16 t + 4 g + e
#pragma unroll
    for (int h = 0; h < H; ++h)
#pragma unroll
      for (int t = 0; t < KEYS; ++t) sc[h][t] = float4v{0.f, 0.f, 0.f, 0.f};
    ask_keys(0);
#pragma unroll
    for (int group = 0; group < GROUPS; ++group) {
      wave_lds_sync();      // (the group before has been read, and the round before's probabilities)
#pragma unroll
      for (int i = 0; i < 8; ++i) *reinterpret_cast<float4v*>(mine + i * 256 + lane * 4) = held[group & 1][i];
      if (group + 1 < GROUPS) ask_keys(group + 1);
      else ask_values(0);
      wave_lds_sync();
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        float kr[KEYS];      // key 16 t + a, dimension 32 group + 4 s + g
#pragma unroll
        for (int t = 0; t < KEYS; ++t) kr[t] = mine[t * 512 + (s / 2) * 128 + a * 8 + 4 * (s & 1) + g];
#pragma unroll
        for (int h = 0; h < H; ++h) {
          const float qr = q_s[(h * STEPS + 8 * group + s) * kWave + lane];
#pragma unroll
          for (int t = 0; t < KEYS; ++t) sc[h][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(kr[t], qr, sc[h][t], 0, 0, 0);
        }
      }
    }
    // a round that holds none of the token's keys leaves its sums as they are
    const bool takes = c0 <= pos && (c0 + kWave - 1 >= first || c0 < keep);
    const auto sees = [&](int c) { return takes && (c >= first || c < keep) && c <= pos; };
    float alpha[H];
#pragma unroll
    for (int h = 0; h < H; ++h) {
      float top = -INFINITY;
#pragma unroll
      for (int t = 0; t < KEYS; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int c = c0 + 16 * t + 4 * g + e;
          if (cap > 0.f) sc[h][t][e] = cap * tanhf(sc[h][t][e] / cap);
          top = fmaxf(top, sees(c) ? sc[h][t][e] : -INFINITY);
        }
      const float m_new = fmaxf(m[h], max32(max16(top)));
      float part[KEYS];      // the sum over the wave's keys, pairs of neighbours first, as lanes of a wave are added
#pragma unroll
      for (int t = 0; t < KEYS; ++t) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float weight = expf(sc[h][t][e] - m_new);
          sc[h][t][e] = sees(c0 + 16 * t + 4 * g + e) ? weight : 0.f;
        }
        part[t] = sum32(sum16((sc[h][t][0] + sc[h][t][1]) + (sc[h][t][2] + sc[h][t][3])));
      }
      static_assert(KEYS == 4, "four 16s of keys a round");
      alpha[h] = 1.f;
      if (takes) {
        alpha[h] = expf(m[h] - m_new);
        l[h] = l[h] * alpha[h] + ((part[0] + part[1]) + (part[2] + part[3]));
        m[h] = m_new;
      }
    }
    wave_lds_sync();      // the keys have been read
#pragma unroll
    for (int h = 0; h < H; ++h)
#pragma unroll
      for (int t = 0; t < KEYS; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) mine[(h * kWave + 16 * t + 4 * g + e) * kTileTokens + a] = sc[h][t][e];
    wave_lds_sync();
    // Where not every token sees every key of the round: a key that is another's or none counts as zeros, and so do numbers of the
    // others that are not finite, which would make NaN of a weight of zero; those are added for the tokens that see them.
    const bool every = c0 + kWave - 1 <= pos0 && (c0 >= first_of(hi) || c0 + kWave <= keep);
    bool apart = false;
#pragma unroll
    for (int h = 0; h < H; ++h)
#pragma unroll
      for (int i = 0; i < DIMS; ++i) acc[h][i] *= alpha[h];
#pragma unroll
    for (int t = 0; t < KEYS; ++t) {
      float pr[H][4];      // column a, key 16 t + 4 s + g
#pragma unroll
      for (int h = 0; h < H; ++h)
#pragma unroll
        for (int s = 0; s < 4; ++s) pr[h][s] = mine[(h * kWave + 16 * t + 4 * s) * kTileTokens + lane];
      if (t + 1 < KEYS) ask_values(t + 1);
      __builtin_amdgcn_sched_barrier(0);
      if (!every) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const int c = c0 + 16 * t + 4 * s + g;
          const bool in = (c >= lo || c < keep) && c <= hi;
#pragma unroll
          for (int i = 0; i < DIMS; ++i) {
            const bool number = fabsf(held[t & 1][i][s]) < INFINITY;
            apart |= in && !number;
            held[t & 1][i][s] = in && number ? held[t & 1][i][s] : 0.f;
          }
        }
      }
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int i = 0; i < DIMS; ++i)
#pragma unroll
          for (int h = 0; h < H; ++h) acc[h][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(held[t & 1][i][s], pr[h][s], acc[h][i], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (__ballot(apart) != 0) {
#pragma unroll 1
      for (int key = 0; key < kWave; ++key) {
        const int c = c0 + key;
        if (c > hi || !(c >= lo || c < keep)) continue;
        const float* const base = v_head + (size_t)scalar(table[c / ps]) * page_elems + (size_t)(c % ps >> 2) * 64 + (c & 3);
#pragma unroll
        for (int i = 0; i < DIMS; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float v = base[(size_t)i * (ps >> 2) * 64 + (4 * g + e) * 4];
            if (!sees(c) || fabsf(v) < INFINITY) continue;
#pragma unroll
            for (int h = 0; h < H; ++h) acc[h][i][e] = fmaf(mine[(h * kWave + key) * kTileTokens + a], v, acc[h][i][e]);
          }
      }
    }
  }
  // merge in wave order, a head after the other
#pragma unroll
  for (int h = 0; h < H; ++h) {
    __syncthreads();
    if (g == 0) {
      m_s[wave][a] = m[h];
      l_s[wave][a] = l[h];
    }
#pragma unroll
    for (int i = 0; i < DIMS; ++i)
      *reinterpret_cast<float4v*>(&shared_s[(wave * kTileTokens + a) * (HD + 4) + 16 * i + 4 * g]) = acc[h][i];
    __syncthreads();
    // every wave's weight and the whole sum once a token, then the dimensions
    if (tid < kTileTokens) {
      const float sink = sinks ? sinks[head0 + h] : -INFINITY;
      float top = m_s[0][tid];
#pragma unroll
      for (int w = 1; w < kWaves; ++w) top = fmaxf(top, m_s[w][tid]);
      top = fmaxf(top, sink);
      float sum = 0.f;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        const float e = expf(m_s[w][tid] - top);
        sum = fmaf(l_s[w][tid], e, sum);
        m_s[w][tid] = e;
      }
      l_s[0][tid] = sinks ? sum + expf(sink - top) : sum;
    }
    __syncthreads();
    for (int at = tid; at < cnt * HD; at += kWaves * kWave) {
      const int t = at / HD, d = at % HD;
      float o = 0.f;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) o = fmaf(shared_s[(w * kTileTokens + t) * (HD + 4) + d], m_s[w][t], o);
      out[((size_t)(n0 + t) * nh + head0 + h) * HD + d] = o / l_s[0][t];
    }
  }
}

// Heads of a block of that kernel.  Two read a key's operands once for both, but their blocks are half as many and take twice the products:
// heads of 128 where one a block would be more blocks than CUs.  us with one and two, 16 heads over 8 kv heads: 17 tokens 16 | 24, 300 39 |
// 33, 64 behind 2,000 87 | 114, 1,024 150 | 114.  Heads of 64, whose blocks of one head have two to a CU, one: 17 tokens 12 | 17, 300 18 | 22, 1,024
// 78 | 73.  Beside the form on the vector unit, 972 portions of 2 to 2,048 tokens, 2 to 64 heads: 1.05 to 3.5 times as fast (0.82 with two a block throughout).
static int tile_heads(int num_tiles, int nh, int nkv, int hd) { return hd == 128 && nh / nkv % 2 == 0 && (long)num_tiles * nh > 256 ? 2 : 1; }

// Whether a portion's tiles took that kernel.
template <typename T>
static bool launch_float32_tiles(const T*, const T*, const T*, const int*, const int*, const int*, GenericItems, int, T*, int, int, int, int, int,
                                 int, float, int, int, const float*, float, hipStream_t) {
  return false;
}
template <>
bool launch_float32_tiles<float>(const float* q, const float* k_cache, const float* v_cache, const int* block_tables, const int* positions,
                                 const int* req_of_token, GenericItems items, int num_tiles, float* out, int nh, int nkv, int hd, int vd,
                                 int ps, int max_pages, float scale, int span, int keep, const float* sinks, float cap, hipStream_t stream) {
  if (hd != vd || (hd != 64 && hd != 128) || ps % 16 != 0) return false;
#define TK_TILES(HD_, H_)                                                                                                   \
  attention_float32_tiles_kernel<HD_, H_><<<dim3(num_tiles, nh / H_), kWaves * kWave, 0, stream>>>(                          \
      q, k_cache, v_cache, block_tables, positions, req_of_token, items, out, nh, nkv, ps, max_pages, scale, span, keep, sinks, cap)
  if (hd == 64) TK_TILES(64, 1);
  else if (tile_heads(num_tiles, nh, nkv, hd) == 2) TK_TILES(128, 2);
  else TK_TILES(128, 1);
#undef TK_TILES
  return true;
}

// Heads of a group that share a block at most.
static int heads_a_block(int group) { return group <= 4 ? 4 : kQueries; }

// Whether the heads of a group share a block for tokens that run alone (the result is the same either way): where each in a block of its
// own would be more blocks than two a CU and some (float32, whose keys are twice the bytes: than two), and the shared ones, which take two to
// four times as long, are enough of them.  us alone and shared over 600 keys, heads of 128: bfloat16, 16 heads over 8 kv heads, 32 tokens 26 |
// 38, 44 43 | 44, 52 50 | 44, 32 over 8, 16 tokens 22 | 38, 24 39 | 38, 32 52 | 39, 64 over 8, 12 tokens (96 shared blocks) 35 | 56, 18 54 | 57, 24 66 | 58;
// float32, 16 over 8, 24 32 | 39, 32 45 | 41, 48 72 | 51, 64 over 8, 8 23 | 56, 16 48 | 58, 18 65 | 57, 24 103 | 57.  2,432 launches of each type (groups
// of 2 to 16, heads of 64 to 256, 1 to 96 tokens over 100 to 6,000 keys): 1 % and 2 % behind the faster form on average, 0.56 and 0.49 at worst.
static bool heads_share(bool float32, long tokens, int nh, int nkv) {
  const int group = nh / nkv, qt = heads_a_block(group);
  return group > 1 && tokens * nh > (float32 ? 511 : 576) && tokens * nkv * ((group + qt - 1) / qt) >= (float32 ? 160 : 192);
}

template <typename T, int SLOTS>
static void launch_generic(const T* q, const T* k_cache, const T* v_cache, const int* block_tables,
                           const int* positions, const int* req_of_token, GenericItems items,
                           int num_single, int num_tiles, T* out, int nh, int nkv, int hd, int vd, int ps,
                           int max_pages, float scale, int span, int keep, int share_heads, const float* sinks,
                           float cap, hipStream_t stream) {
  const int group = nh / nkv;
#define TK_ALONE(QT_, MANY_)                                                                        \
  paged_attention_generic_kernel<T, QT_, true, SLOTS, MANY_>                                        \
      <<<dim3(num_single, nkv, (group + QT_ - 1) / QT_), kWaves * kWave, 0, stream>>>(              \
          q, k_cache, v_cache, block_tables, positions, req_of_token, items, out, nh, nkv, hd, vd,  \
          ps, max_pages, scale, span, keep, sinks, cap)
  if (num_single > 0) {
    const int qt = heads_a_block(group);
    const bool shared = share_heads < 0 ? heads_share(sizeof(T) == 4, num_single, nh, nkv) : group > 1 && share_heads > 0;
    if (!shared && (long)num_single * nh > 256) TK_ALONE(1, true);
    else if (!shared) TK_ALONE(1, false);
    else if (qt == 4) TK_ALONE(4, false);
    else TK_ALONE(kQueries, false);
  }
#undef TK_ALONE
  if (num_tiles > 0 && !launch_float32_tiles<T>(q, k_cache, v_cache, block_tables, positions, req_of_token, items, num_tiles, out, nh, nkv,
                                                hd, vd, ps, max_pages, scale, span, keep, sinks, cap, stream))
    paged_attention_generic_kernel<T, kQueries, false, SLOTS>
        <<<dim3(num_tiles, nh, kTileTokens / kQueries), kWaves * kWave, 0, stream>>>(
            q, k_cache, v_cache, block_tables, positions, req_of_token, items, out, nh, nkv, hd, vd, ps,
            max_pages, scale, span, keep, sinks, cap);
}

// tile_first / tile_count (num_tiles of them) and single (num_single token rows): the step's work
// lists, which together name every token once.  With tile_first null every one of the N tokens
// runs alone.  share_heads: whether the query heads of a group share a block for the tokens
// that run alone (1), or not (0), or as fills the GPU (-1); the result is the same.  sinks: null, or
// float32 [nh]: head a's softmax has exp(sinks[a]) as one more term of its denominator.  cap > 0: every score
// becomes cap tanh(score / cap) first (not the sink's).
TK_API int tk_paged_attention_generic(int dtype, const void* q, const void* k_cache,
                                      const void* v_cache, const int* block_tables,
                                      const int* positions, const int* req_of_token, void* out,
                                      int N, int nh, int nkv, int hd, int vd, int ps, int max_pages,
                                      float scale, int span, int keep, const int* tile_first,
                                      const int* tile_count, int num_tiles, const int* single,
                                      int num_single, int share_heads, const float* sinks, float cap, hipStream_t stream) {
  if (N <= 0) return 0;
  if (keep < 0 || (keep > 0 && span <= 0) || !(cap >= 0.f)) return -1;
  if (hd > kMaxHd || hd % 8 != 0 || vd > kMaxHd || vd % 16 != 0 || nkv <= 0 || nh % nkv != 0 || ps <= 0 || ps % 4 != 0 || nh > 65535) return -1;
  if (tile_first == nullptr) {
    num_tiles = 0;
    single = nullptr;
    num_single = N;
  } else if (num_tiles < 0 || num_single < 0 || tile_count == nullptr || (num_single > 0 && single == nullptr)) {
    return -1;
  }
  const GenericItems items{single, tile_first, tile_count};
#define TK_GENERIC(T_, SLOTS_)                                                                      \
  launch_generic<T_, SLOTS_>((const T_*)q, (const T_*)k_cache, (const T_*)v_cache, block_tables,    \
                             positions, req_of_token, items, num_single, num_tiles, (T_*)out, nh,   \
                             nkv, hd, vd, ps, max_pages, scale, span, keep, share_heads, sinks, cap, stream)
  if (dtype == 0) {
    if (vd <= 128) TK_GENERIC(float, 2);
    else if (vd <= 256) TK_GENERIC(float, 4);
    else TK_GENERIC(float, 8);
  } else {
    if (vd <= 128) TK_GENERIC(bf16_t, 2);
    else if (vd <= 256) TK_GENERIC(bf16_t, 4);
    else TK_GENERIC(bf16_t, 8);
  }
#undef TK_GENERIC
  return launch_status();
}

// Whether the heads of a group share a block (1 or 0) for so many tokens that run alone.
TK_API int tk_attention_heads_share(int float32, int tokens, int nh, int nkv) { return heads_share(float32 != 0, tokens, nh, nkv); }

// Heads of a block for so many tiles of a float32 portion.
TK_API int tk_attention_tile_heads(int num_tiles, int nh, int nkv, int hd) { return tile_heads(num_tiles, nh, nkv, hd); }

// the same entry points in slot form (slots.h), for launch lists
TK_SLOTS(tk_paged_attention_generic)
