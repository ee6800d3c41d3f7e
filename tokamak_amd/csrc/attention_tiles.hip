// Paged attention of prompt portions on the matrix cores for the shapes the tuned kernels of
// attention_mfma.hip do not take: keys and values of unlike sizes (up to 512 channels each, keys in
// pieces of 8, values in blocks of 16), any number of query heads a kv head, a window or chunks, a sink.
// bf16 in, float32 softmax and accumulation.  Tokens that run alone have a form of their own (third
// kernel below) where a kv head has many query heads.
//
// A wave owns one tile (up to 16 consecutive tokens of one request) at one query head.  With one query head a
// kv head, and with two or three of more than 128 or up to 64 channels, the four waves of a block take four heads of the same tile and every
// wave fetches its operands itself; else the waves of a block are heads of one kv head and
// share the operands through LDS (second kernel below).  Keys are walked 16 at a time, operands straight from the pages (no LDS):
//   S^T[key][token] = K[key][:] . Q[token][:]      v_mfma_f32_16x16x32_bf16, K rows as A (a lane
//       (key, kb) reads the 16-byte piece of dims 32 c + 8 kb of its key), Q rows as B, kept in registers
//   P^T = exp2(S^T * c - m[token])                  float32, a token's column per lane
//   O^T[dim][token] += V^T[dim][key] P^T[key][token] v_mfma_f32_16x16x16_bf16, V^T rows as A (a lane
//       (dim, kb) reads the 8 bytes of keys 4 kb .. 4 kb + 3 of its dim), P^T as B: the first product's
//       result layout is the second's B operand layout.
// What a token sees besides causality is given by `span`: 0 everything before it, W > 0 the last W
// positions, -C < 0 the positions of its own chunk of C; with a window, `keep` > 0 leaves the first
// `keep` positions of the sequence visible too (their stages of 16 keys are walked first, then the walk
// jumps to the window's first stage).  sinks: null, or float32 [nh]: exp(sinks[a])
// is one more term of head a's denominator.  CAP instances bound every score softly first (soft_cap.h).
//
// Cache pages: K [nkv][hd/8][ps][8], V [nkv][vd/16][ps/4][16][4]; ps a multiple of 16, so that 16
// consecutive keys from a multiple of 16 lie in one page.
#include "common.h"
#include "lds_copy.h"
#include "lds_limit.h"
#include "slots.h"
#include "soft_cap.h"

using namespace tk;

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short short4v __attribute__((ext_vector_type(4)));
typedef float float4v __attribute__((ext_vector_type(4)));

union Frag8 {
  uint4 u;
  bf16x8 v;
};
union Frag4 {
  uint2 u;
  short4v v;
};

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

constexpr int kHeadsPerBlock = 4;

// KCH: 32-wide chunks of the key size the instance holds (hd <= 32 KCH); DBL: 16-wide blocks of the
// value size (vd <= 16 DBL).  Chunks and blocks behind the true sizes are skipped (the same for every lane).
template <int KCH, int DBL, bool CAP>
__global__ __launch_bounds__(kHeadsPerBlock * 64) void attention_tiles_kernel(
    const bf16_t* __restrict__ q, const bf16_t* __restrict__ k_cache, const bf16_t* __restrict__ v_cache,
    const int* __restrict__ block_tables, int max_pages, const int* __restrict__ positions,
    const int* __restrict__ req_of_token, const int* __restrict__ tile_first, const int* __restrict__ tile_count,
    bf16_t* __restrict__ out, int nh, int nkv, int hd, int vd, int ps, float scale_log2, int span, int keep,
    const float* __restrict__ sinks, SoftCap cap) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, kb = lane >> 4;
  const int head = blockIdx.y * kHeadsPerBlock + wave;
  if (head >= nh) return;   // (the waves of a block never wait for one another)
  const int tile = blockIdx.x;
  const int n0 = tile_first[tile], cnt = tile_count[tile];
  const int kvh = head / (nh / nkv);
  const int pos0 = positions[n0];                 // the tile's tokens stand at pos0, pos0 + 1, ...
  const int my = min(col, cnt - 1);               // (columns behind the tile's last token repeat it and are not written)
  const int pos = pos0 + my;
  const int first = span > 0 ? max(pos - span + 1, 0) : span < 0 ? pos - pos % (-span) : 0;
  const int lo = span > 0 ? max(pos0 - span + 1, 0) : span < 0 ? pos0 - pos0 % (-span) : 0;   // the first token's first key
  const int hi = pos0 + cnt - 1;
  const int* table = block_tables + (size_t)req_of_token[n0] * max_pages;
  const size_t k_page = (size_t)nkv * hd * ps, v_page = (size_t)nkv * vd * ps;
  const size_t k_head = (size_t)kvh * hd * ps, v_head = (size_t)kvh * vd * ps;
  const int kch = (hd + 31) >> 5, dbl = vd >> 4;

  bf16x8 qreg[KCH];
  const bf16_t* qp = q + ((size_t)(n0 + my) * nh + head) * hd + kb * 8;
#pragma unroll
  for (int c = 0; c < KCH; ++c) {
    Frag8 f;
    f.u = (c * 32 + kb * 8 < hd) ? *reinterpret_cast<const uint4*>(qp + c * 32) : make_uint4(0, 0, 0, 0);
    qreg[c] = f.v;
  }
  float m_run = -INFINITY, l_run = 0.f;
  float4v acc[DBL];
#pragma unroll
  for (int d = 0; d < DBL; ++d) acc[d] = float4v{0.f, 0.f, 0.f, 0.f};

  const int c_first = lo & ~15;
  for (int c0 = keep > 0 ? 0 : c_first; c0 <= hi; c0 = (c0 + 16 >= keep && c0 + 16 < c_first) ? c_first : c0 + 16) {
    const int page = table[c0 / ps], off = c0 % ps;
    const bf16_t* kp = k_cache + (size_t)page * k_page + k_head + (size_t)(off + col) * 8;
    const bf16_t* vp = v_cache + (size_t)page * v_page + v_head + (size_t)((off >> 2) + kb) * 64 + col * 4;
    Frag8 kreg[KCH];
#pragma unroll
    for (int c = 0; c < KCH; ++c)
      kreg[c].u = (c * 32 + kb * 8 < hd) ? *reinterpret_cast<const uint4*>(kp + (size_t)(c * 4 + kb) * ps * 8)
                                         : make_uint4(0, 0, 0, 0);
    Frag4 vreg[DBL];
#pragma unroll
    for (int d = 0; d < DBL; ++d)
      vreg[d].u = d < dbl ? *reinterpret_cast<const uint2*>(vp + (size_t)d * (ps >> 2) * 64) : make_uint2(0, 0);
    float4v sc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < KCH; ++c)
      if (c < kch) sc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kreg[c].v, qreg[c], sc, 0, 0, 0);
    // this lane: keys c0 + 4 kb + e of token `col`
    float sv[4];
    bool seen[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int key = c0 + kb * 4 + e;
      seen[e] = (key >= first || key < keep) && key <= pos;
      sv[e] = seen[e] ? (CAP ? cap.log2_score(sc[e]) : sc[e] * scale_log2) : -INFINITY;     // (a key that no token wrote may hold anything: chosen, not computed)
    }
    float tmax = fmaxf(fmaxf(sv[0], sv[1]), fmaxf(sv[2], sv[3]));
    tmax = max16(tmax);
    tmax = max32(tmax);
    const float m_new = fmaxf(m_run, tmax);
    const float m_safe = m_new == -INFINITY ? 0.f : m_new;   // a token that has seen no key yet
    const float alpha = fast_exp2(m_run - m_safe);
    m_run = m_new;
    float pr[4], psum = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      pr[e] = seen[e] ? fast_exp2(sv[e] - m_safe) : 0.f;
      psum += pr[e];
    }
    l_run = l_run * alpha + psum;
    Frag4 pb;
    pb.u = make_uint2(pack_bf16x2(pr[0], pr[1]), pack_bf16x2(pr[2], pr[3]));
    const bool edge = c0 + 15 > hi;   // keys behind the tile's last token are not written yet
    const bool rescale = __builtin_amdgcn_ballot_w64(alpha != 1.f) != 0;
#pragma unroll
    for (int d = 0; d < DBL; ++d) {
      if (d >= dbl) continue;
      short4v tv = vreg[d].v;
      if (edge) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (c0 + kb * 4 + e > hi) tv[e] = 0;
      }
      float4v a = acc[d];
      if (rescale) a *= alpha;
      acc[d] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(tv, pb.v, a, 0, 0, 0);
    }
  }

  float l = l_run;
  l = sum16(l);
  l = sum32(l);
  if (sinks) l += fast_exp2(sinks[head] * 1.4426950408889634f - m_run);
  if (col >= cnt) return;
  const float inv = 1.f / l;
  // acc[d][e] = O^T[dim 16 d + 4 kb + e][token col]
  bf16_t* op = out + ((size_t)(n0 + col) * nh + head) * vd + kb * 4;
#pragma unroll
  for (int d = 0; d < DBL; ++d) {
    if (d >= dbl) continue;
    uint2 o;
    o.x = pack_bf16x2(acc[d][0] * inv, acc[d][1] * inv);
    o.y = pack_bf16x2(acc[d][2] * inv, acc[d][3] * inv);
    *reinterpret_cast<uint2*>(op + d * 16) = o;
  }
}

// The same products for kv heads with several query heads: a block of HB waves takes HB heads of
// ONE kv head at one tile and shares every 16 keys' operands through LDS (each wave of the kernel above
// fetches them from L2 for itself: with 32 heads on one kv head that is L2's rate, not the matrix
// cores').  A stage is the 16 keys' slice of the K page (hd/8 runs of 256 bytes) and of the V page
// (vd/16 runs of 512 bytes), copied as they lie, so the operand reads are those of the pages: a lane's
// 16-byte key piece at ((4 c + kb) 16 + key) 8, its 8-byte value piece at ((4 d + kb) 16 + dim) 4.
// A ring of four stages, copied from the pages to LDS without registers (lds_copy.h) three stages ahead of their
// products, the pages' numbers a stage before that; one barrier a stage.  A stage's products are shorter than a trip to memory:
// fetched through registers one stage ahead, with the page's number asked for on the way, a stage of 512 + 448 channels took 5 us.
// 2,048 tokens, 32 heads on one kv head of 512 / 448 channels, window 1,024: 690 -> 280 us (0.35 PFLOP/s); 32 / 8 heads of 128,
// window 1,024 + 4: 192 -> 118.  What bounds it now: a stage's chain (barrier, scores, softmax, output) at two waves a SIMD, some
// 4,500 clocks a stage of 960 channels of which LDS is busy 1,900 and the matrix cores 1,000.
// Also for two and three heads a kv head where a ring is 24 to 32 KB (16 / 8 heads of 128, 1,024 tokens 88 -> 71 us, 300 behind
// 2,000 96 -> 65; 1.26 times as fast over 26 portions of 2 to 1,024 tokens, of 96 and of 128 / 64 1.11 and 1.07, 0.95 at worst); of larger heads a
// block of two waves would have the CU's LDS to itself, of 64 / 64, whose stages are short, it is level (0.89 to 1.20, 16 / 8 heads, 1,024 tokens 67 | 75).
// Of operands two groups are held in registers, the one that is multiplied and the next (whole stages would be more than the 256
// registers that two waves a SIMD leave each).
constexpr int kStages = 4;
__host__ __device__ constexpr int stage_kb(int channels) { return (2 * channels + 63) / 64; }      // of 16 keys: whole runs of 64 pieces

template <int KCH, int DBL, int HB, bool CAP>
__global__ __launch_bounds__(HB * 64) void attention_tiles_shared_kernel(
    const bf16_t* __restrict__ q, const bf16_t* __restrict__ k_cache, const bf16_t* __restrict__ v_cache,
    const int* __restrict__ block_tables, int max_pages, const int* __restrict__ positions,
    const int* __restrict__ req_of_token, const int* __restrict__ tile_first, const int* __restrict__ tile_count,
    bf16_t* __restrict__ out, int nh, int nkv, int hd, int vd, int ps, float scale_log2, int span, int keep,
    const float* __restrict__ sinks, SoftCap cap) {
  extern __shared__ __attribute__((aligned(16))) bf16_t stage_s[];   // kStages stages of stage_bytes(hd, vd)
  constexpr int PER = (KCH + DBL / 2 + HB - 1) / HB;                  // KB of a stage that a wave copies
  // chunks and blocks of a group (two groups' reads are held in registers), and those that are walked or passed over together
  constexpr int KG = KCH > 4 ? 2 : 4, KPART = KCH > 4 ? KCH / 2 : KCH, VG = DBL > 8 ? 4 : 8, VPART = DBL > 8 ? DBL / 2 : DBL;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), col = lane & 15, kb = lane >> 4;
  const int group = nh / nkv, blocks_per_kv = (group + HB - 1) / HB;
  const int kvh = blockIdx.y / blocks_per_kv;
  const int in_group = (blockIdx.y % blocks_per_kv) * HB + wave;
  const bool computes = in_group < group;                   // (a wave without a head still copies and waits)
  const int head = kvh * group + (computes ? in_group : 0);
  const int tile = gridDim.x - 1 - blockIdx.x;              // (a portion's last tiles walk furthest: they start first)
  const int n0 = tile_first[tile], cnt = tile_count[tile];
  const int pos0 = positions[n0];
  const int my = min(col, cnt - 1);
  const int pos = pos0 + my;
  const int first = span > 0 ? max(pos - span + 1, 0) : span < 0 ? pos - pos % (-span) : 0;
  const int lo = span > 0 ? max(pos0 - span + 1, 0) : span < 0 ? pos0 - pos0 % (-span) : 0;
  const int hi = pos0 + cnt - 1;
  const int* table = block_tables + (size_t)req_of_token[n0] * max_pages;
  const size_t k_page = (size_t)nkv * hd * ps, v_page = (size_t)nkv * vd * ps;
  const size_t k_head = (size_t)kvh * hd * ps, v_head = (size_t)kvh * vd * ps;
  const int kch = (hd + 31) >> 5, dbl = vd >> 4;
  const int k_kb = stage_kb(hd), all_kb = k_kb + stage_kb(vd);

  bf16x8 qreg[KCH];
  const bf16_t* qp = q + ((size_t)(n0 + my) * nh + head) * hd + kb * 8;
#pragma unroll
  for (int c = 0; c < KCH; ++c) {
    Frag8 f;
    f.u = (c * 32 + kb * 8 < hd) ? *reinterpret_cast<const uint4*>(qp + c * 32) : make_uint4(0, 0, 0, 0);
    qreg[c] = f.v;
  }
  // (the queries are here before the first copy is asked for: a wait for them in the walk would be one for every copy)
#pragma unroll
  for (int c = 0; c < KCH; ++c) asm volatile("" : "+v"(qreg[c]));
  float m_run = -INFINITY, l_run = 0.f;
  float4v acc[DBL];
#pragma unroll
  for (int d = 0; d < DBL; ++d) acc[d] = float4v{0.f, 0.f, 0.f, 0.f};

  // What this wave copies of a stage: PER runs of 64 pieces of 16 bytes, of K (piece p: 8 dims p / 16, key p % 16) or of V (block
  // p / 32, 16 bytes p % 32 of its 512).  Runs behind the last are the last once more (every wave copies as much, so that its
  // count of copies says which stage has come), pieces behind the last of K or V its last.
  uint32_t from[PER], to[PER];
  bool of_k[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int run = min(wave + i * HB, all_kb - 1);
    of_k[i] = run < k_kb;
    const int piece = min((of_k[i] ? run : run - k_kb) * 64 + lane, 2 * (of_k[i] ? hd : vd) - 1);
    from[i] = of_k[i] ? (uint32_t)(((piece >> 4) * ps + (piece & 15)) * 16)
                      : (uint32_t)((piece >> 5) * (ps >> 2) * 128 + (piece & 31) * 16);
    to[i] = run * 1024;
  }
  const uint32_t lds = (uint32_t)(uintptr_t)(TK_LDS char*)stage_s, stage_size = all_kb * 1024;
  const int c_first = lo & ~15;
  const int c_start = keep > 0 ? 0 : c_first;
  const auto behind = [&](int c) { return (c + 16 >= keep && c + 16 < c_first) ? c_first : c + 16; };   // (past the kept first positions: on to the window)
  const auto copy = [&](int c, int page, int slot) {
    const int off = c % ps;
    const char* const kp = reinterpret_cast<const char*>(k_cache + (size_t)page * k_page + k_head + (size_t)off * 8);
    const char* const vp = reinterpret_cast<const char*>(v_cache + (size_t)page * v_page + v_head + (size_t)(off >> 2) * 64);
#pragma unroll
    for (int i = 0; i < PER; ++i) copy_to_lds<false>(lds + slot * stage_size + to[i], from[i], of_k[i] ? kp : vp);
  };
  int c_copy = c_start, slot_copy = 0, ahead = 0;      // the next stage to copy, its place, stages copied and not yet used
#pragma unroll
  for (int i = 0; i < kStages - 1; ++i) {
    if (c_copy <= hi) {
      copy(c_copy, table[c_copy / ps], slot_copy++);
      c_copy = behind(c_copy);
      ++ahead;
    }
  }
  int page_copy = c_copy <= hi ? table[c_copy / ps] : 0;
  int buf = 0;
  for (int c0 = c_start; c0 <= hi; c0 = behind(c0)) {
    // this wave's part of the stage has come when only those of the stages behind it are on their way; everyone's, behind the
    // barrier, where nobody reads the stage before any more either: its place is the next copy's
    static_assert(kStages == 4, "the counts below");
    if (ahead >= 3) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * PER) : "memory");
    else if (ahead == 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PER) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    --ahead;
    if (c_copy <= hi) {
      copy(c_copy, page_copy, slot_copy);
      slot_copy = (slot_copy + 1) % kStages;
      c_copy = behind(c_copy);
      ++ahead;
      if (c_copy <= hi) page_copy = table[c_copy / ps];
    }
    if (c0 + 15 > hi) {      // the last stage: values of positions that hold nothing yet are zeros, whatever their weight of zero meets
      bf16_t* const vz = stage_s + (size_t)buf * (stage_size / 2) + k_kb * 512;
      for (int p = threadIdx.x; p < vd * 4; p += HB * 64) {      // 8 bytes: keys 4 (p / 16 % 4) .. + 3 of a channel
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (c0 + (p >> 4 & 3) * 4 + e > hi) vz[(size_t)p * 4 + e] = 0;
      }
      __syncthreads();
    }
    if (computes) {
      const bf16_t* ks = stage_s + (size_t)buf * (stage_size / 2);
      const bf16_t* vs = ks + k_kb * 512;
      // Operands are asked for a group ahead of the group whose products run, with nothing that branches around a read: a read
      // behind a branch of its own is waited for there.
      float4v sc = {0.f, 0.f, 0.f, 0.f}, sc2 = {0.f, 0.f, 0.f, 0.f};
      const auto keys = [&](int c) { return *reinterpret_cast<const uint4*>(ks + (size_t)((c * 4 + kb) * 16 + col) * 8); };
#pragma unroll
      for (int part = 0; part < KCH; part += KPART) {
        if (part >= kch) continue;      // (the same for every lane)
        Frag8 kf[2][KG];
#pragma unroll
        for (int i = 0; i < KG; ++i) kf[0][i].u = keys(part + i);
#pragma unroll
        for (int c = part; c < part + KPART; c += KG) {
          Frag8(&now)[KG] = kf[c / KG & 1];
          if (c + KG < part + KPART) {
#pragma unroll
            for (int i = 0; i < KG; ++i) kf[(c / KG & 1) ^ 1][i].u = keys(c + KG + i);
          }
          __builtin_amdgcn_sched_barrier(0);
          if ((c + KG) * 32 > hd) {      // (pieces behind the key's end: zeros, whatever lies there)
#pragma unroll
            for (int i = 0; i < KG; ++i)
              if ((c + i) * 32 + kb * 8 >= hd) now[i].u = make_uint4(0, 0, 0, 0);
          }
#pragma unroll
          for (int i = 0; i < KG; i += 2) {
            sc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(now[i].v, qreg[c + i], sc, 0, 0, 0);
            sc2 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(now[i + 1].v, qreg[c + i + 1], sc2, 0, 0, 0);
          }
        }
      }
      sc += sc2;
      float sv[4];
      bool seen[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int key = c0 + kb * 4 + e;
        seen[e] = (key >= first || key < keep) && key <= pos;
        sv[e] = seen[e] ? (CAP ? cap.log2_score(sc[e]) : sc[e] * scale_log2) : -INFINITY;
      }
      float tmax = fmaxf(fmaxf(sv[0], sv[1]), fmaxf(sv[2], sv[3]));
      tmax = max16(tmax);
      tmax = max32(tmax);
      const float m_new = fmaxf(m_run, tmax);
      const float m_safe = m_new == -INFINITY ? 0.f : m_new;
      const float alpha = fast_exp2(m_run - m_safe);
      m_run = m_new;
      float pr[4], psum = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        pr[e] = seen[e] ? fast_exp2(sv[e] - m_safe) : 0.f;
        psum += pr[e];
      }
      l_run = l_run * alpha + psum;
      Frag4 pb;
      pb.u = make_uint2(pack_bf16x2(pr[0], pr[1]), pack_bf16x2(pr[2], pr[3]));
      if (__builtin_amdgcn_ballot_w64(alpha != 1.f) != 0) {
#pragma unroll
        for (int d = 0; d < DBL; ++d) acc[d] *= alpha;
      }
      const auto values = [&](int d) { return *reinterpret_cast<const uint2*>(vs + (size_t)((d * 4 + kb) * 16 + col) * 4); };
#pragma unroll
      for (int part = 0; part < DBL; part += VPART) {
        if (part >= dbl) continue;
        Frag4 vf[2][VG];              // (of blocks behind the last whatever lies there, in sums that are never stored)
#pragma unroll
        for (int i = 0; i < VG; ++i) vf[0][i].u = values(part + i);
#pragma unroll
        for (int d = part; d < part + VPART; d += VG) {
          if (d + VG < part + VPART) {
#pragma unroll
            for (int i = 0; i < VG; ++i) vf[(d / VG & 1) ^ 1][i].u = values(d + VG + i);
          }
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int i = 0; i < VG; ++i) acc[d + i] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(vf[d / VG & 1][i].v, pb.v, acc[d + i], 0, 0, 0);
        }
      }
    }
    buf = (buf + 1) % kStages;
  }

  if (!computes) return;
  float l = l_run;
  l = sum16(l);
  l = sum32(l);
  if (sinks) l += fast_exp2(sinks[head] * 1.4426950408889634f - m_run);
  if (col >= cnt) return;
  const float inv = 1.f / l;
  bf16_t* op = out + ((size_t)(n0 + col) * nh + head) * vd + kb * 4;
#pragma unroll
  for (int d = 0; d < DBL; ++d) {
    if (d >= dbl) continue;
    uint2 o;
    o.x = pack_bf16x2(acc[d][0] * inv, acc[d][1] * inv);
    o.y = pack_bf16x2(acc[d][2] * inv, acc[d][3] * inv);
    *reinterpret_cast<uint2*>(op + d * 16) = o;
  }
}

template <int KCH, int DBL, int HB, bool CAP>
static int launch_shared(const void* q, const void* k_cache, const void* v_cache, const int* block_tables, int max_pages,
                         const int* positions, const int* req_of_token, const int* tile_first, const int* tile_count,
                         int num_tiles, void* out, int nh, int nkv, int hd, int vd, int ps, float scale, int span, int keep,
                         const float* sinks, float softcap, hipStream_t stream) {
  const int group = nh / nkv;
  // (up to 128 KB; reads of chunks and blocks behind the true sizes stay inside, also in the last stage)
  const int all_kb = stage_kb(hd) + stage_kb(vd);
  const size_t lds = (size_t)(kStages * all_kb + KCH + DBL / 2 - all_kb) * 1024;
  if (lds > 48 * 1024) {
    static LdsLimits limits;      // per template instance
    if (!raise_lds_limit(reinterpret_cast<const void*>(&attention_tiles_shared_kernel<KCH, DBL, HB, CAP>), 128 * 1024, limits)) return -2;
  }
  const dim3 grid(num_tiles, nkv * ((group + HB - 1) / HB));
  if (grid.y > 65535) return -1;
  attention_tiles_shared_kernel<KCH, DBL, HB, CAP><<<grid, HB * 64, lds, stream>>>(
      (const bf16_t*)q, (const bf16_t*)k_cache, (const bf16_t*)v_cache, block_tables, max_pages, positions, req_of_token,
      tile_first, tile_count, (bf16_t*)out, nh, nkv, hd, vd, ps, scale * 1.4426950408889634f, span, keep, sinks,
      soft_cap(scale, softcap));
  return launch_status();
}

// Tokens that run alone (decode) at kv heads with many query heads: the 16 columns of a wave's products
// are 16 HEADS of one kv head at one token, so a key or value fetched once serves them all.  The token's
// visible keys are walked 16 at a time; step t goes to wave t % (4 nsplit) of the token's nsplit blocks
// of four waves, operands straight from the pages.  Every wave leaves an unnormalised partial result
// (its maximum, its sum, its output) and a second kernel merges a head's partials in their order and
// adds the sink: no wave waits for another.
template <int KCH, int DBL, bool CAP>
__global__ __launch_bounds__(256) void attention_heads_kernel(
    const bf16_t* __restrict__ q, const bf16_t* __restrict__ k_cache, const bf16_t* __restrict__ v_cache,
    const int* __restrict__ block_tables, int max_pages, const int* __restrict__ positions,
    const int* __restrict__ req_of_token, const int* __restrict__ single, float* __restrict__ part_o,
    float* __restrict__ part_ml, int nsplit, int nh, int nkv, int hd, int vd, int ps, float scale_log2, int span,
    int keep, SoftCap cap) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, kb = lane >> 4;
  const int group = nh / nkv, pieces = (group + 15) >> 4;
  const int kvh = blockIdx.y / pieces, in_group = (blockIdx.y % pieces) * 16 + col;
  const bool c_valid = in_group < group;
  const int head = kvh * group + min(in_group, group - 1);
  const int item = blockIdx.x, n0 = single[item];
  const int pos = positions[n0];
  const int first = span > 0 ? max(pos - span + 1, 0) : span < 0 ? pos - pos % (-span) : 0;
  const int* table = block_tables + (size_t)req_of_token[n0] * max_pages;
  const size_t k_page = (size_t)nkv * hd * ps, v_page = (size_t)nkv * vd * ps;
  const size_t k_head = (size_t)kvh * hd * ps, v_head = (size_t)kvh * vd * ps;
  const int kch = (hd + 31) >> 5, dbl = vd >> 4;
  const int parts = nsplit * 4, part = blockIdx.z * 4 + wave;

  bf16x8 qreg[KCH];
  const bf16_t* qp = q + ((size_t)n0 * nh + head) * hd + kb * 8;
#pragma unroll
  for (int c = 0; c < KCH; ++c) {
    Frag8 f;
    f.u = (c * 32 + kb * 8 < hd) ? *reinterpret_cast<const uint4*>(qp + c * 32) : make_uint4(0, 0, 0, 0);
    qreg[c] = f.v;
  }
  float m_run = -INFINITY, l_run = 0.f;
  float4v acc[DBL];
#pragma unroll
  for (int d = 0; d < DBL; ++d) acc[d] = float4v{0.f, 0.f, 0.f, 0.f};

  // the stages of the walk in order: those of the kept first positions that lie before the window's first
  // stage, then the window's; stage s goes to part s % parts
  const int c_first = first & ~15;
  const int kept = min((keep + 15) >> 4, c_first >> 4);
  for (int st = part;; st += parts) {
    const int c0 = st < kept ? st * 16 : c_first + (st - kept) * 16;
    if (c0 > pos) break;
    const int page = table[c0 / ps], off = c0 % ps;
    const bf16_t* kp = k_cache + (size_t)page * k_page + k_head + (size_t)(off + col) * 8;
    const bf16_t* vp = v_cache + (size_t)page * v_page + v_head + (size_t)((off >> 2) + kb) * 64 + col * 4;
    Frag8 kreg[KCH];
#pragma unroll
    for (int c = 0; c < KCH; ++c)
      kreg[c].u = (c * 32 + kb * 8 < hd) ? *reinterpret_cast<const uint4*>(kp + (size_t)(c * 4 + kb) * ps * 8)
                                         : make_uint4(0, 0, 0, 0);
    Frag4 vreg[DBL];
#pragma unroll
    for (int d = 0; d < DBL; ++d)
      vreg[d].u = d < dbl ? *reinterpret_cast<const uint2*>(vp + (size_t)d * (ps >> 2) * 64) : make_uint2(0, 0);
    float4v sc = {0.f, 0.f, 0.f, 0.f}, sc2 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < KCH; c += 2) {
      if (c < kch) sc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kreg[c].v, qreg[c], sc, 0, 0, 0);
      if (c + 1 < kch) sc2 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kreg[c + 1].v, qreg[c + 1], sc2, 0, 0, 0);
    }
    sc += sc2;
    float sv[4];
    bool seen[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int key = c0 + kb * 4 + e;
      seen[e] = (key >= first || key < keep) && key <= pos;
      sv[e] = seen[e] ? (CAP ? cap.log2_score(sc[e]) : sc[e] * scale_log2) : -INFINITY;
    }
    float tmax = fmaxf(fmaxf(sv[0], sv[1]), fmaxf(sv[2], sv[3]));
    tmax = max16(tmax);
    tmax = max32(tmax);
    const float m_new = fmaxf(m_run, tmax);   // finite: a step holds at least one visible key
    const float alpha = fast_exp2(m_run - m_new);
    m_run = m_new;
    float pr[4], psum = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      pr[e] = seen[e] ? fast_exp2(sv[e] - m_new) : 0.f;
      psum += pr[e];
    }
    l_run = l_run * alpha + psum;
    Frag4 pb;
    pb.u = make_uint2(pack_bf16x2(pr[0], pr[1]), pack_bf16x2(pr[2], pr[3]));
    const bool edge = c0 + 15 > pos;
#pragma unroll
    for (int d = 0; d < DBL; ++d) {
      if (d >= dbl) continue;
      short4v tv = vreg[d].v;
      if (edge) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (c0 + kb * 4 + e > pos) tv[e] = 0;
      }
      float4v a = acc[d];
      a *= alpha;
      acc[d] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(tv, pb.v, a, 0, 0, 0);
    }
  }
  float l = l_run;
  l = sum16(l);
  l = sum32(l);
  if (!c_valid) return;
  // partial rows [item][head][part]: (maximum, sum), then the output
  const size_t prow = ((size_t)item * nh + head) * parts + part;
  if (kb == 0) {
    part_ml[prow * 2] = m_run;
    part_ml[prow * 2 + 1] = l;
  }
  float* po = part_o + prow * vd + kb * 4;
#pragma unroll
  for (int d = 0; d < DBL; ++d) {
    if (d >= dbl) continue;
    *reinterpret_cast<float4*>(po + d * 16) = make_float4(acc[d][0], acc[d][1], acc[d][2], acc[d][3]);
  }
}

// out[token][head] = sum_p w_p o_p / (sum_p w_p l_p + exp(sink)), w_p = exp2(m_p - max m); a part without
// keys has m = -inf and weighs nothing (whatever lies in its output).  A block is 256 channels of a (token, head), a lane one of them, or
// (SHARED, of more than 16 parts) 64, of which its waves take every fourth part and add up in wave order.  Lane p of every wave finds
// part p's weight (up to 64 parts) while the outputs are on their way, a lane's LOADS asked for together: fetched eight at a time, each behind a
// look at its weight, 36 parts of 448 channels of 32 heads took 9.8 us, so 3.  Few parts are a step of many tokens, bound by its blocks and
// loads: with four waves a channel and 16 loads whatever the parts, 100 tokens of 32 heads of 512 / 448, 300 keys, took 69 us with their attention, so 48.
template <bool SHARED, int LOADS>
__global__ __launch_bounds__(256) void attention_heads_merge_kernel(
    const float* __restrict__ part_o, const float* __restrict__ part_ml, const int* __restrict__ single,
    bf16_t* __restrict__ out, int parts, int nh, int vd, const float* __restrict__ sinks) {
  constexpr int kEvery = SHARED ? 4 : 1;
  __shared__ float sums[4][64];
  const int item = blockIdx.x, head = blockIdx.y, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int d = SHARED ? blockIdx.z * 64 + lane : blockIdx.z * 256 + threadIdx.x, first = SHARED ? wave : 0;
  if (!SHARED && d - lane >= vd) return;      // (the whole wave)
  const size_t row = ((size_t)item * nh + head) * parts;
  const float2 ml = reinterpret_cast<const float2*>(part_ml)[row + min(lane, parts - 1)];
  const float* po = part_o + row * vd + min(d, vd - 1);
  float v[LOADS];
#pragma unroll
  for (int u = 0; u < LOADS; ++u) v[u] = po[(size_t)min(first + kEvery * u, parts - 1) * vd];
  const float m = lane < parts ? ml.x : -INFINITY;
  const float mx = wave_max(m);                       // finite: the part that holds the token's own key
  const float w = m == -INFINITY ? 0.f : fast_exp2(m - mx);
  float denom = wave_sum(m == -INFINITY ? 0.f : w * ml.y);
  if (sinks) denom += fast_exp2(sinks[head] * 1.4426950408889634f - mx);
  float o = 0.f;
#pragma unroll
  for (int u = 0; u < LOADS; ++u) {
    const float of = __shfl(w, min(first + kEvery * u, 63), kWave);      // (zero from `parts` on)
    o = of != 0.f ? fmaf(of, v[u], o) : o;
  }
  bf16_t* const op = out + ((size_t)single[item] * nh + head) * vd + d;
  if constexpr (SHARED) {
    sums[wave][lane] = o;
    __syncthreads();
    if (wave == 0 && d < vd) *op = float_to_bf16(((sums[0][lane] + sums[1][lane]) + (sums[2][lane] + sums[3][lane])) / denom);
  } else if (d < vd) {
    *op = float_to_bf16(o / denom);
  }
}

// Whether the heads of a kv head share its keys and values through LDS (see the shared kernel).
bool tiles_share(int group, int hd, int vd) { return group >= 4 || (group >= 2 && hd <= 128 && vd <= 128 && hd + vd > 128); }

}  // namespace

// Tiles of up to 16 consecutive tokens of one request (tile_first, tile_count), bfloat16.  Returns -2
// for a shape the kernel does not take (the caller uses the generic kernel).
TK_API int tk_attention_tiles(const void* q, const void* k_cache, const void* v_cache, const int* block_tables,
                              int max_pages, const int* positions, const int* req_of_token, const int* tile_first,
                              const int* tile_count, int num_tiles, void* out, int nh, int nkv, int hd, int vd, int ps,
                              float scale, int span, int keep, const float* sinks, float softcap, hipStream_t stream) {
  if (num_tiles <= 0) return 0;
  if (keep < 0 || (keep > 0 && span <= 0) || !(softcap >= 0.f)) return -1;
  if (nkv <= 0 || nh % nkv != 0 || hd < 8 || hd % 8 != 0 || vd < 16 || vd % 16 != 0 || ps < 16 || ps % 16 != 0) return -2;
  if (hd > 512 || vd > 512 || (uintptr_t)q % 16 != 0 || (uintptr_t)k_cache % 16 != 0 || (uintptr_t)v_cache % 16 != 0 ||
      (uintptr_t)out % 8 != 0)
    return -2;
  const int group = nh / nkv;
  if (tiles_share(group, hd, vd)) {
#define TK_SHARED_AS(KCH_, DBL_, HB_, CAP_)                                                                     \
  launch_shared<KCH_, DBL_, HB_, CAP_>(q, k_cache, v_cache, block_tables, max_pages, positions, req_of_token,   \
                                       tile_first, tile_count, num_tiles, out, nh, nkv, hd, vd, ps, scale, span, \
                                       keep, sinks, softcap, stream)
#define TK_SHARED(KCH_, DBL_, HB_) \
  (softcap > 0.f ? TK_SHARED_AS(KCH_, DBL_, HB_, true) : TK_SHARED_AS(KCH_, DBL_, HB_, false))
    if (hd <= 128 && vd <= 128) return group > 4 ? TK_SHARED(4, 8, 8) : group > 2 ? TK_SHARED(4, 8, 4) : TK_SHARED(4, 8, 2);
    if (hd <= 256 && vd <= 256) return group > 4 ? TK_SHARED(8, 16, 8) : TK_SHARED(8, 16, 4);
    return group > 4 ? TK_SHARED(16, 32, 8) : TK_SHARED(16, 32, 4);
#undef TK_SHARED
#undef TK_SHARED_AS
  }
  const dim3 grid(num_tiles, (nh + kHeadsPerBlock - 1) / kHeadsPerBlock);
  if (grid.y > 65535) return -1;
#define TK_TILES_AS(KCH_, DBL_, CAP_)                                                                          \
  attention_tiles_kernel<KCH_, DBL_, CAP_><<<grid, kHeadsPerBlock * 64, 0, stream>>>(                          \
      (const bf16_t*)q, (const bf16_t*)k_cache, (const bf16_t*)v_cache, block_tables, max_pages, positions,    \
      req_of_token, tile_first, tile_count, (bf16_t*)out, nh, nkv, hd, vd, ps, scale * 1.4426950408889634f,    \
      span, keep, sinks, soft_cap(scale, softcap))
#define TK_TILES(KCH_, DBL_)                          \
  do {                                                \
    if (softcap > 0.f) TK_TILES_AS(KCH_, DBL_, true); \
    else TK_TILES_AS(KCH_, DBL_, false);              \
  } while (0)
  if (hd <= 128 && vd <= 128) TK_TILES(4, 8);
  else if (hd <= 256 && vd <= 256) TK_TILES(8, 16);
  else TK_TILES(16, 32);
#undef TK_TILES
#undef TK_TILES_AS
  return launch_status();
}

// Single tokens (`single`: their rows, num_single of them), bfloat16, for kv heads with many query heads.
// part_o: float32 [num_single * nh * 4 nsplit * vd], part_ml: float32 [num_single * nh * 4 nsplit * 2].
TK_API int tk_attention_heads(const void* q, const void* k_cache, const void* v_cache, const int* block_tables,
                              int max_pages, const int* positions, const int* req_of_token, const int* single,
                              int num_single, void* out, float* part_o, float* part_ml, int nsplit, int nh, int nkv,
                              int hd, int vd, int ps, float scale, int span, int keep, const float* sinks,
                              float softcap, hipStream_t stream) {
  if (num_single <= 0) return 0;
  if (keep < 0 || (keep > 0 && span <= 0) || !(softcap >= 0.f)) return -1;
  if (nkv <= 0 || nh % nkv != 0 || hd < 8 || hd % 8 != 0 || vd < 16 || vd % 16 != 0 || ps < 16 || ps % 16 != 0) return -2;
  if (hd > 512 || vd > 512 || (uintptr_t)q % 16 != 0 || (uintptr_t)k_cache % 16 != 0 || (uintptr_t)v_cache % 16 != 0 ||
      (uintptr_t)part_o % 16 != 0 || (uintptr_t)part_ml % 8 != 0 || nsplit < 1 || nsplit > 16 || nh > 65535)    // (the merge: up to 64 parts)
    return -2;
  const int group = nh / nkv;
  const dim3 grid(num_single, nkv * ((group + 15) / 16), nsplit);
  if (grid.y > 65535) return -1;
#define TK_HEADS_AS(KCH_, DBL_, CAP_)                                                                         \
  attention_heads_kernel<KCH_, DBL_, CAP_><<<grid, 256, 0, stream>>>(                                         \
      (const bf16_t*)q, (const bf16_t*)k_cache, (const bf16_t*)v_cache, block_tables, max_pages, positions,   \
      req_of_token, single, part_o, part_ml, nsplit, nh, nkv, hd, vd, ps, scale * 1.4426950408889634f, span, keep, \
      soft_cap(scale, softcap))
#define TK_HEADS(KCH_, DBL_)                          \
  do {                                                \
    if (softcap > 0.f) TK_HEADS_AS(KCH_, DBL_, true); \
    else TK_HEADS_AS(KCH_, DBL_, false);              \
  } while (0)
  if (hd <= 128 && vd <= 128) TK_HEADS(4, 8);
  else if (hd <= 256 && vd <= 256) TK_HEADS(8, 16);
  else TK_HEADS(16, 32);
#undef TK_HEADS
#undef TK_HEADS_AS
  const int parts = nsplit * 4;
#define TK_MERGE(SHARED_, LOADS_, CHANNELS_)                                                                              \
  attention_heads_merge_kernel<SHARED_, LOADS_>                                                                           \
      <<<dim3(num_single, nh, (vd + CHANNELS_ - 1) / CHANNELS_), CHANNELS_ > vd && !SHARED_ ? (vd + 63) / 64 * 64 : 256, 0, stream>>>( \
          part_o, part_ml, single, (bf16_t*)out, parts, nh, vd, sinks)
  if (parts <= 4) TK_MERGE(false, 4, 256);
  else if (parts <= 8) TK_MERGE(false, 8, 256);
  else if (parts <= 16) TK_MERGE(false, 16, 256);
  else TK_MERGE(true, 16, 64);
#undef TK_MERGE
  return launch_status();
}

// Whether tk_attention_tiles has the heads of a kv head share a block (1 or 0).
TK_API int tk_attention_tiles_share(int group, int hd, int vd) { return tiles_share(group, hd, vd); }

TK_SLOTS(tk_attention_tiles)
TK_SLOTS(tk_attention_heads)
