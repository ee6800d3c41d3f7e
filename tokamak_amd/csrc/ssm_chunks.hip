// The selective state-space scan in chunks of 64 tokens on the matrix cores (gfx950): the form of portions for the scan
// of ssm.hip.
//
// Requests of `least` tokens and more; shorter ones are the walk's, whoever stands beside them.
//
//     S <- a_t S + dt_t B_t x_t^T,  y_t = S^T C_t + D x_t,   dt_t = softplus(dt_in + bias), a_t = exp(-exp(A_log) dt_t)
//
// The decay is one number a head and token, so with S the state before a chunk
//     y_i = (prod_(l <= i) a_l) S^T C_i + sum_(j <= i) (C_i . B_j) dt_j (prod_(j < l <= i) a_l) x_j + D x_i
//     S' = (prod a_l) S + sum_j dt_j (prod_(l > j) a_l) B_j x_j^T
// and a portion's chunks run side by side: every chunk's own sum (sums), per request the chunks in order (starts), every
// chunk's outputs (outputs).  Products of decays are formed as products, at most one; none is divided by another.
// Everything is float32 behind the convolution's output, the products are the float32 matrix instruction's (16 x 16 x
// 4).  Its k index may name any four places as long as both operands agree: index g of step r is place 4 g + r
// of a group of 16, so that a lane's operands of four steps are one 16-byte read.  Sums run in four accumulators: one
// chain of up to 192 products was further from the 64-bit result than the walk, whose sums run over lanes.  Products of
// decays are rounded once, the newest tokens join a state's sum last, and from chunk to chunk a state is carried in float64:
// outputs 0.91 to 0.99, states 0.93 to 1.00 of the walk's distance (products of decays rounded at each factor and states
// carried in float32: up to 1.06 and 1.05).  float32 storage keeps the walk: with operands of 24 bits the products C B^T
// round where the walk does not, and its outputs would be 1.2 to 1.4 times as far.
//
// Walked a token at a time (four state rows by four columns a thread, twice over in chunks) this was bound by
// the LDS reads of B and C, two 16-byte reads a token for 32 multiply-adds: 2,048 tokens of 32
// heads of 128 x 64, one group, 273 us, 82 here; of 128 heads in 8 groups 920, 233 here.  B and C belong to a group of
// heads: a block takes a few heads of a group and forms C B^T, and reads its operands of B and C, once for them.
#include "common.h"
#include "request_tiles.h"
#include "short_conv.h"
#include "slots.h"

using namespace tk;

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kTokens = 64;       // tokens of a chunk: four tiles of 16, one a wave
constexpr int kThreads = 256;
constexpr int kMaxDim = 128;
constexpr int kMaxHeads = 4;      // heads a block takes, one after the other

struct Shape {
  int R, heads, groups, vdim, C, dt_col, per, least;      // per: heads a block takes (a divisor of a group's heads)
  long ld;
};

__device__ __forceinline__ f32x4 load4(const bf16_t* p) {
  const uint2 u = *reinterpret_cast<const uint2*>(p);
  return f32x4{__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u), __uint_as_float(u.y << 16), __uint_as_float(u.y & 0xffff0000u)};
}

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// step sizes and decays of the block's heads over the chunk (behind its end: nothing enters, nothing decays)
// `pad`: places before the first token
__device__ __forceinline__ void step_sizes(const RowsIn& in, const Shape& sh, const float* dt_bias, const float* a_log, int head0,
                                           int first, int count, int pad, float (*dts)[kTokens], float (*as)[kTokens]) {
  const int h = threadIdx.x / kTokens, place = threadIdx.x % kTokens, t = place - pad;
  if (h >= sh.per) return;
  const bool there = t >= 0 && t < count;
  const float dt = softplus(load_in<bf16_t>(in, (size_t)(first + max(0, min(t, count - 1))) * sh.ld + sh.dt_col + head0 + h) + dt_bias[head0 + h]);
  dts[h][place] = there ? dt : 0.f;
  as[h][place] = there ? expf(-expf(a_log[head0 + h]) * dt) : 1.f;
}

__device__ __forceinline__ f32x4 sum4(const f32x4 (&x)[4]) { return (x[0] + x[1]) + (x[2] + x[3]); }

// x of a head's chunk, times `scale` a place, into dst [64][pitch] (zeros before its first and behind its last token)
template <typename SCALE>
__device__ __forceinline__ void stage_x(float* dst, int pitch, const bf16_t* u, const Shape& sh, int head, int first, int count, int pad,
                                        SCALE scale) {
  const int quads = sh.vdim / 4;
  for (int e = threadIdx.x; e < kTokens * quads; e += kThreads) {
    const int place = e / quads, v = (e - place * quads) * 4, t = place - pad;
    f32x4 x = load4(u + (size_t)(first + max(0, min(t, count - 1))) * sh.C + head * sh.vdim + v);
    x = t >= 0 && t < count ? x * scale(place) : f32x4{0.f, 0.f, 0.f, 0.f};
    *reinterpret_cast<f32x4*>(dst + place * pitch + v) = x;
  }
}

// (an odd multiple of 16: four rows' 16 columns lie in different banks)
__host__ __device__ inline int sums_pitch(int vdim) { return (vdim / 16 | 1) * 16; }

// chunk_state[chunk][head] = sum_j dt_j (prod_(l > j) a_l) B_j x_j^T, chunk_decay[chunk][head] = prod a_l.  A wave takes the
// tiles w and w + 4 of 16 state rows; its operands of B stay in registers over the heads.  Tokens enter in their order, the
// newest, which weigh most, last: what is rounded before them is small.  So a chunk of few tokens holds them in its last
// places here.
template <int S16>
__global__ __launch_bounds__(kThreads) void ssm_chunk_sums_kernel(const bf16_t* __restrict__ u, RowsIn dt_in, const float* __restrict__ dt_bias,
                                                                  const float* __restrict__ a_log, const int* __restrict__ q_start,
                                                                  float* __restrict__ chunk_state, double* __restrict__ chunk_decay, Shape sh) {
  constexpr int ns = 16 * S16, TILES = (S16 + 3) / 4;
  extern __shared__ __attribute__((aligned(16))) float xx[];
  __shared__ float dts[kMaxHeads][kTokens], as[kMaxHeads][kTokens], ws[kMaxHeads][kTokens];
  RequestTile rt;
  if (!find_request_tile(q_start, sh.R, kTokens, blockIdx.x, rt, sh.least)) return;
  const int first = q_start[rt.req] + rt.index * kTokens, count = min(kTokens, q_start[rt.req + 1] - first);
  const int head0 = blockIdx.y * sh.per, group = head0 / (sh.heads / sh.groups), vp = sums_pitch(sh.vdim);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, quad = lane >> 4;
  const int pad = kTokens - count;
  step_sizes(dt_in, sh, dt_bias, a_log, head0, first, count, pad, dts, as);
  float b[TILES][16];
#pragma unroll
  for (int i = 0; i < TILES; ++i)
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        b[i][4 * s + r] = Elem<bf16_t>::load(u + (size_t)(first + max(16 * s + 4 * r + quad - pad, 0)) * sh.C + sh.heads * sh.vdim +
                                        group * ns + min(16 * (wave + 4 * i), ns - 16) + col);
  __syncthreads();
  static_assert(kTokens == kWave, "a lane a token");
  if (wave < sh.per) {      // the products of the decays behind a token, rounded once (a state lives on; rounded at each of their
    double p = lane + 1 < kTokens ? as[wave][lane + 1] : 1.f;      // factors it was 1.03 to 1.18 times as far off as the walk's)
#pragma unroll
    for (int m = 1; m < kTokens; m <<= 1) {
      const double further = __shfl_down(p, m, kWave);
      if (lane + m < kTokens) p *= further;
    }
    ws[wave][lane] = (float)(dts[wave][lane] * p);
    if (lane == 0) chunk_decay[(size_t)blockIdx.x * sh.heads + head0 + wave] = p * as[wave][0];
  }
  const int skipped = pad / 16;      // groups of 16 places without a token
  for (int h = 0; h < sh.per; ++h) {
    __syncthreads();
    stage_x(xx, vp, u, sh, head0 + h, first, count, pad, [&](int place) { return ws[h][place]; });
    __syncthreads();
    float* out = chunk_state + ((size_t)blockIdx.x * sh.heads + head0 + h) * ns * sh.vdim;
    for (int v0 = 0; v0 < sh.vdim; v0 += 16) {
      f32x4 acc[TILES][4];
#pragma unroll
      for (int i = 0; i < TILES; ++i)
#pragma unroll
        for (int s = 0; s < 4; ++s) acc[i][s] = f32x4{0.f, 0.f, 0.f, 0.f};
      f32x4 sum[TILES];      // the newest four tokens, which weigh most, join the others' sum
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        if (s < skipped) continue;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float x = xx[(16 * s + 4 * r + quad) * vp + v0 + col];
#pragma unroll
          for (int i = 0; i < TILES; ++i) {
            if (r == 3 && s == 3) sum[i] = mfma4(x, b[i][4 * s + r], sum4(acc[i]));
            else acc[i][s] = mfma4(x, b[i][4 * s + r], acc[i][s]);
          }
        }
      }
#pragma unroll
      for (int i = 0; i < TILES; ++i)
        if (16 * (wave + 4 * i) < ns)
          *reinterpret_cast<f32x4*>(out + ((size_t)(v0 / 4 + quad) * ns + 16 * (wave + 4 * i) + col) * 4) = sum[i];
    }
  }
}

// Per (request, head), a thread an element of the state: chunk_state holds every chunk's own sum on entry and its start
// state on return; the request's state moves to the end of the step's tokens.  Eight chunks' sums in flight.
__global__ __launch_bounds__(256) void ssm_chunk_starts_kernel(float* __restrict__ state, const int* __restrict__ q_start,
                                                               const int* __restrict__ state_slots, float* __restrict__ chunk_state,
                                                               const double* __restrict__ chunk_decay, int heads, int elems, int least) {
  const int req = blockIdx.x, head = blockIdx.y, e = blockIdx.z * blockDim.x + threadIdx.x;
  const int count = request_tiles(q_start, req, kTokens, least);
  if (count == 0) return;
  const int before = tiles_before(q_start, req, kTokens, least);
  if (e >= elems) return;
  float* S = state + ((size_t)state_slots[req] * heads + head) * elems + e;
  float* cs = chunk_state + ((size_t)before * heads + head) * elems + e;
  const double* decay = chunk_decay + (size_t)before * heads + head;
  const size_t stride = (size_t)heads * elems;
  double s = *S;      // (rounded where a chunk reads it, not from chunk to chunk)
  for (int c0 = 0; c0 < count; c0 += 8) {
    float own[8];
    double d[8];
#pragma unroll
    for (int x = 0; x < 8; ++x) {
      const int c = min(c0 + x, count - 1);
      own[x] = cs[c * stride];
      d[x] = decay[(size_t)c * heads];
    }
#pragma unroll
    for (int x = 0; x < 8; ++x) {
      if (c0 + x < count) {
        cs[(c0 + x) * stride] = (float)s;
        s = fma(d[x], s, (double)own[x]);
      }
    }
  }
  *S = (float)s;
}

// The outputs of a chunk, wave w the tokens 16 w .. + 16: its rows of C and of C B^T stay in registers over the heads; a head's
// x and start state pass LDS, and so do its products of decays, on their way from a lane a column to the operand's order.
template <int S16>
__global__ __launch_bounds__(kThreads) void ssm_chunk_outputs_kernel(const bf16_t* __restrict__ u, RowsIn dt_in, const float* __restrict__ dt_bias,
                                                                     const float* __restrict__ a_log, const float* __restrict__ skip,
                                                                     const int* __restrict__ q_start, const float* __restrict__ chunk_state,
                                                                     float* __restrict__ y, Shape sh) {
  constexpr int ns = 16 * S16, sp = ns + 4, pp = kTokens + 4;
  extern __shared__ __attribute__((aligned(16))) float lds[];
  __shared__ float dts[kMaxHeads][kTokens], as[kMaxHeads][kTokens];
  __shared__ __attribute__((aligned(16))) float whole[kTokens];
  RequestTile rt;
  if (!find_request_tile(q_start, sh.R, kTokens, blockIdx.x, rt, sh.least)) return;
  const int first = q_start[rt.req] + rt.index * kTokens, count = min(kTokens, q_start[rt.req + 1] - first);
  const int head0 = blockIdx.y * sh.per, group = head0 / (sh.heads / sh.groups), vp = sh.vdim + 4;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, quad = lane >> 4;
  float* const pd = lds;                      // [64][pp]
  float* const xx = pd + kTokens * pp;        // [64][vp]
  float* const st = xx + kTokens * vp;        // [vdim][sp]
  step_sizes(dt_in, sh, dt_bias, a_log, head0, first, count, 0, dts, as);
  const bool works = wave * 16 < count;
  const bf16_t* const bc = u + sh.heads * sh.vdim + group * ns + 4 * quad;       // a row's B from here; its C groups * ns further
  f32x4 c[S16], g[4];
#pragma unroll
  for (int s = 0; s < S16; ++s) c[s] = load4(bc + (size_t)(first + min(16 * wave + col, count - 1)) * sh.C + sh.groups * ns + 16 * s);
#pragma unroll
  for (int jt = 0; jt < 4; ++jt) {
    f32x4 sum[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) sum[s] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (works && jt <= wave) {
      f32x4 b[S16];
#pragma unroll
      for (int s = 0; s < S16; ++s) b[s] = load4(bc + (size_t)(first + min(16 * jt + col, count - 1)) * sh.C + 16 * s);
#pragma unroll
      for (int s = 0; s < S16; ++s)
#pragma unroll
        for (int r = 0; r < 4; ++r) sum[s & 3] = mfma4(c[s][r], b[s][r], sum[s & 3]);
    }
    g[jt] = sum4(sum);
  }
  for (int h = 0; h < sh.per; ++h) {
    const int head = head0 + h;
    __syncthreads();
    stage_x(xx, vp, u, sh, head, first, count, 0, [](int) { return 1.f; });
    const float* const S = chunk_state + ((size_t)blockIdx.x * sh.heads + head) * ns * sh.vdim;
    for (int e = threadIdx.x; e < sh.vdim / 4 * ns; e += kThreads) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(S + 4 * e);
      const int v = e / ns * 4, d = e % ns;
#pragma unroll
      for (int r = 0; r < 4; ++r) st[(v + r) * sp + d] = x[r];
    }
    __syncthreads();
    if (!works) continue;
    // lane j: dt_j times the products of decays from behind j to each of the wave's rows; column 0 also the whole products.
    // Rounded once; a group of 16 places is gone past by its own product, found by a scan over the lanes.
    {
      const float dt = dts[h][lane], a0 = as[h][0];
      double p = (lane & 15) < 15 ? as[h][lane + 1] : 1.f;      // (behind j to the end of its group)
#pragma unroll
      for (int m = 1; m < 16; m <<= 1) {
        const double further = __shfl_down(p, m, kWave);
        if ((lane & 15) + m < 16) p *= further;
      }
      const double group_product = p * as[h][lane];              // (of its group, in the group's first lane)
#pragma unroll
      for (int s = 1; s < 3; ++s) {
        const double product = __shfl(group_product, 16 * s, kWave);
        if (s < wave && lane < 16 * s) p *= product;
      }
      if (lane >= 16 * wave) p = 1.0;
#pragma unroll
      for (int x = 0; x < 16; ++x) {
        const int i = 16 * wave + x;
        p *= i > lane ? as[h][i] : 1.f;
        pd[i * pp + lane] = i >= lane ? (float)(p * dt) : 0.f;
        if (lane == 0) whole[i] = (float)(p * a0);
      }
    }
    wave_lds_sync();
#pragma unroll
    for (int jt = 0; jt < 4; ++jt)
      if (jt <= wave)
#pragma unroll
        for (int r = 0; r < 4; ++r) pd[(16 * wave + 4 * quad + r) * pp + 16 * jt + col] *= g[jt][r];
    wave_lds_sync();
    f32x4 p[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) p[s] = *reinterpret_cast<const f32x4*>(pd + (16 * wave + col) * pp + 16 * s + 4 * quad);
    const f32x4 scale = *reinterpret_cast<const f32x4*>(whole + 16 * wave + 4 * quad);
    const float own = skip[head];
    for (int v0 = 0; v0 < sh.vdim; v0 += 16) {
      f32x4 fars[4], nears[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) fars[s] = nears[s] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < S16; ++s) {
        const f32x4 x = *reinterpret_cast<const f32x4*>(st + (v0 + col) * sp + 16 * s + 4 * quad);
#pragma unroll
        for (int r = 0; r < 4; ++r) fars[s & 3] = mfma4(c[s][r], x[r], fars[s & 3]);
      }
#pragma unroll
      for (int s = 0; s < 4; ++s)
        if (s <= wave)
#pragma unroll
          for (int r = 0; r < 4; ++r) nears[s] = mfma4(p[s][r], xx[(16 * s + 4 * quad + r) * vp + v0 + col], nears[s]);
      const f32x4 far = sum4(fars), near = sum4(nears);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = 16 * wave + 4 * quad + r;
        if (i < count)
          y[((size_t)(first + i) * sh.heads + head) * sh.vdim + v0 + col] = fmaf(own, xx[i * vp + v0 + col], fmaf(scale[r], far[r], near[r]));
      }
    }
  }
}

template <int S16>
int launch(const bf16_t* u, RowsIn dt, const float* dt_bias, const float* a_log, const float* skip, float* state, const int* q_start,
           const int* slots, float* y, int chunks, const Shape& sh, float* chunk_state, double* chunk_decay, hipStream_t stream) {
  constexpr int ns = 16 * S16;
  const int vp = sh.vdim + 4, elems = ns * sh.vdim;
  const size_t sums_lds = (size_t)kTokens * sums_pitch(sh.vdim) * 4;
  const size_t out_lds = ((size_t)kTokens * (kTokens + 4) + (size_t)kTokens * vp + (size_t)sh.vdim * (ns + 4)) * 4;
  static bool raised[64] = {};      // (the attribute belongs to a function on a device)
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return -1;
  if (!raised[dev]) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(&ssm_chunk_sums_kernel<S16>), hipFuncAttributeMaxDynamicSharedMemorySize, 128 * 1024) != hipSuccess ||
        hipFuncSetAttribute(reinterpret_cast<const void*>(&ssm_chunk_outputs_kernel<S16>), hipFuncAttributeMaxDynamicSharedMemorySize, 128 * 1024) != hipSuccess)
      return -1;
    raised[dev] = true;
  }
  const dim3 grid(chunks, sh.heads / sh.per);
  ssm_chunk_sums_kernel<S16><<<grid, kThreads, sums_lds, stream>>>(u, dt, dt_bias, a_log, q_start, chunk_state, chunk_decay, sh);
  ssm_chunk_starts_kernel<<<dim3(sh.R, sh.heads, (elems + 255) / 256), 256, 0, stream>>>(state, q_start, slots, chunk_state, chunk_decay,
                                                                                       sh.heads, elems, sh.least);
  ssm_chunk_outputs_kernel<S16><<<grid, kThreads, out_lds, stream>>>(u, dt, dt_bias, a_log, skip, q_start, chunk_state, y, sh);
  return launch_status();
}

}  // namespace

// Operands, state and y as in tk_ssd_scan (ssm.hip), bfloat16 storage; ns 16, 32, 64 or 128, vdim a multiple of 16 up to 128, u on a 16-byte
// border.  least: requests of fewer tokens are left alone; chunks: at least the chunks of 64 tokens that the others have together; per: heads a block takes, a divisor of
// the heads of a group, up to 4; chunk_state float32 [chunks, heads, vdim / 4, ns, 4] and chunk_decay float64 [chunks,
// heads] are scratch.
TK_API int tk_ssm_chunks(const void* u, const void* dt, int dt_f32, int dt_parts, long dt_stride, long ld, int dt_col,
                         const float* dt_bias, const float* a_log, const float* skip, float* state, const int* q_start,
                         const int* state_slots, float* y, int R, int heads, int groups, int ns, int vdim, int least, int chunks, int per,
                         float* chunk_state, double* chunk_decay, hipStream_t stream) {
  if (R <= 0) return 0;
  if (heads < 1 || heads > 65535 || groups < 1 || heads % groups != 0 || (ns != 16 && ns != 32 && ns != 64 && ns != 128) || vdim < 16 ||
      vdim > kMaxDim || vdim % 16 != 0 || least < 1 || chunks < 1 || per < 1 || per > kMaxHeads || (heads / groups) % per != 0 || dt_parts < 1 ||
      (dt_parts > 1 && !dt_f32) || (uintptr_t)u % 16 != 0 || chunk_state == nullptr || chunk_decay == nullptr)
    return -1;
  const RowsIn in{dt, dt_f32, dt_parts, dt_stride};
  const Shape sh{R, heads, groups, vdim, heads * vdim + 2 * groups * ns, dt_col, per, least, ld};
#define TK_GO(S16_) return launch<S16_>((const bf16_t*)u, in, dt_bias, a_log, skip, state, q_start, state_slots, y, chunks, sh, chunk_state, chunk_decay, stream)
  if (ns == 16) TK_GO(1);
  if (ns == 32) TK_GO(2);
  if (ns == 64) TK_GO(4);
  TK_GO(8);
#undef TK_GO
}

TK_SLOTS(tk_ssm_chunks)
