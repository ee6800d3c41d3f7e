// Token selection from float32 logits [M, V]: greedy argmax, and temperature /
// top-k / top-p sampling with a per-request counter-based random number.
//
// Filter order and rules follow the reference sampler
// (src/tokamak/sampling/sampler.py:34-39,64-84): divide by temperature; top-k
// keeps every logit >= the k-th largest (ties at the threshold survive); top-p
// sorts descending and drops a token iff the mass ranked before it already
// reaches top_p (the best token always survives); softmax over what is left;
// one draw.  No sort is done here: thresholds are found over the ordered-integer image of the float values, first
// the histogram bin that holds one (one pass over the row), then among that bin's values alone, by ranks where they
// are few and by two more radix levels where they are many.
#include "common.h"
#include "no_alloc.h"

#include <cstring>
#include <mutex>
#include <type_traits>

using namespace tk;

// ---------------------------------------------------------------------------
// argmax: first maximum wins (lowest index), NaN never wins.  A row is cut into
// kArgmaxSegments pieces, one block each, so that a few rows still fill the chip;
// a second small kernel picks among the pieces' winners.
// ---------------------------------------------------------------------------
constexpr int kArgmaxSegments = 32;
constexpr int kArgmaxThreads = 256;

__device__ __forceinline__ void argmax_take(float& bv, int& bi, float v, int i) {
  if (v > bv || (v == bv && i < bi)) {
    bv = v;
    bi = i;
  }
}

constexpr int kBins = 4096;  // histogram bins of one radix pass (12 bits)
constexpr int kCoarse = kBins / kWave;
constexpr int kHistWords = kBins + kCoarse;     // of a row in memory
constexpr int kCandidates = 16384;
constexpr int kShareThreads = 256;
constexpr int kFew = 256;          // values among which a threshold is found by ranks
constexpr int kLevelBins = 1024;   // of the second and the third level (ten bits each)

struct FirstLevel {
  int bin;                          // the first histogram's bin that holds the threshold
  uint32_t k_remaining;             // of top-k: how many of that bin's values still count
  unsigned long long p_remaining;   // of top-p alone: how much of that bin's mass
  uint32_t total;                   // values in that bin and above it (of a row whose first pass is still to be made: 0)
  uint32_t inside;                  // values in that bin
};

// Scratch of the rows with thresholds, null: every row is sampled by one block alone.  The argmax pass zeroes what the
// kernels add into (hist32, hist64, count), and says of every row that has a threshold that its first pass is still to be made (level).
struct SharedRows {
  uint32_t* hist32;              // [M][kBins + kCoarse]: the bins, then the sums of every 64 of them
  unsigned long long* hist64;    // [M][kBins + kCoarse]
  uint32_t* count;               // [M] entries of the list
  uint32_t* cand;                // [M][kCandidates] ordered images
  uint8_t* segment;              // [M][kCandidates]
  unsigned long long* above;     // [M][segments] mass of what is kept for certain and not listed
  FirstLevel* level;             // [M] where the first threshold lies
};

// A step's sampling parameters in device memory.
struct RowParams {
  const unsigned long long *seeds, *draws;     // [M] the request's seed and how many draws it has made
  const float *temperature, *top_p;            // [M]
  const int* top_k;                            // [M]
  const int* rows;                             // [shared] the rows that have a threshold, ascending (those left out are a block's alone)
};

// The same of up to kInlineRows rows as an argument of the first launch, which leaves them in device memory for the others: a copy
// through pinned memory costs the GPU 3.5 us and the host 9.
constexpr int kInlineRows = 64;
struct InlineParams {
  unsigned long long seeds[kInlineRows], draws[kInlineRows];
  float temperature[kInlineRows], top_p[kInlineRows];
  int top_k[kInlineRows], rows[kInlineRows];
  RowParams to;
  int shared;
};
struct NoParams {};      // an argmax alone

__device__ __forceinline__ bool has_threshold(float temperature, int top_k, float top_p, int V, bool& k_on, bool& p_on) {
  k_on = top_k > 0 && top_k < V;
  p_on = top_p < 1.f;
  return temperature > 0.f && (k_on || p_on);
}

// Eight loads a thread of a run of quads, asked for together (a segment of 152 k logits is five: one trip to memory, not one
// after the other), and early: what a kernel has to know before it can use them is fetched meanwhile.
constexpr int kHeldQuads = 8;
template <int THREADS>
__device__ __forceinline__ void ask_quads(const float4* __restrict__ p, int quads, int base, float4 (&v)[kHeldQuads]) {
  const int wave0 = __builtin_amdgcn_readfirstlane(threadIdx.x & ~(kWave - 1));
#pragma unroll
  for (int u = 0; u < kHeldQuads; ++u)
    if (base + u * THREADS + wave0 < quads) v[u] = p[min(base + u * THREADS + (int)threadIdx.x, quads - 1)];
}

// f(4 q, p[q]) for q below `quads`, each by one of the block's THREADS threads in ascending order; v: what ask_quads has for base 0.
template <int THREADS, typename F>
__device__ __forceinline__ void use_quads(const float4* __restrict__ p, int quads, float4 (&v)[kHeldQuads], F f) {
  for (int base = 0; base < quads; base += kHeldQuads * THREADS) {
    if (base > 0) ask_quads<THREADS>(p, quads, base, v);
#pragma unroll
    for (int u = 0; u < kHeldQuads; ++u) {
      const int q = base + u * THREADS + (int)threadIdx.x;
      if (q < quads) f(4 * q, v[u]);
    }
  }
}

// With parameters: for a row with temperature > 0 and no threshold the block also leaves the sum of e^((x - its segment's maximum) /
// temperature) over its segment, from which the sampler has the mass of every segment without a pass of its own over the row.
template <typename P>
__global__ __launch_bounds__(kArgmaxThreads) void argmax_segments_kernel(
    const float* __restrict__ logits, float* __restrict__ part_v, int* __restrict__ part_i, int V, long ld, P params, float* __restrict__ part_mass,
    SharedRows clear) {
  __shared__ float best_v[kArgmaxThreads / kWave];
  __shared__ int best_i[kArgmaxThreads / kWave];
  const int seg = blockIdx.x, r = blockIdx.y;
  const float* row = logits + (size_t)r * ld;
  // segment bounds in whole float4s when the row allows it
  const int per = ((V + kArgmaxSegments - 1) / kArgmaxSegments + 3) & ~3;
  const int begin = seg * per, end = min(V, begin + per);
  float bv = -INFINITY;
  int bi = 0x7fffffff;
  const bool vec = ((reinterpret_cast<uintptr_t>(row) & 15) == 0);
  const int quads = max(0, end - begin) / 4, left = begin + 4 * quads;      // (what is left over: up to three)
  const float4* const row4 = reinterpret_cast<const float4*>(row + begin);
  float4 held[kHeldQuads];
  if (vec) ask_quads<kArgmaxThreads>(row4, quads, 0, held);
  float temperature = 0.f;
  bool thresholds = false;
  if constexpr (!std::is_same_v<P, NoParams>) {
    bool k_on, p_on;
    temperature = params.temperature[r];
    thresholds = has_threshold(temperature, params.top_k[r], params.top_p[r], V, k_on, p_on);
  }
  if constexpr (std::is_same_v<P, InlineParams>) {
    if (seg == 0 && threadIdx.x == 0) {
      const_cast<unsigned long long*>(params.to.seeds)[r] = params.seeds[r];
      const_cast<unsigned long long*>(params.to.draws)[r] = params.draws[r];
      const_cast<float*>(params.to.temperature)[r] = temperature;
      const_cast<float*>(params.to.top_p)[r] = params.top_p[r];
      const_cast<int*>(params.to.top_k)[r] = params.top_k[r];
      if (r < params.shared) const_cast<int*>(params.to.rows)[r] = params.rows[r];
    }
  }
  // scratch of a row with thresholds that later kernels add into, shared out over its blocks
  if (clear.hist32 != nullptr && thresholds) {
    for (int i = blockIdx.x * kArgmaxThreads + threadIdx.x; i < kHistWords; i += kArgmaxSegments * kArgmaxThreads) {
      clear.hist32[(size_t)blockIdx.y * kHistWords + i] = 0u;
      clear.hist64[(size_t)blockIdx.y * kHistWords + i] = 0ull;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      clear.count[blockIdx.y] = 0u;
      clear.level[blockIdx.y].total = 0u;
    }
  }
  if (vec) {
    use_quads<kArgmaxThreads>(row4, quads, held, [&](int at, const float4& v) {
      argmax_take(bv, bi, v.x, begin + at);
      argmax_take(bv, bi, v.y, begin + at + 1);
      argmax_take(bv, bi, v.z, begin + at + 2);
      argmax_take(bv, bi, v.w, begin + at + 3);
    });
    if (left + (int)threadIdx.x < end) argmax_take(bv, bi, row[left + threadIdx.x], left + threadIdx.x);
  } else {
    for (int i = begin + threadIdx.x; i < end; i += kArgmaxThreads) argmax_take(bv, bi, row[i], i);
  }
  wave_best(bv, bi, argmax_take);
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  if (lane == 0) {
    best_v[wave] = bv;
    best_i[wave] = bi;
  }
  __syncthreads();
  for (int w = 0; w < kArgmaxThreads / kWave; ++w) argmax_take(bv, bi, best_v[w], best_i[w]);  // every thread: the segment's
  if (threadIdx.x == 0) {
    part_v[r * kArgmaxSegments + seg] = bv;
    part_i[r * kArgmaxSegments + seg] = bi;
  }
  if (part_mass == nullptr || !(temperature > 0.f) || thresholds) return;      // (with thresholds the sampler sums what it keeps)
  // the segment again: its mass relative to its own maximum
  const float scale = 1.4426950408889634f / temperature;  // e^(y / t) = 2^(y log2 e / t)
  float mass = 0.f;
  const auto add = [&](float x) {
    const float y = (x - bv) * scale;
    if (y == y) mass += __builtin_amdgcn_exp2f(y);  // a NaN (also -inf - -inf of a segment without a number) adds nothing
  };
  if (vec) {
    if (quads > kHeldQuads * kArgmaxThreads) ask_quads<kArgmaxThreads>(row4, quads, 0, held);      // (else still there)
    use_quads<kArgmaxThreads>(row4, quads, held, [&](int, const float4& v) {
      add(v.x);
      add(v.y);
      add(v.z);
      add(v.w);
    });
    if ((int)threadIdx.x == quads % kArgmaxThreads)      // (as if the last, partial four were one more of the walk)
      for (int j = left; j < end; ++j) add(row[j]);
  } else {
    for (int i = begin + threadIdx.x; i < end; i += kArgmaxThreads) add(row[i]);
  }
  mass = wave_sum(mass);
  __syncthreads();  // best_v has been read
  if (lane == 0) best_v[wave] = mass;
  __syncthreads();
  if (threadIdx.x == 0) {
    float total = 0.f;
    for (int w = 0; w < kArgmaxThreads / kWave; ++w) total += best_v[w];
    part_mass[r * kArgmaxSegments + seg] = total;
  }
}

__global__ __launch_bounds__(kWave) void argmax_pick_kernel(const float* __restrict__ part_v,
                                                            const int* __restrict__ part_i,
                                                            int* __restrict__ out,
                                                            float* __restrict__ out_value) {
  const int r = blockIdx.x, lane = threadIdx.x;
  float bv = lane < kArgmaxSegments ? part_v[r * kArgmaxSegments + lane] : -INFINITY;
  int bi = lane < kArgmaxSegments ? part_i[r * kArgmaxSegments + lane] : 0x7fffffff;
  wave_best(bv, bi, argmax_take);
  if (lane == 0) {
    out[r] = (bi == 0x7fffffff) ? 0 : bi;
    if (out_value != nullptr) out_value[r] = bv;
  }
}

// part_v, part_i: scratch of M * tk_argmax_segments() floats and ints.  out_value
// (optional, [M]) receives each row's maximum (-inf if the row holds no number).
TK_API int tk_argmax_segments() { return kArgmaxSegments; }

TK_API int tk_argmax(const float* logits, int* out, float* out_value, float* part_v, int* part_i, int M,
                     int V, long ld, hipStream_t stream) {
  if (M <= 0) return 0;
  if (V <= 0 || M > 65535) return -1;
  argmax_segments_kernel<<<dim3(kArgmaxSegments, M), kArgmaxThreads, 0, stream>>>(logits, part_v, part_i, V, ld, NoParams{}, nullptr, SharedRows{});
  argmax_pick_kernel<<<M, kWave, 0, stream>>>(part_v, part_i, out, out_value);
  return launch_status();
}

// The same two kernels with their scratch in a fixed device array (see no_alloc.h).
// `g_argmax_scratch` names the array for the device compiler; in host code the name is
// only a handle, so the address each GPU gave its copy is looked up once per device
// and the kernels get that pointer.
constexpr int kNoAllocRows = TK_ARGMAX_NO_ALLOC_MAX_ROWS;
constexpr int kMaxDevices = 64;
struct ArgmaxScratch {
  float value[kNoAllocRows * kArgmaxSegments];
  int index[kNoAllocRows * kArgmaxSegments];
};
static __device__ __align__(256) ArgmaxScratch g_argmax_scratch;
static ArgmaxScratch* g_argmax_scratch_ptr[kMaxDevices] = {};
static std::mutex g_argmax_scratch_mutex;

static ArgmaxScratch* argmax_scratch_of_current_device() {
  int device = -1;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= kMaxDevices) return nullptr;
  std::lock_guard<std::mutex> guard(g_argmax_scratch_mutex);
  if (g_argmax_scratch_ptr[device] == nullptr) {
    void* ptr = nullptr;
    if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(g_argmax_scratch)) != hipSuccess || ptr == nullptr) {
      (void)hipGetLastError();
      return nullptr;
    }
    g_argmax_scratch_ptr[device] = static_cast<ArgmaxScratch*>(ptr);
  }
  return g_argmax_scratch_ptr[device];
}

TK_API int tk_argmax_no_alloc_max_rows() { return kNoAllocRows; }

TK_API int tk_argmax_no_alloc(const float* logits, int* out, float* out_value, int M, int V, long ld,
                              hipStream_t stream) {
  if (M <= 0) return 0;
  if (V <= 0 || logits == nullptr || out == nullptr || ld < V) return -1;
  if (M > kNoAllocRows) return -3;
  ArgmaxScratch* scratch = argmax_scratch_of_current_device();
  if (scratch == nullptr) return -4;
  argmax_segments_kernel<<<dim3(kArgmaxSegments, M), kArgmaxThreads, 0, stream>>>(
      logits, scratch->value, scratch->index, V, ld, NoParams{}, nullptr, SharedRows{});
  argmax_pick_kernel<<<M, kWave, 0, stream>>>(scratch->value, scratch->index, out, out_value);
  return launch_status();
}

// ---------------------------------------------------------------------------
// sampling
// ---------------------------------------------------------------------------
// monotone map float -> uint32 (larger float, larger integer)
__device__ __forceinline__ uint32_t ordered(float f) {
  const uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

constexpr uint32_t kOrderedMinusInf = 0x007fffffu;      // ordered(-infinity)

__device__ __forceinline__ float unordered(uint32_t o) {
  const uint32_t u = (o & 0x80000000u) ? (o & 0x7fffffffu) : ~o;
  return __uint_as_float(u);
}

// splitmix64-style mix of (seed, counter) -> uniform in [0, 1)
__device__ __forceinline__ float uniform01(uint64_t seed, uint64_t counter) {
  uint64_t z = seed * 0x9e3779b97f4a7c15ull + (counter + 1) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  z ^= z >> 31;
  return (float)(z >> 40) * (1.0f / 16777216.0f);
}

constexpr int kSampleThreads = 1024;

// Prefix sums of one value per thread over the block, threads in index order; `scan`
// holds an entry a wave.  Returns the sum over the threads before this one;
// `inclusive` is that plus the thread's own value as the scan computed it (so the
// ranges [exclusive, inclusive) of the threads tile [0, total) exactly, also in
// floating point); `total` is the sum over all threads.
template <typename T>
__device__ __forceinline__ T block_scan(T v, T* scan, T& inclusive, T& total) {
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave, waves = blockDim.x / kWave;
  T upto = v;
#pragma unroll
  for (int step = 1; step < kWave; step <<= 1) {
    const T other = __shfl_up(upto, step, kWave);
    if (lane >= step) upto += other;
  }
  __syncthreads();
  if (lane == kWave - 1) scan[wave] = upto;
  __syncthreads();
  T before = 0;                      // of the waves before this one
  total = 0;
  for (int w = 0; w < waves; ++w) {
    if (w == wave) before = total;
    total += scan[w];
  }
  inclusive = before + upto;
  const T left = __shfl_up(inclusive, 1, kWave);     // (a wave's first thread starts where the wave before it ends)
  return lane > 0 ? left : before;
}

// Walking the bins from the highest down: the bin in which the running sum first
// reaches `target` (sum of higher bins < target <= that sum + the bin), and the sum
// of the higher bins.  Every thread gets the result.  `nbins` is 4096 or 1024.
template <typename T>
__device__ __forceinline__ void crossing_bin(const T* hist, int nbins, T target, T* scan, int* found_bin,
                                             T* found_above, int& bin, T& above) {
  const int tid = threadIdx.x, threads = blockDim.x;
  const int per = nbins / threads > 0 ? nbins / threads : 1;
  // thread t owns bins [top - per*t, top - per*t - per + 1], highest first
  T mine = 0;
  const int first = nbins - 1 - tid * per;
  if (first >= 0)
    for (int j = 0; j < per; ++j) mine += hist[first - j];
  T total, upto;
  const T before = block_scan<T>(mine, scan, upto, total);
  if (tid == 0) {  // target beyond everything (rounding): the lowest bin
    *found_bin = 0;
    *found_above = total - hist[0];
  }
  __syncthreads();
  if (first >= 0 && before < target && target <= upto) {
    T run = before;
    for (int j = 0; j < per; ++j) {
      const T h = hist[first - j];
      if (run + h >= target) {
        *found_bin = first - j;
        *found_above = run;
        break;
      }
      run += h;
    }
  }
  __syncthreads();
  bin = *found_bin;
  above = *found_above;
  __syncthreads();
}

// logit / temperature; a NaN is treated as -inf (never kept, never drawn), as the argmax does
__device__ __forceinline__ float scaled(float logit, float inv_t) {
  const float x = logit * inv_t;
  return x == x ? x : -INFINITY;
}

// e^x on the exponential unit (2^(x log2 e)): within some 1e-6 of expf for the exponents that
// count here (0 down to -100), at a tenth of its instructions; a block walks its row alone,
// and 152 k expf a pass were most of a pass's time
__device__ __forceinline__ float exp_unit(float x) { return __builtin_amdgcn_exp2f(x * 1.4426950408889634f); }

// exp(x - max) as a 32.32 fixed-point number: integer sums do not depend on the
// order of addition, so thresholds found from them are the same on every run
__device__ __forceinline__ unsigned long long fixed_mass(float x, float mx) {
  return (unsigned long long)(exp_unit(x - mx) * 4294967296.f);
}

// What the draw counts: the mass of what a row with thresholds keeps, a segment of the argmax pass at a time, is a sum of
// e^(x - max) in fixed point too, so that it does not depend on which blocks form it and in what order: a row draws
// the same token from the same number whatever else is in the step.  As many bits behind the point as V of them leave
// (45 for 151,936): all that is cut off together is less than 2^-26 of the best token's mass up to 512 k tokens, less
// than float32 sums lose.  (32 bits, the thresholds' own, would lose a flat tail's tokens below 2^-32.)
__device__ __forceinline__ float draw_scale(int V) { return ldexpf(1.f, 31 + __clz(V)); }
__device__ __forceinline__ unsigned long long draw_mass(float x, float mx, float scale) {
  return (unsigned long long)(exp_unit(x - mx) * scale);
}

// f(index, value) for every element of a row, each by one thread of the block.  A block reads
// its row alone, so what counts is the bytes it has in flight: 16-byte loads where the row's
// address allows them (a pass over 152 k logits: 14 us instead of 29 and more).
template <typename F>
__device__ __forceinline__ void for_row(const float* __restrict__ row, int V, F f) {
  const int tid = threadIdx.x;
  const int head = min(V, (int)((16 - (reinterpret_cast<uintptr_t>(row) & 15)) & 15) / 4);  // before the first 16-byte boundary
  if (tid < head) f(tid, row[tid]);
  const float4* row4 = reinterpret_cast<const float4*>(row + head);
  const int n4 = (V - head) / 4;
#pragma unroll 8
  for (int i = tid; i < n4; i += kSampleThreads) {
    const float4 v = row4[i];
    const int at = head + 4 * i;
    f(at, v.x);
    f(at + 1, v.y);
    f(at + 2, v.z);
    f(at + 3, v.w);
  }
  const int done = head + 4 * n4;
  if (tid < V - done) f(done + tid, row[done + tid]);
}

// Rows with a threshold, shared between blocks: a row is cut into the segments of the argmax pass, a block each.
//   sample_hist:    the first level's histogram of the whole row (counts, and probability mass if only top-p is asked
//                   for), added into the row's in memory; and the pick of the argmax pass for every row.
//   sample_collect: the values in the bin that holds the threshold, with their segments, into the row's list (in any
//                   order: sums over the list are of integers), and the mass of the bins above it in each segment; with
//                   both thresholds the bins above it are listed too, top-p's may lie there.
// The sampler then starts from the histogram and the list and reads the row again only where the drawn number falls.
// (A block that reads its row alone moves some 45 GB/s.  40 rows of 151,936 logits, 24 of them with thresholds: argmax 6.9, histograms 8.6, lists
// 10.5 and the rest 14.5 us, 54.6 -> 40.6 for the whole with its parameters, which came by a copy of their own: only rows that have a threshold
// get blocks (10.0 us, in two rounds, for the histograms of all), a wave finds the first level's bin from sums of 64 bins (the
// block's search 3.8 us, this 2.2), what cannot be listed is passed over by one comparison, and the rest asks for its
// list and its numbers at once and stops at the level that leaves a few values.)

// A segment of a row as the threads of a block see it: asked for at once, used later (f(value) for every element, each by
// one thread).
struct Segment {
  const float* row;
  int begin, end, quads;
  bool wide;
  float4 held[kHeldQuads];

  __device__ __forceinline__ Segment(const float* __restrict__ row_, int V, int seg) : row(row_) {
    const int per = ((V + kArgmaxSegments - 1) / kArgmaxSegments + 3) & ~3;
    begin = min(V, seg * per);
    end = min(V, begin + per);
    quads = (end - begin) / 4;
    wide = (reinterpret_cast<uintptr_t>(row) & 15) == 0;
    if (wide) ask_quads<kShareThreads>(reinterpret_cast<const float4*>(row + begin), quads, 0, held);
  }

  template <typename F>
  __device__ __forceinline__ void each(F f) {
    if (wide) {
      use_quads<kShareThreads>(reinterpret_cast<const float4*>(row + begin), quads, held, [&](int, const float4& v) {
        f(v.x);
        f(v.y);
        f(v.z);
        f(v.w);
      });
      const int done = begin + 4 * quads;
      if ((int)threadIdx.x < end - done) f(row[done + threadIdx.x]);
    } else {
      for (int i = begin + threadIdx.x; i < end; i += kShareThreads) f(row[i]);
    }
  }
};

// Where the first threshold of a row lies, from its first histograms in LDS (a thread's bins lie side by side).  A block of
// kSampleThreads calls; `scan` an entry a wave, `found` one.
__device__ __forceinline__ FirstLevel first_level(const uint32_t* h32, const unsigned long long* h64, bool k_on, int k, float p_keep,
                                                  unsigned long long* scan, FirstLevel* found) {
  constexpr int PER = kBins / kSampleThreads;
  const int tid = threadIdx.x, low = kBins - PER * (tid + 1);     // this thread's bins [low, low + PER), walked from the top
  uint32_t c[PER], count = 0, upto_c, all_c;
  unsigned long long m[PER], mass = 0;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    c[j] = h32[low + j];
    m[j] = 0;
  }
  if (!k_on) {
#pragma unroll
    for (int j = 0; j < PER; ++j) m[j] = h64[low + j];
  }
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    count += c[j];
    mass += m[j];
  }
  const uint32_t before_c = block_scan<uint32_t>(count, reinterpret_cast<uint32_t*>(scan), upto_c, all_c);
  unsigned long long target = (unsigned long long)k, run = before_c, upto = upto_c, whole;
  if (!k_on) {
    run = block_scan<unsigned long long>(mass, scan, upto, whole);
    // the share of the whole mass that top_p allows (at least one unit)
    const double share = (double)p_keep * (double)whole;
    target = share < 1.0 ? 1ull : (unsigned long long)share;
  }
  if (tid == kSampleThreads - 1 && upto < target) {     // beyond everything (rounding): the lowest bin
    const unsigned long long left = target - (upto - (k_on ? (unsigned long long)c[0] : m[0]));
    *found = {0, (uint32_t)left, left, all_c, c[0]};
  }
  if (run < target && target <= upto) {
    uint32_t seen = before_c;
#pragma unroll
    for (int j = PER - 1; j >= 0; --j) {
      const unsigned long long h = k_on ? (unsigned long long)c[j] : m[j];
      seen += c[j];
      if (run < target && target <= run + h) *found = {low + j, (uint32_t)(target - run), target - run, seen, c[j]};
      run += h;
    }
  }
  __syncthreads();
  return *found;
}

// The sum over the wave of whole numbers, in every lane.
__device__ __forceinline__ uint32_t wave_sum_of(uint32_t v) {
  v += lane_other<0>(v);
  v += lane_other<1>(v);
  v += lane_other<2>(v);
  v += lane_other<3>(v);
  LanePair p = pair16(v);
  p = pair32(p.first + p.second);
  return p.first + p.second;
}

// Walking 64 numbers from the highest place down, a lane each (lane l has place 63 - l): the place at which the running sum first
// reaches `target`, or the lowest one, and the sum above it.
__device__ __forceinline__ int crossing_place(unsigned long long mine, unsigned long long target, unsigned long long& above) {
  const int lane = threadIdx.x & (kWave - 1);
  unsigned long long upto = mine;
#pragma unroll
  for (int step = 1; step < kWave; step <<= 1) {
    const unsigned long long other = __shfl_up(upto, step, kWave);
    if (lane >= step) upto += other;
  }
  const unsigned long long reached = __ballot(target <= upto);
  const int at = reached ? __ffsll(reached) - 1 : kWave - 1;
  above = __shfl(upto - mine, at, kWave);
  return kWave - 1 - at;
}

// The same from a row's histograms in memory, by a wave alone: among the sums of every 64 bins, then among those 64 (two trips to
// memory and no barrier; all bins by the block took 3.8 us).
__device__ __forceinline__ FirstLevel first_level_by_wave(const uint32_t* __restrict__ h32, const unsigned long long* __restrict__ h64, bool k_on,
                                                          int k, float p_keep) {
  const int place = kWave - 1 - (threadIdx.x & (kWave - 1));
  const uint32_t coarse = h32[kBins + place];
  unsigned long long target = (unsigned long long)k, sums = coarse, before;
  if (!k_on) {
    sums = h64[kBins + place];
    unsigned long long whole = sums;
#pragma unroll
    for (int m = 1; m < kWave; m <<= 1) whole += __shfl_xor(whole, m, kWave);
    // the share of the whole mass that top_p allows (at least one unit)
    const double share = (double)p_keep * (double)whole;
    target = share < 1.0 ? 1ull : (unsigned long long)share;
  }
  const int group = crossing_place(sums, target, before);
  const uint32_t c = h32[group * kWave + place];
  unsigned long long inside;
  const int bin = crossing_place(k_on ? (unsigned long long)c : h64[group * kWave + place], target - before, inside);
  // (values at and above the bin: of the groups above it, and of its group)
  const uint32_t seen = wave_sum_of((place > group ? coarse : 0u) + (place >= bin ? c : 0u));
  const unsigned long long left = target - before - inside;
  return {group * kWave + bin, (uint32_t)left, left, seen, __shfl(c, kWave - 1 - bin, kWave)};
}

// The row of a block of the two kernels below, -1 if there is none: the list is the caller's, and a row named twice in a run would be added
// up twice.
__device__ __forceinline__ int shared_row(const int* __restrict__ rows, int M) {
  const int r = rows[blockIdx.y], before = blockIdx.y > 0 ? rows[blockIdx.y - 1] : -1;
  return r > before && r < M ? r : -1;
}

__global__ __launch_bounds__(kShareThreads) void sample_hist_kernel(
    const float* __restrict__ logits, long ld, int M, int V, RowParams params, const float* __restrict__ seg_max, float* __restrict__ row_max,
    SharedRows sh) {
  __shared__ uint32_t h32[kBins];
  __shared__ unsigned long long h64[kBins];
  const int seg = blockIdx.x, r = shared_row(params.rows, M), lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  if (r < 0) return;
  bool k_on, p_on;
  const float temperature = params.temperature[r];
  if (!has_threshold(temperature, params.top_k[r], params.top_p[r], V, k_on, p_on)) return;
  Segment segment(logits + (size_t)r * ld, V, seg);
  // the row's maximum (every wave for itself)
  const float bv = wave_max(lane < kArgmaxSegments ? seg_max[r * kArgmaxSegments + lane] : -INFINITY);
  if (seg == 0 && threadIdx.x == 0) row_max[r] = bv;
  const float inv_t = 1.f / temperature, mx = bv * inv_t;
  if (!(mx > -INFINITY)) return;
  for (int i = threadIdx.x; i < kBins; i += kShareThreads) h32[i] = 0;
  if (!k_on)
    for (int i = threadIdx.x; i < kBins; i += kShareThreads) h64[i] = 0;
  __syncthreads();
  segment.each([&](float logit) {
    const float x = scaled(logit, inv_t);
    const uint32_t bin = ordered(x) >> 20;
    atomicAdd(&h32[bin], 1u);
    if (!k_on) atomicAdd(&h64[bin], fixed_mass(x, mx));
  });
  __syncthreads();
  // a wave 64 neighbouring bins at a time, and their sum (most are empty)
  for (int group = wave; group < kCoarse; group += kShareThreads / kWave) {
    const int i = group * kWave + lane;
    const uint32_t n = h32[i];
    if (__ballot(n != 0) == 0) continue;
    const size_t at = (size_t)r * kHistWords;
    const uint32_t all = wave_sum_of(n);
    if (n != 0) atomicAdd(&sh.hist32[at + i], n);
    if (lane == 0) atomicAdd(&sh.hist32[at + kBins + group], all);
    if (k_on) continue;
    const unsigned long long mass = h64[i];
    unsigned long long sum = mass;
#pragma unroll
    for (int m = 1; m < kWave; m <<= 1) sum += __shfl_xor(sum, m, kWave);
    if (n != 0) atomicAdd(&sh.hist64[at + i], mass);
    if (lane == 0) atomicAdd(&sh.hist64[at + kBins + group], sum);
  }
}

__global__ __launch_bounds__(kShareThreads) void sample_collect_kernel(
    const float* __restrict__ logits, long ld, int M, int V, RowParams params, const float* __restrict__ row_max, SharedRows sh) {
  __shared__ uint32_t kept[kBins];
  __shared__ unsigned long long scan[kShareThreads / kWave];
  __shared__ uint32_t count, first;
  const int seg = blockIdx.x, r = shared_row(params.rows, M);
  if (r < 0) return;
  bool k_on, p_on;
  const float temperature = params.temperature[r], p_keep = params.top_p[r];
  const int k = params.top_k[r];
  if (!has_threshold(temperature, k, p_keep, V, k_on, p_on) || !(row_max[r] > -INFINITY)) return;
  const float inv_t = 1.f / temperature;
  if (threadIdx.x == 0) count = 0;
  Segment segment(logits + (size_t)r * ld, V, seg);
  const FirstLevel level = first_level_by_wave(sh.hist32 + (size_t)r * kHistWords, sh.hist64 + (size_t)r * kHistWords, k_on, k, p_keep);
  if (seg == 0 && threadIdx.x == 0) sh.level[r] = level;
  const int low = level.bin;
  const bool both = k_on && p_on;
  if ((both ? level.total : level.inside) > (uint32_t)kCandidates) return;      // (the sampler walks the row)
  const float mx = row_max[r] * inv_t, scale = draw_scale(V);
  unsigned long long above = 0;
  __syncthreads();
  // this block's values, then side by side into the row's list
  // (what lies below the bin, nearly all, is passed over by one comparison; the lowest bins, where a NaN counts, have none)
  const float least = low > (int)(kOrderedMinusInf >> 20) ? unordered((uint32_t)low << 20) : -INFINITY;
  const bool every = !(least > -INFINITY);
  segment.each([&](float logit) {
    if (!(every || logit * inv_t >= least)) return;
    const float x = scaled(logit, inv_t);
    const uint32_t o = ordered(x);
    const int bin = (int)(o >> 20);
    if (bin == low || (both && bin > low)) {
      const uint32_t at = atomicAdd(&count, 1u);
      if (at < (uint32_t)kBins) kept[at] = o;
      else {                                      // (a segment with more: one by one)
        const uint32_t to = atomicAdd(&sh.count[r], 1u);
        if (to < (uint32_t)kCandidates) {
          sh.cand[(size_t)r * kCandidates + to] = o;
          sh.segment[(size_t)r * kCandidates + to] = (uint8_t)seg;
        }
      }
    } else if (bin > low) {
      above += draw_mass(x, mx, scale);
    }
  });
  unsigned long long upto, whole;
  block_scan<unsigned long long>(above, scan, upto, whole);
  if (threadIdx.x == 0) sh.above[r * kArgmaxSegments + seg] = whole;
  __syncthreads();
  const uint32_t n = min(count, (uint32_t)kBins);
  if (threadIdx.x == 0) first = n ? atomicAdd(&sh.count[r], n) : 0u;
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < n && first + i < (uint32_t)kCandidates; i += kShareThreads) {
    sh.cand[(size_t)r * kCandidates + first + i] = kept[i];
    sh.segment[(size_t)r * kCandidates + first + i] = (uint8_t)seg;
  }
}

// One block per row.
// probs_out (optional, [M, V]) receives the final distribution, for tests.
//
// Both thresholds are found by radix selection over the ordered-integer image of the
// scaled logits: three levels (12, 10 and 10 bits), each filling a histogram in LDS (counts
// for top-k, fixed-point probability mass for top-p) in which the bin that holds the
// threshold is found; the next level looks only at the values of that bin.  A pass over the
// row costs 14 us (one CU reads it alone), so the row is walked as rarely as possible: the
// first pass fills the first level's histogram and tells in which of its bins the threshold
// lies; if the values of that bin and the bins above it are few (up to kCandidates; they
// are, unless the logits are nearly all alike), a second pass copies them into LDS with their segments, and every
// further level of both searches and the segments' masses read those (up to kFew of a bin need no further level: their
// ranks say).  Then the segment that holds the drawn number is walked.  (Without the copies: seven passes and the
// draw's with both thresholds.)  Where shares_rows says so the first pass and the copies are those of sample_hist and
// sample_collect.
__global__ __launch_bounds__(kSampleThreads) void sample_kernel(
    const float* __restrict__ logits, long ld, int V, RowParams params, const float* __restrict__ seg_max, const int* __restrict__ seg_index, const float* __restrict__ seg_mass,
    int* __restrict__ out, float* __restrict__ probs_out, SharedRows shared) {
  __shared__ float upto[kArgmaxSegments];  // the mass of the row's segments up to and with each
  __shared__ unsigned long long hist64[kBins];
  __shared__ uint32_t hist32[kBins];
  __shared__ unsigned long long scan64[kSampleThreads / kWave];
  __shared__ uint32_t cand[kCandidates];  // ordered images of the values that may hold a threshold
  __shared__ uint8_t cand_segment[kCandidates];
  __shared__ FirstLevel first;
  __shared__ uint32_t few[kFew], few_count;
  __shared__ unsigned long long few_mass[kFew];
  __shared__ uint32_t few_cut;
  __shared__ unsigned long long segment_mass[kSampleThreads / kWave][kArgmaxSegments];   // (a copy a wave: its lanes' additions meet nobody else's)
  __shared__ uint32_t cand_count;
  __shared__ int found_bin;
  __shared__ int last_token;
  __shared__ unsigned long long found_above;
  uint32_t* scan32 = reinterpret_cast<uint32_t*>(scan64);
  float* scanf_ = reinterpret_cast<float*>(scan64);

  const int r = blockIdx.x, tid = threadIdx.x, nt = kSampleThreads;
  // the row's maximum and its place from those of its segments, every wave for itself: the token of a greedy row, and of one whose
  // search falls through
  float best = (tid & (kWave - 1)) < kArgmaxSegments ? seg_max[r * kArgmaxSegments + (tid & (kWave - 1))] : -INFINITY;
  int best_at = (tid & (kWave - 1)) < kArgmaxSegments ? seg_index[r * kArgmaxSegments + (tid & (kWave - 1))] : 0x7fffffff;
  wave_best(best, best_at, argmax_take);
  if (tid == 0) out[r] = best_at == 0x7fffffff ? 0 : best_at;
  const float temperature = params.temperature[r];
  if (!(temperature > 0.f)) return;
  // (asked for ahead of their use)
  const float drawn = uniform01(params.seeds[r], params.draws[r]);
  const uint32_t first_cand = shared.hist32 != nullptr ? shared.cand[(size_t)r * kCandidates + tid] : 0u;
  const uint8_t first_segment = shared.hist32 != nullptr ? shared.segment[(size_t)r * kCandidates + tid] : (uint8_t)0;
  FirstLevel made{};
  if (shared.hist32 != nullptr) made = shared.level[r];
  const float* row = logits + (size_t)r * ld;
  const float inv_t = 1.f / temperature;
  const int k = params.top_k[r];
  const float p_keep = params.top_p[r];
  const bool k_on = k > 0 && k < V, p_on = p_keep < 1.f;

  // (temperature > 0 keeps the order; a row without any number has nothing to draw from)
  const float mx = best * inv_t;
  if (!(mx > -INFINITY)) return;

  // First pass: the first level's histogram (counts; probability mass too if only top-p is
  // asked for), the bin of the first threshold to be found, and the candidates.
  uint32_t k_prefix = 0, k_remaining = (uint32_t)max(k, 0);
  uint32_t p_prefix = 0;               // only top-p: its first level is found by the first pass
  unsigned long long p_remaining = 0;
  bool listed = false;                 // what is kept and not in cand has its mass, segment by segment, in shared.above
  bool whole_list = k_on && p_on;      // (all that is kept is in cand)
  const int chunk = ((V + kArgmaxSegments - 1) / kArgmaxSegments + 3) & ~3;      // a segment of the argmax pass
  int ncand = -1;                      // >= 0: cand[0 .. ncand) hold every value that can be a threshold
  if (k_on || p_on) {
    const bool ready = made.total != 0;     // (the row's first pass is done)
    if (tid == 0) cand_count = 0;
    if (!ready) {
      for (int i = tid; i < kBins; i += nt) {
        hist32[i] = 0;
        hist64[i] = 0;
      }
      __syncthreads();
      for_row(row, V, [&](int, float logit) {
        const float x = scaled(logit, inv_t);
        const uint32_t bin = ordered(x) >> 20;
        atomicAdd(&hist32[bin], 1u);
        if (!k_on) atomicAdd(&hist64[bin], fixed_mass(x, mx));
      });
      __syncthreads();
    }
    const FirstLevel level = ready ? made : first_level(hist32, hist64, k_on, k, p_keep, scan64, &first);
    const int low_bin = level.bin;
    if (k_on) {
      k_prefix = (uint32_t)low_bin;
      k_remaining = level.k_remaining;
    } else {
      p_prefix = (uint32_t)low_bin;
      p_remaining = level.p_remaining;
    }
    // the values in that bin and above it; listed: those that may be a threshold (see sample_collect)
    const uint32_t total = level.total, entries = k_on && p_on ? level.total : level.inside;
    if (ready && entries <= (uint32_t)kCandidates) {
      if (tid < (int)entries) {
        cand[tid] = first_cand;
        cand_segment[tid] = first_segment;
      }
#pragma unroll 4
      for (int i = tid + nt; i < (int)entries; i += nt) {
        cand[i] = shared.cand[(size_t)r * kCandidates + i];
        cand_segment[i] = shared.segment[(size_t)r * kCandidates + i];
      }
      ncand = (int)entries;
      listed = true;
    } else if (total <= (uint32_t)kCandidates) {
      for_row(row, V, [&](int i, float logit) {
        const uint32_t o = ordered(scaled(logit, inv_t));
        if ((int)(o >> 20) >= low_bin) {
          const uint32_t at = atomicAdd(&cand_count, 1u);  // (in any order: the sums below are of integers)
          int seg = (int)((float)i * (1.f / (float)chunk));      // (within one of it)
          seg += (long)(seg + 1) * chunk <= i ? 1 : (long)seg * chunk > i ? -1 : 0;
          cand[at] = o;
          cand_segment[at] = (uint8_t)seg;
        }
      });
      ncand = (int)total;
      listed = whole_list = true;
    }
    __syncthreads();
  }
  // f(ordered image, scaled logit) for every value that may still hold a threshold
  const auto each = [&](auto f) {
    if (ncand >= 0) {
      for (int i = tid; i < ncand; i += nt) f(cand[i], unordered(cand[i]));
    } else {
      for_row(row, V, [&](int, float logit) {
        const float x = scaled(logit, inv_t);
        f(ordered(x), x);
      });
    }
  };

  // Among a few values (those of the candidates that `belongs` names, at most kFew) the threshold by ranks: a value is kept
  // iff what lies strictly above it, in numbers or in mass, is less than `target(whole)`; the least kept one.  False if
  // they are more.  (A level of the radix search costs some 2 us whatever it looks at, and there are up to five.)
  const auto among_few = [&](bool masses, auto belongs, auto target, uint32_t& found) {
    if (ncand < 0) return false;
    __syncthreads();      // (the search before this one has been read)
    if (tid == 0) {
      few_count = 0;
      few_cut = 0xffffffffu;
    }
    __syncthreads();
    for (int i = tid; i < ncand; i += nt) {
      const uint32_t o = cand[i];
      if (belongs(o)) {
        const uint32_t at = atomicAdd(&few_count, 1u);
        if (at < (uint32_t)kFew) {
          few[at] = o;
          few_mass[at] = masses ? fixed_mass(unordered(o), mx) : 1ull;
        }
      }
    }
    __syncthreads();
    const int n = (int)few_count;
    if (n > kFew || n == 0) return false;      // (every thread alike)
    for (int v = tid; v < 4 * n; v += kSampleThreads) {      // (four neighbouring threads a value, a quarter of the others each)
      const uint32_t mine = few[v / 4];
      unsigned long long above = 0, whole = 0;
      for (int i = v & 3; i < n; i += 4) {
        const unsigned long long m = few_mass[i];
        whole += m;
        above += few[i] > mine ? m : 0ull;
      }
#pragma unroll
      for (int d = 1; d < 4; d <<= 1) {
        whole += __shfl_xor(whole, d, kWave);
        above += __shfl_xor(above, d, kWave);
      }
      if (above < target(whole)) atomicMin(&few_cut, mine);
    }
    __syncthreads();
    found = few_cut;
    return true;
  };

  // top-k: kth = the k-th largest scaled logit (everything >= it survives)
  uint32_t kth = 0;  // ordered(-inf) is > 0, so 0 keeps everything
  if (k_on && !among_few(false, [&](uint32_t o) { return (o >> 20) == k_prefix; }, [&](unsigned long long) { return (unsigned long long)k_remaining; }, kth)) {
    uint32_t prefix = k_prefix, remaining = k_remaining;
    for (int level = 1; level < 3; ++level) {      // (12 bits are known, ten more each)
      const int shift = level == 1 ? 10 : 0;
      for (int i = tid; i < kLevelBins; i += nt) hist32[i] = 0;
      __syncthreads();
      each([&](uint32_t o, float) {
        if ((o >> (shift + 10)) == prefix) atomicAdd(&hist32[(o >> shift) & (uint32_t)(kLevelBins - 1)], 1u);
      });
      __syncthreads();
      int bin;
      uint32_t above;
      crossing_bin<uint32_t>(hist32, kLevelBins, remaining, scan32, &found_bin,
                             reinterpret_cast<uint32_t*>(&found_above), bin, above);
      remaining -= above;
      prefix = (prefix << 10) | (uint32_t)bin;
      const auto in_bin = [&](uint32_t o) { return (o >> 10) == prefix; };
      if (level == 1 && among_few(false, in_bin, [&](unsigned long long) { return (unsigned long long)remaining; }, prefix)) break;
    }
    kth = prefix;
  }

  // top-p: keep x iff the mass of kept values strictly greater than x is < top_p of
  // the whole; the kept set is {x >= cut}
  uint32_t cut = kth;
  const auto kept_share = [&](unsigned long long whole) {
    const double share = (double)p_keep * (double)whole;
    return share < 1.0 ? 1ull : (unsigned long long)share;
  };
  if (p_on && (k_on ? among_few(true, [&](uint32_t o) { return o >= kth; }, kept_share, cut)
                    : among_few(true, [&](uint32_t o) { return (o >> 20) == p_prefix; }, [&](unsigned long long) { return p_remaining; }, cut))) {
    cut = cut > kth ? cut : kth;
  } else if (p_on) {
    uint32_t prefix = p_prefix;
    unsigned long long remaining = p_remaining;
    for (int level = k_on ? 0 : 1; level < 3; ++level) {  // (without top-k the first pass was the first level)
      const int shift = level == 0 ? 20 : level == 1 ? 10 : 0, nbins = level == 0 ? kBins : kLevelBins;
      for (int i = tid; i < nbins; i += nt) hist64[i] = 0;
      __syncthreads();
      each([&](uint32_t o, float x) {
        const bool in_bin = level == 0 || (o >> (shift + 10)) == prefix;
        if (in_bin && o >= kth) atomicAdd(&hist64[(o >> shift) & (uint32_t)(nbins - 1)], fixed_mass(x, mx));
      });
      __syncthreads();
      if (level == 0) {
        // the whole mass of what top-k keeps (the candidates hold all of it)
        unsigned long long mine = 0, upto, whole;
        for (int i = tid; i < kBins; i += nt) mine += hist64[i];
        block_scan<unsigned long long>(mine, scan64, upto, whole);
        remaining = kept_share(whole);
      }
      int bin;
      unsigned long long above;
      crossing_bin<unsigned long long>(hist64, nbins, remaining, scan64, &found_bin, &found_above, bin, above);
      remaining -= above;
      prefix = (prefix << (level == 0 ? 12 : 10)) | (uint32_t)bin;
      const auto in_bin = [&](uint32_t o) { return (o >> 10) == prefix && o >= kth; };
      if (level == 1 && among_few(true, in_bin, [&](unsigned long long) { return remaining; }, prefix)) break;
    }
    cut = prefix > kth ? prefix : kth;
  }

  // final distribution over {x >= cut}.  The draw walks the tokens in index order: the masses of the row's segments (those
  // of the argmax pass) first, then the segment that holds the target is walked by the whole block.
  // Without a threshold the argmax pass has left their masses (relative to each segment's own maximum); with a list of
  // candidates what is kept is in the list; else a wave sums two segments of the row.
  const int lane = tid & (kWave - 1), wave = tid / kWave;
  const auto kept_mass = [&](float logit) {
    const float x = scaled(logit, inv_t);
    return ordered(x) >= cut ? exp_unit(x - mx) : 0.f;
  };
  const float scale = draw_scale(V);
  __syncthreads();
  if (!k_on && !p_on) {
    if (tid < kArgmaxSegments) {
      const float m = seg_max[r * kArgmaxSegments + tid];
      upto[tid] = m > -INFINITY ? seg_mass[r * kArgmaxSegments + tid] * exp_unit(m * inv_t - mx) : 0.f;
    }
    __syncthreads();
    if (tid == 0)
      for (int w = 1; w < kArgmaxSegments; ++w) upto[w] += upto[w - 1];
  } else {
    for (int i = tid; i < kSampleThreads / kWave * kArgmaxSegments; i += kSampleThreads)
      segment_mass[i / kArgmaxSegments][i % kArgmaxSegments] =
          listed && !whole_list && i < kArgmaxSegments ? shared.above[r * kArgmaxSegments + i] : 0;
    __syncthreads();
    if (listed) {
      for (int i = tid; i < ncand; i += nt)
        if (cand[i] >= cut) atomicAdd(&segment_mass[wave][cand_segment[i]], draw_mass(unordered(cand[i]), mx, scale));
    } else {
      for (int seg = wave; seg < kArgmaxSegments; seg += kSampleThreads / kWave) {
        const int begin = min(V, seg * chunk), end = min(V, begin + chunk);
        unsigned long long mine = 0;
        const auto add = [&](float logit) {
          const float x = scaled(logit, inv_t);
          if (ordered(x) >= cut) mine += draw_mass(x, mx, scale);
        };
        if ((reinterpret_cast<uintptr_t>(row) & 15) == 0) {  // (segments begin at multiples of four tokens)
          const int quads = (end - begin) / 4;
#pragma unroll 8
          for (int q = lane; q < quads; q += kWave) {
            const float4 v = *reinterpret_cast<const float4*>(row + begin + 4 * q);
            add(v.x);
            add(v.y);
            add(v.z);
            add(v.w);
          }
          if (lane < end - begin - 4 * quads) add(row[begin + 4 * quads + lane]);
        } else {
#pragma unroll 8
          for (int i = begin + lane; i < end; i += kWave) add(row[i]);
        }
#pragma unroll
        for (int m = kWave / 2; m >= 1; m >>= 1) mine += __shfl_xor(mine, m, kWave);
        if (lane == 0) segment_mass[0][seg] = mine;
      }
    }
    __syncthreads();
    if (tid < kArgmaxSegments) {
      unsigned long long run = 0;
      for (int w = 0; w < kSampleThreads / kWave; ++w) run += segment_mass[w][tid];
#pragma unroll
      for (int m = 1; m < kArgmaxSegments; m <<= 1) {
        const unsigned long long other = __shfl_up(run, m, kArgmaxSegments);
        if (tid >= m) run += other;
      }
      upto[tid] = (float)run / scale;      // (rounded once: as float32 numbers one after the other small segments beside a large one were lost)
    }
  }
  __syncthreads();
  const float total = upto[kArgmaxSegments - 1];

  if (probs_out) {
    float* po = probs_out + (size_t)r * V;
    for_row(row, V, [&](int i, float logit) {
      const float x = scaled(logit, inv_t);
      po[i] = (ordered(x) >= cut) ? exp_unit(x - mx) / total : 0.f;
    });
  }

  const float target = drawn * total;
  // The chunk that holds the target (every thread finds the same one; the last chunk of
  // the row catches rounding), then all threads walk that chunk: each sums a contiguous
  // run of it, a prefix sum over the block finds the run, and its thread walks it.
  const int last_segment = (V - 1) / chunk;
  const int sel = __ffsll(__ballot(lane >= last_segment || target < upto[min(lane, kArgmaxSegments - 1)])) - 1;
  const float sel_before = sel > 0 ? upto[sel - 1] : 0.f;
  const int s_begin = sel * chunk, s_end = min(V, s_begin + chunk);
  const int run_len = ((s_end - s_begin + kSampleThreads - 1) / kSampleThreads + 3) / 4 * 4;
  const int r_begin = min(s_end, s_begin + tid * run_len), r_end = min(s_end, r_begin + run_len);
  // eight tokens of the run at a time, asked for together; the first eight (all, up to 262 k logits) stay for the second look
  constexpr int kHeld = 8;
  float head[kHeld];
  const auto hold = [&](int from, float (&v)[kHeld]) {
    if ((reinterpret_cast<uintptr_t>(row) & 15) == 0 && from + kHeld <= r_end) {      // (runs begin at multiples of four tokens)
#pragma unroll
      for (int u = 0; u < kHeld; u += 4) {
        const float4 a = *reinterpret_cast<const float4*>(row + from + u);
        v[u] = a.x, v[u + 1] = a.y, v[u + 2] = a.z, v[u + 3] = a.w;
      }
    } else {
#pragma unroll
      for (int u = 0; u < kHeld; ++u) v[u] = from + u < r_end ? row[from + u] : -INFINITY;
    }
  };
  float mine_run = 0.f;
  int last_kept = -1;
  const auto look = [&](int from, const float (&v)[kHeld]) {
#pragma unroll
    for (int u = 0; u < kHeld; ++u)
      if (from + u < r_end) {
        mine_run += kept_mass(v[u]);
        // (a kept token's mass may round to zero; it is kept all the same)
        if (ordered(scaled(v[u], inv_t)) >= cut) last_kept = from + u;
      }
  };
  hold(r_begin, head);
  look(r_begin, head);
  for (int i = r_begin + kHeld; i < r_end; i += kHeld) {
    float more[kHeld];
    hold(i, more);
    look(i, more);
  }
  if (tid == 0) {
    found_bin = -1;   // the token that the target falls on
    last_token = -1;  // the chunk's last kept token
  }
  float incl, chunk_total;
  const float excl = block_scan<float>(mine_run, scanf_, incl, chunk_total);  // (its barriers order the two writes above)
  // (a wave's runs lie in the order of its lanes: the last that keeps a token speaks for it)
  const unsigned long long keeping = __ballot(last_kept >= 0);
  if (keeping != 0 && lane == kWave - 1 - __clzll(keeping)) atomicMax(&last_token, last_kept);
  if (sel_before + excl <= target && target < sel_before + incl) {
    float run = sel_before + excl;
    int pick = -1;
    const auto choose = [&](int from, const float (&v)[kHeld]) {
#pragma unroll
      for (int u = 0; u < kHeld; ++u)
        if (from + u < r_end && ordered(scaled(v[u], inv_t)) >= cut) {
          run += kept_mass(v[u]);
          if (pick < 0 && run > target) pick = from + u;
        }
    };
    choose(r_begin, head);
    for (int i = r_begin + kHeld; i < r_end && pick < 0; i += kHeld) {
      float more[kHeld];
      hold(i, more);
      choose(i, more);
    }
    if (pick < 0) pick = last_kept;  // rounding at the end of the run
    if (pick >= 0) atomicMax(&found_bin, pick);
  }
  __syncthreads();
  // no thread's run held the target (rounding at the chunk's end): the chunk's last kept token
  if (tid == 0) {
    const int chosen = found_bin >= 0 ? found_bin : last_token;
    if (chosen >= 0) out[r] = chosen;
  }
}

// Whether a step's rows with thresholds are shared between blocks: two more kernels (some 8 us, and 0.3 us a row beside its
// bytes) against passes of one block over its row alone, which all rows make side by side.  The line looks at all rows of the step (the
// scratch is theirs), the figures are of steps whose rows all have a threshold: of more rows, few of them with one, sharing would still be
// ahead (one row with top-p 91 us alone, 37 shared, whatever stands beside it).  us with top-k / with top-p
// alone, shared against a block a row: 151,936 logits, 1 row 25 / 37 against 42 / 91, 16 rows 33 / 43 and 44 / 99, 64 rows 59 / 77
// and 60 / 128, 77 rows 66 / 90 and 62 / 131, 140 rows 91 / 123 and 68 / 136; 65,536 logits, 1 row 23 / 28 and 27 / 43, 16
// rows 29 / 37 and 28 / 50, 64 rows 47 / 62 and 31 / 54; 32,003 logits, 1 row 23 / 28 and 21 / 31, 64 rows 47 / 53 and 24 / 36.
constexpr int kSharedVocabulary = 65536;
inline bool shares_rows(int M, int V) { return V >= kSharedVocabulary && M <= (V - kSharedVocabulary / 2) / 1536; }
constexpr size_t kSharedWords = 3 * kHistWords + 2;     // of a row: counts, masses, the list's length

// The same for callers, who need not say which rows have a threshold where none is shared (1 or 0).
TK_API int tk_sample_shares_rows(int M, int V) { return shares_rows(M, V); }

TK_API int tk_sample_scratch_bytes(int M, int V) {
  const long rows = M < 1 ? 0 : M;
  const long parts = rows * kArgmaxSegments * 12 + rows * 4 + 16 + rows * 32;
  return (int)(parts + (shares_rows(M, V) ? rows * ((long)kSharedWords * 4 + (long)kCandidates * 5 + kArgmaxSegments * 8 + (long)sizeof(FirstLevel)) : 0));
}

// Every row's next token: greedy rows (temperature 0) their argmax, the others a draw; a row whose search falls through
// (rounding at an edge) keeps its argmax.  scratch: tk_sample_scratch_bytes(M, V), on a 16-byte border.  params: seeds and draw counts
// (M 64-bit numbers each), temperatures and top-p (M floats each), top-k (M integers) and the numbers of the `shared` rows that
// have a threshold (integers, each once, ascending; the kernels that share such rows are left out where there are none, and a row that is not
// named is sampled by a block alone), one behind the other, on an 8-byte border; in device memory, or (on_host, up to kInlineRows rows)
// in host memory that is free again when the call returns.
TK_API int tk_sample(const float* logits, long ld, int M, int V, const void* params, int on_host, int shared, int* out, float* probs_out,
                     void* scratch, hipStream_t stream) {
  if (M <= 0) return 0;
  if (V <= 0 || M > 65535 || scratch == nullptr || (uintptr_t)scratch % 16 != 0 || params == nullptr || (uintptr_t)params % 8 != 0 ||
      shared < 0 || shared > M || (on_host != 0 && M > kInlineRows))
    return -1;
  const bool share = shares_rows(M, V) && shared != 0;
  unsigned char* at = static_cast<unsigned char*>(scratch);
  SharedRows sh{};
  if (share) {      // (per row: 2 kHistWords words of masses, kHistWords of counts, two of the list's length)
    sh.hist64 = reinterpret_cast<unsigned long long*>(at);
    sh.hist32 = reinterpret_cast<uint32_t*>(at + (size_t)M * kHistWords * 8);
    sh.count = sh.hist32 + (size_t)M * kHistWords;
    sh.above = reinterpret_cast<unsigned long long*>(at + (size_t)M * kSharedWords * 4);
    // (the argmax pass clears a row's words so far; M times an odd number of 8 bytes: still on their border)
    sh.level = reinterpret_cast<FirstLevel*>(at + (size_t)M * (kSharedWords * 4 + kArgmaxSegments * 8));
    at += (size_t)M * (kSharedWords * 4 + kArgmaxSegments * 8 + sizeof(FirstLevel));
    static_assert(sizeof(FirstLevel) % 8 == 0 && kSharedWords % 2 == 0, "what lies behind stays on borders of 8 bytes");
  }
  float* seg_max = reinterpret_cast<float*>(at);
  float* seg_mass = seg_max + (size_t)M * kArgmaxSegments;
  int* seg_index = reinterpret_cast<int*>(seg_mass + (size_t)M * kArgmaxSegments);
  float* row_max = reinterpret_cast<float*>(seg_index + (size_t)M * kArgmaxSegments);
  if (share) {
    sh.cand = reinterpret_cast<uint32_t*>(row_max + M);
    sh.segment = reinterpret_cast<uint8_t*>(sh.cand + (size_t)M * kCandidates);
  }
  const auto laid_out = [M](const void* at) {
    const unsigned long long* seeds = static_cast<const unsigned long long*>(at);
    const float* temperature = reinterpret_cast<const float*>(seeds + 2 * M);
    const int* top_k = reinterpret_cast<const int*>(temperature + 2 * M);
    return RowParams{seeds, seeds + M, temperature, temperature + M, top_k, top_k + M};
  };
  const dim3 all(kArgmaxSegments, M);
  RowParams rows;
  if (on_host) {
    // (behind the scratch of the rest, on its border of 8 bytes)
    unsigned char* const end = static_cast<unsigned char*>(scratch) + tk_sample_scratch_bytes(M, V) - (size_t)M * 32;
    rows = laid_out(reinterpret_cast<void*>((uintptr_t)end & ~(uintptr_t)7));
    InlineParams in;
    const RowParams from = laid_out(params);
    std::memcpy(in.seeds, from.seeds, sizeof(*from.seeds) * M);
    std::memcpy(in.draws, from.draws, sizeof(*from.draws) * M);
    std::memcpy(in.temperature, from.temperature, sizeof(float) * M);
    std::memcpy(in.top_p, from.top_p, sizeof(float) * M);
    std::memcpy(in.top_k, from.top_k, sizeof(int) * M);
    std::memcpy(in.rows, from.rows, sizeof(int) * shared);
    unsigned long long named = 0;
    for (int i = 0; i < shared; ++i) {
      if (in.rows[i] < 0 || in.rows[i] >= M || (share && (named >> in.rows[i] & 1))) return -1;
      named |= 1ull << in.rows[i];
    }
    in.to = rows;
    in.shared = shared;
    argmax_segments_kernel<<<all, kArgmaxThreads, 0, stream>>>(logits, seg_max, seg_index, V, ld, in, seg_mass, sh);
  } else {
    rows = laid_out(params);
    argmax_segments_kernel<<<all, kArgmaxThreads, 0, stream>>>(logits, seg_max, seg_index, V, ld, rows, seg_mass, sh);
  }
  if (share) {
    const dim3 shares(kArgmaxSegments, shared);
    sample_hist_kernel<<<shares, kShareThreads, 0, stream>>>(logits, ld, M, V, rows, seg_max, row_max, sh);
    sample_collect_kernel<<<shares, kShareThreads, 0, stream>>>(logits, ld, M, V, rows, row_max, sh);
  }
  sample_kernel<<<M, kSampleThreads, 0, stream>>>(logits, ld, V, rows, seg_max, seg_index, seg_mass, out, probs_out, sh);
  return launch_status();
}
