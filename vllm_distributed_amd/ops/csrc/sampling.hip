// Sampling on fp32 logits: temperature, top-k, top-p, min-p and the draw itself, with no sort
// and no softmax round trip:
//   * top-k / top-p thresholds are exact keys of the order-preserving integer image of the logits, found by
//     counting (or summing fixed-point weights) per bin: no sort, and no dependence on the order of the lanes;
//   * the draw is Gumbel-argmax (argmax of z_i + g_i, g_i ~ Gumbel(0,1)), which is
//     exactly a sample from softmax(z) restricted to the kept tokens.
// Long vocabularies spread every row over several workgroups (the split kernels below; split_min_v says from which length
// on); shorter rows are walked by one workgroup each.
// Reference behaviour: vllm/v1/sample/sampler.py, ops/topk_topp_sampler.py,
// csrc/sampler.cu (apply_repetition_penalties_).
#include <cfloat>

#include "common.h"

__device__ __forceinline__ uint32_t fkey(float f) {
  const uint32_t b = __float_as_uint(f);
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}

__device__ __forceinline__ uint32_t mix32(uint64_t x) {
  x ^= x >> 33; x *= 0xff51afd7ed558ccdULL; x ^= x >> 33; x *= 0xc4ceb9fe1a85ec53ULL; x ^= x >> 33;
  return (uint32_t)(x >> 16);
}

struct ArgMax { float v; int i; };
__device__ __forceinline__ ArgMax amax2(ArgMax a, ArgMax b) {
  // larger value wins; ties go to the smaller index (matches torch.argmax on unique maxima
  // and makes the result independent of thread scheduling)
  return (b.v > a.v || (b.v == a.v && b.i < a.i)) ? b : a;
}
__device__ __forceinline__ ArgMax block_argmax(ArgMax a, float* rv, int* ri) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    ArgMax b{__shfl_xor(a.v, o, 64), __shfl_xor(a.i, o, 64)};
    a = amax2(a, b);
  }
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
  __syncthreads();
  if (lane == 0) { rv[wid] = a.v; ri[wid] = a.i; }
  __syncthreads();
  ArgMax t = lane < nw ? ArgMax{rv[lane], ri[lane]} : ArgMax{-INFINITY, 0x7fffffff};
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    ArgMax b{__shfl_xor(t.v, o, 64), __shfl_xor(t.i, o, 64)};
    t = amax2(t, b);
  }
  return t;
}

// the token of a row's winner; of a row in which nothing wins (all NaN) the first one, which indexes the next embedding safely
__device__ __forceinline__ long winner(ArgMax a) { return a.i == 0x7fffffff ? 0 : a.i; }

template <typename T>
__global__ __launch_bounds__(1024) void argmax_kernel(const T* __restrict__ logits, long* __restrict__ out, int V,
                                                      long stride) {
  __shared__ float rv[16];
  __shared__ int ri[16];
  const T* row = logits + (long)blockIdx.x * stride;
  ArgMax a{-INFINITY, 0x7fffffff};
  // 16 bytes a load and four loads in flight: with one value a load the row's latency chain is the kernel
  constexpr int W = 16 / sizeof(T);
  typedef T vec_t __attribute__((ext_vector_type(W)));
  int i0 = 0;
  if ((reinterpret_cast<uintptr_t>(row) & 15) == 0) {
    const int nv = V / W;
#pragma unroll 4
    for (int i = threadIdx.x; i < nv; i += 1024) {
      const vec_t v = reinterpret_cast<const vec_t*>(row)[i];
#pragma unroll
      for (int j = 0; j < W; ++j) a = amax2(a, ArgMax{(float)v[j], W * i + j});
    }
    i0 = nv * W;
  }
  for (int i = i0 + threadIdx.x; i < V; i += 1024) a = amax2(a, ArgMax{(float)row[i], i});
  a = block_argmax(a, rv, ri);
  if (threadIdx.x == 0) out[blockIdx.x] = winner(a);
}

// The histogram bin (256 of them, the highest keys in bin 255) in which the running sum from the top reaches
// ``remaining``, and what is left of it there.  Nothing reaches it (rounding): the lowest bin that holds anything,
// with nothing left.  Called by every thread; the first wave works, four bins a lane and a scan over the lanes.
// ``fraction`` >= 0: ``remaining`` is that fraction of the histogram's sum (at least 1).
__device__ __forceinline__ void pick_bin(const unsigned long long* hist, unsigned long long remaining, float fraction,
                                         uint32_t* s_sel, unsigned long long* s_rem) {
  if (threadIdx.x < 64) {
    const int lane = threadIdx.x;                      // lane 0 takes the four highest bins
    unsigned long long w[4], sum = 0ull;
#pragma unroll
    for (int j = 0; j < 4; ++j) { w[j] = hist[255 - 4 * lane - j]; sum += w[j]; }
    unsigned long long cum = sum;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const unsigned long long up = __shfl_up(cum, o, 64);
      if (lane >= o) cum += up;
    }
    const unsigned long long total = __shfl(cum, 63, 64);
    if (fraction >= 0.f) {
      remaining = (unsigned long long)((double)fraction * (double)total);
      if (remaining < 1ull) remaining = 1ull;
    }
    cum -= sum;
    int chosen = -1, lowest = -1;
    unsigned long long rem = 0ull;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (w[j] > 0ull) lowest = 255 - 4 * lane - j;
      if (chosen < 0 && w[j] > 0ull && cum + w[j] >= remaining) { chosen = 255 - 4 * lane - j; rem = remaining - cum; }
      cum += w[j];
    }
    const unsigned long long found = __ballot(chosen >= 0), any = __ballot(lowest >= 0);
    if (found) {
      if (lane == __ffsll(found) - 1) { *s_sel = (uint32_t)chosen; *s_rem = rem; }
    } else if (any) {
      if (lane == 63 - __clzll(any)) { *s_sel = (uint32_t)lowest; *s_rem = 0ull; }
    } else if (lane == 0) {
      *s_sel = 0u; *s_rem = 0ull;
    }
  }
}

// keeps the compiler from folding the operation behind ``v`` into what is done with it.  Several kernels compute a scaled
// logit, its weight, its bin and its noise, each from other registers; what one counts another must find, so every step
// of these is rounded by itself, wherever it is compiled.
// (noconvergent: loops with it can still be unrolled.)
__device__ __forceinline__ float opaque(float v) {
  [[clang::noconvergent]] asm("" : "+v"(v));
  return v;
}
// 1 / temperature
__device__ __forceinline__ float inverse(float t) { return opaque(__builtin_amdgcn_rcpf(t)); }
// exp(z - zmax) as a 32.32 fixed-point number; 0 of a NaN, of which both comparisons are false
// (at most 1: a conversion to 32 bits, which ends at their largest and makes 0 of a NaN, and the one that the largest entry lacks
// then; a conversion to 64 bits is ten instructions)
struct FixedWeight { uint32_t low, largest; };           // their sum
__device__ __forceinline__ FixedWeight weight_parts(float z, float zmax) {
  const float w = __expf(opaque(opaque(z) - zmax)) * 4294967296.f;
  FixedWeight f;
  asm("v_cvt_u32_f32 %0, %1" : "=v"(f.low) : "v"(w));
  f.largest = w >= 4294967296.f ? 1u : 0u;
  return f;
}
__device__ __forceinline__ unsigned long long fixed_weight(float z, float zmax) {
  const FixedWeight f = weight_parts(z, zmax);
  return (unsigned long long)f.low + f.largest;
}

// One radix descent by 1024 threads over n entries; at(i) is entry i's scaled logit.  weight(i) = 1 (COUNT) or exp(z_i - zmax) for
// keys >= floor_key; target = a number of entries (COUNT), a fraction of the total weight (target_w = 0), or the
// weight target_w.  Returns the key u* with  W{key >= u*} >= target  and  W{key > u*} < target.  Weights are
// accumulated as 32.32 fixed-point integers: integer addition does not depend on the order in which the lanes'
// atomics land, so the same logits always give the same threshold (a float histogram could flip the boundary key
// between runs and between ranks that must sample identically).
template <bool COUNT, typename At>
__device__ uint32_t radix_threshold(At at, int n, float zmax, float target, unsigned long long target_w,
                                    uint32_t floor_key, unsigned long long* hist /*[256]*/, uint32_t* s_sel,
                                    unsigned long long* s_rem) {
  uint32_t prefix = 0;
  unsigned long long remaining = COUNT ? (unsigned long long)target : target_w;
  for (int pass = 0; pass < 4; ++pass) {
    const int shift = 24 - 8 * pass;
    for (int b = threadIdx.x; b < 256; b += 1024) hist[b] = 0ull;
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += 1024) {
      const float z = at(i);
      const uint32_t k = fkey(z);
      if (k < floor_key) continue;
      if (pass > 0 && (k >> (shift + 8)) != prefix) continue;
      const unsigned long long w = COUNT ? 1ull : fixed_weight(z, zmax);
      if (w) atomicAdd(&hist[(k >> shift) & 255u], w);
    }
    __syncthreads();
    pick_bin(hist, remaining, !COUNT && pass == 0 && target_w == 0ull ? target : -1.f, s_sel, s_rem);
    __syncthreads();
    prefix = (prefix << 8) | *s_sel;
    remaining = *s_rem;
    __syncthreads();
  }
  return prefix;
}

// z_i + Gumbel noise: the noise is a function of the row's seed and the token alone.  (The logarithms' arguments are at least
// 2^-25, so the bare instruction does.)  The largest word's u rounds to 1, whose noise would be infinite and win whatever the
// logit: one draw in 131 over 128256 tokens was such a token.  It takes the number below 1.
__device__ __forceinline__ float gumbel(float z, uint32_t rnd) {
  const float u = fminf(((float)(rnd >> 8) + 0.5f) * (1.f / 16777216.f), 0x1.fffffep-1f);     // (0, 1)
  const float e = -(__builtin_amdgcn_logf(u) * 0.6931471805599453f);
  return opaque(z) - opaque(__builtin_amdgcn_logf(e) * 0.6931471805599453f);
}
__device__ __forceinline__ uint64_t noise_base(uint64_t seed) { return seed * 0x9E3779B97F4A7C15ULL + 0x632BE59BD9B4E019ULL; }
__device__ __forceinline__ float noisy(float z, uint64_t seed, int i) { return gumbel(z, mix32(noise_base(seed) + (uint64_t)i)); }
// The same for tokens a .. b - 1 between which the upper word of the hash's start does not change (SAME): its part of the hash is
// worked out once, a seventh of the instructions that a token costs.
struct Noise {
  uint64_t base;
  uint32_t lo, hi_shifted, hi_times;
  bool same;
};
__device__ __forceinline__ Noise noise_of(uint64_t seed, int a, int b) {
  Noise n;
  n.base = noise_base(seed);
  const uint64_t first = n.base + (uint64_t)a;
  n.lo = (uint32_t)n.base;
  n.hi_shifted = (uint32_t)(first >> 33);
  n.hi_times = (uint32_t)(first >> 32) * 0xed558ccdu;
  n.same = a < b && (uint32_t)((n.base + (uint64_t)(b - 1)) >> 32) == (uint32_t)(first >> 32);
  return n;
}
template <bool SAME>
__device__ __forceinline__ float noisy(float z, const Noise& n, int i) {
  if (!SAME) return gumbel(z, mix32(n.base + (uint64_t)i));
  const uint32_t lo = (n.lo + (uint32_t)i) ^ n.hi_shifted;               // (mix32's steps, word by word)
  uint64_t x = (uint64_t)lo * 0xed558ccdu + ((uint64_t)(lo * 0xff51afd7u + n.hi_times) << 32);
  x ^= x >> 33; x *= 0xc4ceb9fe1a85ec53ULL; x ^= x >> 33;
  return gumbel(z, (uint32_t)(x >> 16));
}

struct SampleArgs {
  const float* logits;
  long* out;
  const float* temperature;    // null: 1; below 1e-5: greedy
  const int* top_k;            // null or 0: off
  const float* top_p;          // null or 1: off
  const float* min_p;          // null or 0: off
  const long* seeds;
  int V;
  long stride;
  bool late;                   // (several workgroups a row) rows without a filter draw in the second launch
};

// One row by one workgroup of 1024.
__device__ void sample_row(const SampleArgs& p, int rowi, float zmax_known, bool know_max, float* red, float* rv, int* ri,
                           unsigned long long* hist, uint32_t* s_sel, unsigned long long* s_rem) {
  const float* row = p.logits + (long)rowi * p.stride;
  const int V = p.V;
  const float temp = p.temperature ? p.temperature[rowi] : 1.f;
  if (temp < 1e-5f) {
    ArgMax a{-INFINITY, 0x7fffffff};
    for (int i = threadIdx.x; i < V; i += 1024) a = amax2(a, ArgMax{row[i], i});
    a = block_argmax(a, rv, ri);
    if (threadIdx.x == 0) p.out[rowi] = winner(a);
    return;
  }
  const float inv_t = inverse(temp);
  float zmax = zmax_known;
  if (!know_max) {
    float mx = -INFINITY;
    for (int i = threadIdx.x; i < V; i += 1024) mx = fmaxf(mx, row[i] * inv_t);
    zmax = block_max(mx, red);
  }
  auto at = [&](int i) { return row[i] * inv_t; };

  uint32_t thr = 0;   // keep keys >= thr
  const int k = p.top_k ? p.top_k[rowi] : 0;
  const float tp = p.top_p ? p.top_p[rowi] : 1.f;
  const float mp = p.min_p ? p.min_p[rowi] : 0.f;
  if (k > 0 && k < V) thr = radix_threshold<true>(at, V, zmax, (float)k, 0ull, 0u, hist, s_sel, s_rem);
  if (tp < 1.f)      // the fraction of the weight that survived top-k (the descent sums it in its first pass)
    thr = max(thr, radix_threshold<false>(at, V, zmax, tp, 0ull, thr, hist, s_sel, s_rem));
  if (mp > 0.f) thr = max(thr, fkey(zmax + __logf(mp)));

  const uint64_t seed = (uint64_t)(p.seeds ? p.seeds[rowi] : 0);
  ArgMax a{-INFINITY, 0x7fffffff};
  for (int i = threadIdx.x; i < V; i += 1024) {
    const float z = at(i);
    if (fkey(z) >= thr) a = amax2(a, ArgMax{noisy(z, seed, i), i});
  }
  a = block_argmax(a, rv, ri);
  if (threadIdx.x == 0) p.out[rowi] = winner(a);
}

__global__ __launch_bounds__(1024) void sample_kernel(SampleArgs p) {
  __shared__ float red[16];
  __shared__ float rv[16];
  __shared__ int ri[16];
  __shared__ unsigned long long hist[256];
  __shared__ uint32_t s_sel;
  __shared__ unsigned long long s_rem;
  sample_row(p, blockIdx.x, 0.f, false, red, rv, ri, hist, &s_sel, &s_rem);
}

// ---- rows over several workgroups --------------------------------------------------------------------------------
// One workgroup per row spends up to ten passes over 0.5 MB (V = 128256) on one CU, most of the time in LDS atomics that
// all hit the few leading bytes real logits share: 447 us for 61 rows of V = 128256, 73 us for one.  Here a row takes G
// workgroups and three launches:
//   survey   the maximum of a workgroup's share and, from its registers, counts (top-k) or weights (top-p) of what lies below that
//            maximum.  The bins lie on a grid that does not depend on the row, so that the shares' sums can meet in the next launch; shares
//            whose entries lie close together (flat heads, high temperatures) fill a finer grid and from it the coarser ones.
//            Rows without a filter draw here at once, greedy ones take their argmax
//   collect  the bin in which the running sum over the row's bins reaches the target; draws among the entries above it, collects
//            that bin's entries (top-k and top-p together: all entries down to it), and sums the exact weights
//   finish   the exact threshold key among the collected entries, the draw among them, and the row's winner
// The survey's weights are estimates, relative to the top of their bin (the row's maximum is not known yet) and of 2^-16 each.  Where the target
// comes that close to a bin's edge, both bins are collected; and the finish, which has the exact sums, hands a row whose collected bins do not
// hold its threshold to the one-workgroup form, so the result never hangs on the estimate.  A row whose bins overflow a list (thousands of equal
// logits, or of logits within 1 / 128 beside others that are further apart than a finer grid reaches), with NaN under a top-k, or with a maximum
// beyond the grid goes the same way.
// The result is that of the one-workgroup form: the bins are monotone in the key, sums are integers, and each number is rounded alike
// in every kernel (opaque).
// Bound by issue and by trips to memory of a microsecond each: 61 rows, kernel times: 14 where rows without a filter draw (the noise's 64-bit hash
// is 45 issue slots an entry) and 12 where bins are counted, of 8.6 for a read; 19 in the collecting launch for rows of top-p (exact weights 12 slots
// an entry; what is drawn from is brought together 64 entries at a time), 9 in the last.  us a call, with a launch more, in which statistics came
// ahead of bins between the row's extremes -> this: 61 rows of 128256 48 -> 38, one 19 -> 16.5, 256 of 151936 128 -> 104, 148 of 32000 60 -> 35, five
// 26 -> 20.  Normally distributed logits of a standard deviation of 2, 0.3, 0.04 and 0.005, 61 rows of 128256 under a top-p of 0.9: 37, 45, 48.6 and 49.4
// (most entries of the last ones are drawn from), with one grid alone 37, 44, 265 and 262; 256 of 151936 98, 131, 134 and 136.  All bins of a row
// in every workgroup instead of groups first: 42 instead of 38.  One launch for collect and finish, the row's last workgroup finishing it, is no
// way: the fences it needs took it from 20 to 155 us.
constexpr int SPLIT_BINS = 4096;      // a ring in groups of 64: bin b of the grid is at b mod SPLIT_BINS; the row's top SPLIT_GROUPS groups count
constexpr int SPLIT_GROUPS = SPLIT_BINS / 64;          // a lane each
constexpr int SPLIT_LEVELS = 4;       // grids: 128 bins a unit of logit (counts) or of scaled logit (weights, whose 2^-32 is 22.2 units down), then eight for one
// A finer grid is for rows of more than SPLIT_CROWD entries a bin between their ends, and has at most SPLIT_SPREAD bins between them, so that
// the shares' entries lie in the row's ring though the ends are those of a few of the entries.
constexpr float SPLIT_CROWD = 400.f, SPLIT_SPREAD = 1500.f;
constexpr int SPLIT_LIST = 4096;      // collected entries of a row
constexpr int SPLIT_MAX_G = 64;
constexpr int SPLIT_MIN_V = 8192;     // shorter rows: the launches cost more than the one-workgroup form's passes
constexpr int SPLIT_HOLDS = 16;       // entries of a thread that the survey holds at once
// A maximum further from zero than this many bins is not binned.  Counts have to be exact, so bins are whole 32-bit numbers there; weights
// are summed exactly later (a temperature of 1e-4 takes logits of 20 beyond 2^24 bins).
constexpr float SPLIT_FAR = 0x1p30f, SPLIT_FAR_COUNTS = 0x1p23f;
// Without top-k and top-p the one-workgroup form walks a row twice, not ten times, and many rows fill the chip by themselves:
// the launches pay from longer rows on.  Kernel times in us, one workgroup a row / several, draws: 8 x 16384 11.3 / 9.2, 8 x 32000 17.7 / 9.5,
// 64 x 24576 14.8 / 11.3, 256 x 32000 27.7 / 17.4, 600 x 24576 41 / 34, 600 x 50257 95 / 50; with min-p, which takes a launch more: 8 x 16384
// 11.4 / 14, 64 x 32000 21.7 / 20, 256 x 50257 42 / 33, 600 x 32000 51 / 57.  Filtered: 8 x 8192 24.9 / 20, 256 x 8192 26 / 27, 600 x 8192 55 / 54.
static int split_min_v(int S, bool filtered) {
  return filtered ? SPLIT_MIN_V : S <= 32 ? 24576 : S <= 256 ? 40960 : 65536;
}
constexpr int SPLIT_ROWS = 512;       // rows of one set of launches (bounds the workspace)

struct SplitRow {                     // workspace of one row: a word of each of its workgroups
  unsigned long long total[SPLIT_MAX_G], above[SPLIT_MAX_G];      // exact weights: of everything, of what lies above the collected bins
  float part_max[SPLIT_MAX_G];        // in logits (counts) or scaled logits
  float part_v[SPLIT_MAX_G];
  int part_i[SPLIT_MAX_G];
  uint32_t part_n[SPLIT_MAX_G];       // collected entries, also past the list's end
  uint32_t finite[SPLIT_MAX_G];       // entries above -inf (counts), SPLIT_LEVEL times the share's finest grid, SPLIT_NAN
  uint32_t rem, counts, pad[2];       // what is left of a count in the collected bins, where one is left
};
constexpr int SPLIT_GRID = SPLIT_BINS + SPLIT_GROUPS;
struct SplitPart {                    // workspace of one workgroup
  union {
    struct {
      uint32_t grid[SPLIT_GRID];      // bins, and the groups' sums: counts, or weights relative to the group's top as a float
      uint2 list[SPLIT_LIST];         // (key, token)
    };
    uint32_t finer[SPLIT_LEVELS - 1][SPLIT_GRID];      // (in a second one, where its entries lie close together)
  };
};
constexpr uint32_t SPLIT_NAN = 0x80000000u, SPLIT_LEVEL = 0x08000000u, SPLIT_ALONE = 0xffffffffu;
constexpr int SPLIT_RANKED = 256;     // entries that can be ranked at once
constexpr int SPLIT_DIRECT = 96;      // and that are: n of them are n^2 / 8 cycles of LDS reads
struct KeyWeight { uint32_t key; unsigned long long weight; };

enum SplitMode { MODE_NONE, MODE_BOUNDARY, MODE_ALL };
// what a row asks for: a count (k > 0) and / or a weight fraction (tp < 1)
struct SplitFilter {
  float inv_t, tp, mp;
  int k, mode;
  bool greedy;
};
__device__ __forceinline__ SplitFilter split_filter(const SampleArgs& p, int rowi) {
  SplitFilter f;
  const float temp = p.temperature ? p.temperature[rowi] : 1.f;
  f.greedy = temp < 1e-5f;
  f.inv_t = f.greedy ? 1.f : inverse(temp);
  const int k = p.top_k ? p.top_k[rowi] : 0;
  f.k = k > 0 && k < p.V ? k : 0;
  f.tp = p.top_p ? p.top_p[rowi] : 1.f;
  f.mp = p.min_p ? p.min_p[rowi] : 0.f;
  const bool weighs = f.tp < 1.f;
  f.mode = f.k && weighs ? MODE_ALL : (f.k || weighs) ? MODE_BOUNDARY : MODE_NONE;
  return f;
}

// a workgroup's share of the row, read four entries at a time where the row is aligned
struct SplitChunk { int a, b; bool vec; };
__host__ __device__ __forceinline__ int split_share(int V, int G) { return ((V + G - 1) / G + 3) & ~3; }
__device__ __forceinline__ SplitChunk split_chunk(const float* row, int V, int G) {
  const int per = split_share(V, G);
  SplitChunk c;
  c.a = min((int)blockIdx.x * per, V);
  c.b = min(c.a + per, V);
  c.vec = (reinterpret_cast<uintptr_t>(row) & 15) == 0;
  return c;
}
// E entries a thread from ``at`` on, all asked for at once, in rising order; -inf past the share's end
template <bool VEC> __device__ __forceinline__ int split_index(int at, int e) {
  return VEC ? at + 4 * (int)threadIdx.x + 4096 * (e >> 2) + (e & 3) : at + (int)threadIdx.x + 1024 * e;
}
// whether any of the workgroup's entries e is in the share (the same for every thread)
template <bool VEC> __device__ __forceinline__ bool split_any(int at, int e, int end) {
  return (VEC ? at + 4096 * (e >> 2) : at + 1024 * e) < end;
}
template <bool VEC, int E> __device__ __forceinline__ void split_load(const float* row, int at, int end, float (&v)[E]) {
  if (VEC) {
#pragma unroll
    for (int u = 0; u < E / 4; ++u) {
      const int i = split_index<true>(at, 4 * u);
      f32x4 q = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
      if (!split_any<true>(at, 4 * u, end)) {}
      else if (i + 4 <= end) q = *reinterpret_cast<const f32x4*>(row + i);
      else
#pragma unroll
        for (int j = 0; j < 3; ++j)
          if (i + j < end) q[j] = row[i + j];
#pragma unroll
      for (int j = 0; j < 4; ++j) v[4 * u + j] = q[j];
    }
  } else {
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int i = split_index<false>(at, e);
      v[e] = -INFINITY;
      if (split_any<false>(at, e, end) && i < end) v[e] = row[i];
    }
  }
}
// a grid's bins a unit and the width of one: powers of two
__device__ __forceinline__ float split_per(int level) { return __int_as_float((127 + 7 + 3 * level) << 23); }
__device__ __forceinline__ float split_width(int level) { return __int_as_float((127 - 7 - 3 * level) << 23); }
// the bin of x on a grid, a whole number; NaN and infinities stay what they are
__device__ __forceinline__ float split_bin(float x, float per) { return floorf(opaque(x) * per); }
// The finest grid for a share of a row of V, with entries (above -inf) from some mn to mx
__device__ __forceinline__ int split_level(float mx, float mn, int V) {
  const float spread = mx - mn, far = fmaxf(fabsf(mx), fabsf(mn));
  int level = 0;
  while (level < SPLIT_LEVELS - 1 && SPLIT_CROWD * (spread * split_per(level)) < (float)V && spread * split_per(level + 1) <= SPLIT_SPREAD &&
         far * split_per(level + 1) < SPLIT_FAR_COUNTS) ++level;
  return mx == -INFINITY ? SPLIT_LEVELS - 1 : level;     // (no entry)
}

// an inclusive scan over a row of 16 lanes; ``none``: what joins nothing
template <typename T, typename F> __device__ __forceinline__ T row_scan(T v, T none, F join) {
  const auto from = [&](auto ctrl) {
    return __builtin_bit_cast(T, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, none), __builtin_bit_cast(int, v), decltype(ctrl)::value, 0xf, 0xf,
                                                             false));
  };
  using std::integral_constant;
  v = join(v, from(integral_constant<int, 0x111>()));
  v = join(v, from(integral_constant<int, 0x112>()));
  v = join(v, from(integral_constant<int, 0x114>()));
  v = join(v, from(integral_constant<int, 0x118>()));
  return v;
}
// the sum over it, in its last lane
template <typename T> __device__ __forceinline__ T row_sum(T v) { return row_scan(v, T(0), [](T a, T b) { return a + b; }); }
// a thread's sum of weights (below 2^45) added over the wave, in its last lane: 20 bits and the rest
__device__ __forceinline__ unsigned long long wave_weight(unsigned long long w) {
  return ((unsigned long long)scan_add((uint32_t)(w >> 20)) << 20) + scan_add((uint32_t)w & 0xfffffu);
}

// log2 of the weight between two bins, and the weight of a bin ``down`` bins below another
__device__ __forceinline__ float split_unit(int level) { return 1.4426950408889634f * split_width(level); }
__device__ __forceinline__ float split_weight(int down, float unit) { return __builtin_amdgcn_exp2f((float)-down * unit); }

// a thread walks its share in order: the first of equals stays
__device__ __forceinline__ void later(ArgMax& a, float v, int i) {
  if (v > a.v) { a.v = v; a.i = i; }
}

struct SurveyLds {
  float red[16], low[16], rv[16];
  int ri[16];
  uint32_t finite;
  uint4 hist[SPLIT_BINS / 2];         // two copies of each word: lanes that meet in one wait for each other
};
// best entry of a share: the largest (no noise), or with its noise
template <bool VEC, typename F>
__device__ __forceinline__ ArgMax split_best(const float* row, const SplitChunk& c, F value) {
  ArgMax a{-INFINITY, 0x7fffffff};
  float v[SPLIT_HOLDS];
  for (int at = c.a; at < c.b; at += 1024 * SPLIT_HOLDS) {
    split_load<VEC>(row, at, c.b, v);
#pragma unroll
    for (int e = 0; e < SPLIT_HOLDS; ++e) {
      if (!split_any<VEC>(at, e, c.b)) break;
      const int i = split_index<VEC>(at, e);
      later(a, value(v[e], i), i);
    }
  }
  return a;
}
template <bool VEC>
__device__ __forceinline__ void split_survey(const SampleArgs& p, const SplitFilter& f, int rowi, const float* row, const SplitChunk& c,
                                             SplitRow* ws, SplitPart* part, float unit, SurveyLds& s) {
  if (f.greedy || f.mode == MODE_NONE) {
    ArgMax a;
    if (f.greedy || f.mp > 0.f || p.late) a = split_best<VEC>(row, c, [&](float v, int) { return v * f.inv_t; });      // (the maximum, for the floor)
    else {
      const Noise n = noise_of((uint64_t)(p.seeds ? p.seeds[rowi] : 0), c.a, c.b);
      a = n.same ? split_best<VEC>(row, c, [&](float v, int i) { return noisy<true>(v * f.inv_t, n, i); })
                 : split_best<VEC>(row, c, [&](float v, int i) { return noisy<false>(v * f.inv_t, n, i); });
    }
    a = block_argmax(a, s.rv, s.ri);
    if (threadIdx.x == 0) { ws->part_max[blockIdx.x] = a.v; ws->part_v[blockIdx.x] = a.v; ws->part_i[blockIdx.x] = a.i; ws->part_n[blockIdx.x] = 0u; }
    return;
  }
  s.hist[threadIdx.x] = s.hist[threadIdx.x + 1024] = uint4{0u, 0u, 0u, 0u};
  if (threadIdx.x == 0) s.finite = 0u;
  const float scale = f.k ? 1.f : f.inv_t;
  float v[SPLIT_HOLDS], mx = -INFINITY, first = 0.f;
  uint32_t finite = 0u;
  bool nan = false;
  int at = c.a;
  for (;;) {
    split_load<VEC>(row, at, c.b, v);
#pragma unroll
    for (int e = 0; e < SPLIT_HOLDS; ++e) {
      if (!split_any<VEC>(at, e, c.b)) break;
      mx = fmaxf(mx, v[e] * scale);
      if (f.k) {
        finite += v[e] > -INFINITY;
        nan |= v[e] != v[e];
      }
    }
    if (at == c.a) first = v[0];
    if (at + 1024 * SPLIT_HOLDS >= c.b) break;
    at += 1024 * SPLIT_HOLDS;
  }
  const int lane = threadIdx.x & 63;
  mx = all_max(mx);
  // Whether the entries lie close together, as far as one a thread says: a guess is enough, what a ring does not hold lies below what it holds
  first = first > -INFINITY ? first * scale : INFINITY;
  float mn = -INFINITY;
  if (!__any(first < mx - SPLIT_SPREAD * split_width(1))) mn = -all_max(-first);
  if (lane == 0) { s.red[threadIdx.x >> 6] = mx; s.low[threadIdx.x >> 6] = -mn; }
  __syncthreads();
  {
    const float both = row_scan(lane < 16 ? s.red[lane] : s.low[lane & 15], -INFINITY, [](float a, float b) { return fmaxf(a, b); });
    mx = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(both), 15));
    mn = -__int_as_float(__builtin_amdgcn_readlane(__float_as_int(both), 31));
  }
  if (f.k) {
    finite = scan_add(finite);
    const bool any = __any(nan);
    if (lane == 63) atomicAdd(&s.finite, finite);
    if (any && lane == 0) atomicOr(&s.finite, SPLIT_NAN);
  }
  const int finest = split_level(mx, mn, p.V);
  const float per = split_per(finest), top_group = floorf(split_bin(mx, per) * (1.f / 64.f)), width_log = split_unit(finest);
  uint32_t* hist = reinterpret_cast<uint32_t*>(s.hist) + (threadIdx.x & 1);
  for (;;) {                                            // from the entries that are still held backwards
#pragma unroll
    for (int e = 0; e < SPLIT_HOLDS; ++e) {
      if (!split_any<VEC>(at, e, c.b)) break;
      const float x = v[e] * scale, b = split_bin(x, per);
      if (top_group - floorf(b * (1.f / 64.f)) < (float)SPLIT_GROUPS) {
        uint32_t w = 1u;
        if (!f.k) w = (uint32_t)fmaf(__builtin_amdgcn_exp2f((x * per - (b + 1.f)) * width_log), unit, 0.5f);
        atomicAdd(hist + 2 * ((int)b & (SPLIT_BINS - 1)), w);
      }
    }
    if (at == c.a) break;
    at -= 1024 * SPLIT_HOLDS;
    split_load<VEC>(row, at, c.b, v);
  }
  // this grid and, eight bins to one, those before it: the row takes the finest that all its shares have
  int top = mx > -INFINITY ? (int)top_group : 0;
  for (int level = finest;; --level) {
    __syncthreads();
    const uint4 q0 = s.hist[2 * threadIdx.x], q1 = s.hist[2 * threadIdx.x + 1];
    const uint4 h = {q0.x + q0.y, q0.z + q0.w, q1.x + q1.y, q1.z + q1.w};
    uint32_t* grid = level == 0 ? part->grid : part[gridDim.x * gridDim.y].finer[level - 1];
    *reinterpret_cast<uint4*>(grid + 4 * threadIdx.x) = h;
    const int down = 63 - 4 * (threadIdx.x & 15);       // 16 threads a group
    const float u = split_unit(level);
    const uint32_t group = f.k ? row_sum(h.x + h.y + h.z + h.w)
                               : __float_as_uint(row_sum((float)h.x * split_weight(down, u) + (float)h.y * split_weight(down - 1, u) +
                                                         (float)h.z * split_weight(down - 2, u) + (float)h.w * split_weight(down - 3, u)));
    if ((threadIdx.x & 15) == 15) grid[SPLIT_BINS + (threadIdx.x >> 4)] = group;
    if (level == 0) break;
    __syncthreads();
    s.hist[threadIdx.x] = s.hist[threadIdx.x + 1024] = uint4{0u, 0u, 0u, 0u};
    __syncthreads();
    const int bin = 64 * (top - ((top - (int)(threadIdx.x >> 4)) & (SPLIT_GROUPS - 1))) + 4 * (threadIdx.x & 15), to = 7 - (bin & 7);
    const uint32_t sum = f.k ? h.x + h.y + h.z + h.w
                             : (uint32_t)((float)h.x * split_weight(to, u) + (float)h.y * split_weight(to - 1, u) +
                                          (float)h.z * split_weight(to - 2, u) + (float)h.w * split_weight(to - 3, u) + 0.5f);
    if (sum) atomicAdd(hist + 2 * ((bin >> 3) & (SPLIT_BINS - 1)), sum);
    top >>= 3;
  }
  if (threadIdx.x == 0) { ws->part_max[blockIdx.x] = mx; ws->finite[blockIdx.x] = s.finite | (uint32_t)finest * SPLIT_LEVEL; }
}
__global__ __launch_bounds__(1024, 8) void split_survey_kernel(SampleArgs p, SplitRow* ws_rows, SplitPart* ws_parts, int row0, float unit) {
  __shared__ SurveyLds s;
  const int rowi = row0 + blockIdx.y;
  const float* row = p.logits + (long)rowi * p.stride;
  const SplitChunk c = split_chunk(row, p.V, gridDim.x);
  const SplitFilter f = split_filter(p, rowi);
  SplitPart* part = ws_parts + (long)blockIdx.y * gridDim.x + blockIdx.x;
  if (c.vec) split_survey<true>(p, f, rowi, row, c, ws_rows + blockIdx.y, part, unit, s);
  else split_survey<false>(p, f, rowi, row, c, ws_rows + blockIdx.y, part, unit, s);
}

// Where a row is cut: entries of ``draw_from`` and more are drawn from at once, others of ``list_from`` and more (and above -inf) are
// collected.  In logits (counts) or scaled logits: a bin's edges are multiples of its grid's width.
struct SplitCut {
  float draw_from, list_from;
  uint32_t rem, n;                    // counts: what is left of k in the collected bins, the entries that these hold
  bool counts;                        // whether a count cuts among them
};
struct CollectLds {
  float rv[16];
  int ri[16];
  uint32_t n;
  unsigned long long sum[2];
  uint2 queue[16][128];
};

// Where a row's bins reach the target, the same in all of its workgroups and waves: the group by the groups' sums, a lane each, then the bin among
// the group's 64.  (All bins of all shares at once are G^2 histograms a row: as much to read as the logits, 4 us of 61 rows.)
constexpr int SPLIT_ASKED = 8;        // workgroups whose sums are asked for at once
struct SplitSums { uint32_t h[SPLIT_ASKED]; };
__device__ __forceinline__ SplitSums split_sums(const SplitPart* parts, int w0, int G, int word) {
  SplitSums r;
#pragma unroll
  for (int j = 0; j < SPLIT_ASKED; ++j) r.h[j] = (&parts[min(w0 + j, G - 1)].finer[0][0])[word];
  return r;
}
// a lane's word over the workgroups.  A ring's word stands for one of the row's groups if that is not above the workgroup's own highest group
// (``highest``, of the workgroup that is this lane's number).
template <typename F>
__device__ __forceinline__ void split_join(const SplitPart* parts, SplitSums sums, int G, int word, int group, int highest, F add) {
  for (int w = 0;;) {
#pragma unroll
    for (int j = 0; j < SPLIT_ASKED; ++j) {
      const int own = __builtin_amdgcn_readlane(highest, min(w + j, SPLIT_MAX_G - 1));
      add(w + j < G && group <= own ? sums.h[j] : 0u);
    }
    w += SPLIT_ASKED;
    if (w >= G) return;
    sums = split_sums(parts, w, G, word);
  }
}
__device__ __forceinline__ SplitCut split_cut(const SplitFilter& f, const SplitPart* parts, const SplitSums& sums, int G, int highest, int row_top,
                                              uint32_t finite, float margin, int level) {
  const int lane = threadIdx.x & 63, row_group = row_top >> 6, grid = level > 0 ? (level - 1) * SPLIT_GRID : 0;
  const float width = split_width(level), unit = split_unit(level);
  // sums came by word of the ring; from the row's highest group down: lane l takes the word of group row_group - l
  const int word = lane, mine = row_group - ((row_group - word) & (SPLIT_GROUPS - 1));
  const int from = 4 * ((row_group - lane) & (SPLIT_GROUPS - 1));
  const auto edge = [&](int bin) { return (float)bin * width; };
  SplitCut cut{-FLT_MAX, INFINITY, 0u, 0u, false};
  if (f.k) {
    const uint32_t k = (uint32_t)f.k;
    uint32_t count = 0u;
    split_join(parts, sums, G, grid + SPLIT_BINS + word, mine, highest, [&](uint32_t h) { count += h; });
    count = (uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)count);
    const uint32_t cum = scan_add(count), all = last_lane(cum);
    if (k <= all) {
      const int l = __ffsll(__ballot(cum >= k)) - 1, group = row_group - l, at = grid + 64 * (group & (SPLIT_GROUPS - 1)) + 63 - lane;
      const uint32_t before = (uint32_t)__builtin_amdgcn_readlane((int)(cum - count), l);
      uint32_t bin = 0u;
      split_join(parts, split_sums(parts, 0, G, at), G, at, group, highest, [&](uint32_t h) { bin += h; });
      const uint32_t upto = before + scan_add(bin);
      const int b = __ffsll(__ballot(upto >= k)) - 1;
      const uint32_t n = (uint32_t)__builtin_amdgcn_readlane((int)bin, b), above = (uint32_t)__builtin_amdgcn_readlane((int)upto, b) - n;
      cut = SplitCut{edge(64 * group + 64 - b), edge(64 * group + 63 - b), k - above, n, true};
    } else if (k <= finite) {
      cut = SplitCut{edge(64 * (row_group - SPLIT_GROUPS + 1)), -INFINITY, k - all, finite - all, true};
    }
    if (f.mode == MODE_ALL) {          // (a count that keeps every finite entry: the fraction is one of all of them)
      cut.n = !cut.counts ? finite : cut.n + f.k - cut.rem;
      cut.rem = (uint32_t)f.k;
      if (!cut.counts) cut.list_from = -INFINITY;
      cut.draw_from = INFINITY;
    }
  } else {
    float weight = 0.f;
    split_join(parts, sums, G, grid + SPLIT_BINS + word, mine, highest, [&](uint32_t h) { weight += __uint_as_float(h); });
    weight = __int_as_float(__builtin_amdgcn_ds_bpermute(from, __float_as_int(weight)));
    // (relative to the maximum's group's top)
    weight *= split_weight(64 * lane, unit);
    const float cum = scan_add(weight), all = last_lane(cum), target = f.tp * all, off = margin * (float)(1 + level) * all;
    const unsigned long long reached = __ballot(cum + off >= target);
    const int l = reached ? __ffsll(reached) - 1 : 0, group = row_group - l, at = grid + 64 * (group & (SPLIT_GROUPS - 1)) + 63 - lane;
    const float before = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(cum - weight), l));
    float bin = 0.f;
    split_join(parts, split_sums(parts, 0, G, at), G, at, group, highest, [&](uint32_t h) { bin += (float)h; });
    const float upto = before + scan_add(bin * split_weight(64 * l + lane, unit));
    const unsigned long long lo = __ballot(upto + off >= target), hi = __ballot(upto - off >= target);
    // (the target at the group's end: the next group's first bin joins, and the finish has the last word)
    const int b = lo ? __ffsll(lo) - 1 : 63, e = hi ? __ffsll(hi) - 1 : 64;
    // (from 2^23 bins on the next bin is the next number)
    const float at_b = edge(64 * group + 63 - b);
    cut.draw_from = abs(64 * group) < 0x7fffc0 ? edge(64 * group + 64 - b)
                                               : __int_as_float(__float_as_int(at_b) + (at_b > 0.f ? 1 : -1));
    cut.list_from = edge(64 * group + 63 - e);
  }
  return cut;
}

// COUNTS, WEIGHS: which of them cuts the row; neither: every entry is drawn from
template <bool VEC, bool SAME, bool COUNTS, bool WEIGHS>
__device__ __forceinline__ ArgMax split_collect(const SplitFilter& f, const float* row, const SplitChunk& c, float (&v)[8], const Noise& noise,
                                                float zmax, SplitCut cut, SplitPart* part, CollectLds& s) {
  const int lane = threadIdx.x & 63;
  const float floor_z = f.mp > 0.f ? zmax + __logf(f.mp) : -INFINITY;
  const uint32_t floor_key = f.mp > 0.f ? fkey(floor_z) : 0u;
  const float list_from = fmaxf(cut.list_from, -FLT_MAX);
  uint2* queue = s.queue[threadIdx.x >> 6];
  // (the total is one of the weights' lower parts here; their ``largest`` lies among what is drawn from or collected)
  unsigned long long total = 0ull, above = 0ull;
  ArgMax a{-INFINITY, 0x7fffffff};
  int held = 0;                                         // of the wave's queue, below 64 between two entries
  auto draw = [&](int from, int n) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if (lane < n) {
      const uint2 q = queue[from + lane];
      const float z = __uint_as_float(q.x);
      if (WEIGHS) {
        const FixedWeight w = weight_parts(z, zmax);
        above += (unsigned long long)w.low + w.largest;
        total += w.largest;
      }
      if (fkey(z) >= floor_key) a = amax2(a, ArgMax{noisy<SAME>(z, noise, (int)q.y), (int)q.y});
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  };
  for (int at = c.a; at < c.b;) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      if (!split_any<VEC>(at, e, c.b)) break;
      const int i = split_index<VEC>(at, e);
      const float z = v[e] * f.inv_t, x = WEIGHS ? z : v[e];
      if (!COUNTS && !WEIGHS) {
        if (fkey(z) >= floor_key) later(a, noisy<SAME>(z, noise, i), i);
        continue;
      }
      if (WEIGHS) total += weight_parts(z, zmax).low;
      const bool drawn = x >= cut.draw_from && (WEIGHS || z >= floor_z);
      const unsigned long long mask = __ballot(drawn);
      if (mask) {
        if (drawn) queue[held + __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u))] =
            make_uint2(__float_as_uint(z), (uint32_t)i);
        held += __popcll(mask);
        if (held >= 64) {
          held -= 64;
          draw(held, 64);
        }
      }
      if (x >= list_from && x < cut.draw_from) {
        if (WEIGHS) total += weight_parts(z, zmax).largest;
        const uint32_t to = atomicAdd(&s.n, 1u);
        if (to < (uint32_t)SPLIT_LIST) part->list[to] = make_uint2(fkey(z), (uint32_t)i);
      }
    }
    at += 8192;
    if (at < c.b) split_load<VEC>(row, at, c.b, v);
  }
  draw(0, held);
  if (WEIGHS) {
    total = wave_weight(total);
    above = wave_weight(above);
    if (lane == 63) {
      atomicAdd(&s.sum[0], total);
      atomicAdd(&s.sum[1], above);
    }
  }
  return a;
}

// (64 registers, and fewer scalar ones than the 106 that it took by itself, leave a CU its second workgroup)
__global__ __launch_bounds__(1024, 8) void split_collect_kernel(SampleArgs p, SplitRow* ws_rows, SplitPart* ws_parts, int row0, float margin) {
  __shared__ CollectLds s;
  const int rowi = row0 + blockIdx.y, G = gridDim.x, lane = threadIdx.x & 63;
  SplitRow* ws = ws_rows + blockIdx.y;
  const float* row = p.logits + (long)rowi * p.stride;
  const SplitChunk c = split_chunk(row, p.V, G);
  // everything that is wanted first is on its way before anything is known of the row
  float v[8];
  if (c.vec) split_load<true>(row, c.a, c.b, v);
  else split_load<false>(row, c.a, c.b, v);
  const float part_max = lane < G ? ws->part_max[lane] : -INFINITY;
  const uint32_t part_finite = lane < G ? ws->finite[lane] : 0u;
  const SplitPart* parts = ws_parts + (long)blockIdx.y * G;
  SplitSums sums;
  if (p.top_k || p.top_p) sums = split_sums(parts, 0, G, SPLIT_BINS + lane);
  const SplitFilter f = split_filter(p, rowi);
  if (f.greedy || (f.mode == MODE_NONE && !(f.mp > 0.f) && !p.late)) return;
  if (threadIdx.x == 0) { s.n = 0u; s.sum[0] = s.sum[1] = 0ull; }
  const float mx = all_max(part_max), zmax = f.k ? mx * f.inv_t : mx;
  SplitCut cut{-FLT_MAX, INFINITY, 0u, 0u, false};
  bool alone = false;
  if (f.mode != MODE_NONE) {
    const int finest = (int)(part_finite / SPLIT_LEVEL) & 15;
    int level = 0;
    if (!__any(lane < G && finest == 0)) {              // entries close together: the finest grid that all have, and whose ring holds all of them
      level = last_lane(wave_scan(lane < G ? finest : SPLIT_LEVELS - 1, SPLIT_LEVELS - 1, [](int a, int b) { return min(a, b); }));
      const float lowest = -all_max(part_max > -INFINITY ? -part_max : -INFINITY);
      while (level > 0 && (mx - lowest) * split_per(level) > SPLIT_SPREAD) --level;
      if (level > 0) {
        parts += G * gridDim.y;
        sums = split_sums(parts, 0, G, (level - 1) * SPLIT_GRID + SPLIT_BINS + lane);
      }
    }
    const float per = split_per(level), top = split_bin(mx, per);
    alone = !(fabsf(top) < (f.k ? SPLIT_FAR_COUNTS : SPLIT_FAR)) || (f.k && __any((part_finite & SPLIT_NAN) != 0u));
    if (!alone) {
      const uint32_t finite = last_lane(scan_add(part_finite & (SPLIT_LEVEL - 1u)));
      cut = split_cut(f, parts, sums, G, (int)fmaxf(split_bin(part_max, per), -SPLIT_FAR) >> 6, (int)top, finite, margin, level);
      alone = cut.n > (uint32_t)SPLIT_LIST;
    }
  }
  ArgMax a{-INFINITY, 0x7fffffff};
  if (!alone) {
    __syncthreads();                                     // (what thread 0 cleared)
    SplitPart* part = ws_parts + (long)blockIdx.y * G + blockIdx.x;
    const Noise n = noise_of((uint64_t)(p.seeds ? p.seeds[rowi] : 0), c.a, c.b);
#define COLLECT(VEC, SAME)                                                                                       \
    a = f.mode == MODE_NONE ? split_collect<VEC, SAME, false, false>(f, row, c, v, n, zmax, cut, part, s)        \
        : f.k ? split_collect<VEC, SAME, true, false>(f, row, c, v, n, zmax, cut, part, s)                       \
              : split_collect<VEC, SAME, false, true>(f, row, c, v, n, zmax, cut, part, s)
    if (c.vec && n.same) COLLECT(true, true);
    else if (c.vec) COLLECT(true, false);
    else if (n.same) COLLECT(false, true);
    else COLLECT(false, false);
#undef COLLECT
  }
  a = block_argmax(a, s.rv, s.ri);
  if (threadIdx.x == 0) {
    const int w = blockIdx.x;
    ws->part_v[w] = a.v;
    ws->part_i[w] = a.i;
    ws->part_n[w] = alone ? SPLIT_ALONE : s.n;
    ws->total[w] = s.sum[0];
    ws->above[w] = s.sum[1];
    if (w == 0) { ws->rem = cut.rem; ws->counts = cut.counts; }
  }
}

// The same threshold as radix_threshold over a list of SPLIT_RANKED entries at most, in one go: four threads an entry sum what lies
// above it.  The key is the lowest of those above which less than the target lies (0 where there is no weight at all; SPLIT_NOT where
// the list holds less than the target).  at(i): entry i's key and its weight.
constexpr uint32_t SPLIT_NOT = 0xffffffffu;
template <bool COUNT, typename At>
__device__ uint32_t ranked_threshold(At at, int n, unsigned long long target, float fraction, uint32_t floor_key, uint32_t* s_key) {
  const int i = threadIdx.x >> 2;
  if (threadIdx.x == 0) s_key[0] = SPLIT_NOT;
  const KeyWeight mine = i < n ? at(i) : KeyWeight{0u, 0ull};
  unsigned long long above = 0ull, total = 0ull;
  if (i < n) {
#pragma unroll 4
    for (int j = threadIdx.x & 3; j < n; j += 4) {
      const KeyWeight other = at(j);
      const unsigned long long w = COUNT ? 1ull : other.weight;
      above += other.key > mine.key ? w : 0ull;
      if (!COUNT) total += other.key >= floor_key ? w : 0ull;
    }
  }
#pragma unroll
  for (int o = 1; o < 4; o <<= 1) {
    above += __shfl_xor(above, o, 64);
    if (!COUNT) total += __shfl_xor(total, o, 64);
  }
  if (!COUNT && fraction >= 0.f) {
    target = (unsigned long long)((double)fraction * (double)total);
    if (target < 1ull) target = 1ull;
  }
  if (threadIdx.x == 0) s_key[1] = !COUNT && target > total;
  const bool in = i < n && mine.key >= floor_key && above < target && (COUNT || mine.weight > 0ull);
  uint32_t lowest = in ? mine.key : SPLIT_NOT;
#pragma unroll
  for (int o = 4; o < 64; o <<= 1) lowest = min(lowest, (uint32_t)__shfl_xor((int)lowest, o, 64));
  __syncthreads();
  if ((threadIdx.x & 63) == 0 && lowest != SPLIT_NOT) atomicMin(s_key, lowest);
  __syncthreads();
  const uint32_t found = s_key[0], lacks = s_key[1];
  __syncthreads();
  if (!COUNT && fraction < 0.f && lacks) return SPLIT_NOT;
  return found == SPLIT_NOT ? 0u : found;
}

// The same for more entries: a histogram of 1024 bins between the lowest and the highest key, and the one that holds the threshold ranked.
// (The radix descent's four passes of five barriers each: 11.6 us of the launch where this takes 9.)  SPLIT_MANY: that bin holds more than SPLIT_RANKED.
constexpr uint32_t SPLIT_MANY = 0xfffffffeu;
struct RefineLds {
  unsigned long long hist[1024], wave[16], rem;
  KeyWeight few[SPLIT_RANKED];
  uint32_t low, high, bin, n, key[2];
};
template <bool COUNT, typename At>
__device__ uint32_t refined_threshold(At at, int n, unsigned long long target, float fraction, uint32_t floor_key, RefineLds& s) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  s.hist[threadIdx.x] = 0ull;
  if (threadIdx.x == 0) { s.low = 0xffffffffu; s.high = 0u; s.bin = 0xffffffffu; s.n = 0u; }
  __syncthreads();
  uint32_t low = 0xffffffffu, high = 0u;
  for (int i = threadIdx.x; i < n; i += 1024) {
    const uint32_t key = at(i).key;
    if (key < floor_key) continue;
    low = min(low, key);
    high = max(high, key);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    low = min(low, (uint32_t)__shfl_xor((int)low, o, 64));
    high = max(high, (uint32_t)__shfl_xor((int)high, o, 64));
  }
  if (lane == 0) { atomicMin(&s.low, low); atomicMax(&s.high, high); }
  __syncthreads();
  low = s.low;
  high = s.high;
  if (low > high) return 0u;
  const int shift = max(0, 22 - __clz((high - low) | 1u));
  for (int i = threadIdx.x; i < n; i += 1024) {
    const KeyWeight e = at(i);
    if (e.key >= floor_key) atomicAdd(&s.hist[(high - e.key) >> shift], COUNT ? 1ull : e.weight);
  }
  __syncthreads();
  const unsigned long long mine = s.hist[threadIdx.x];
  unsigned long long cum = wave_weight(mine);            // (a bin's sum is below 2^45)
  if (lane == 63) s.wave[wid] = cum;
  __syncthreads();
  unsigned long long total = 0ull;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    if (i < wid) cum += s.wave[i];
    total += s.wave[i];
  }
  if (!COUNT && fraction >= 0.f) {
    target = (unsigned long long)((double)fraction * (double)total);
    if (target < 1ull) target = 1ull;
  }
  if (mine && cum >= target && cum - mine < target) { s.bin = threadIdx.x; s.rem = target - (cum - mine); }
  __syncthreads();
  const uint32_t bin = s.bin;
  if (bin == 0xffffffffu) return !COUNT && fraction < 0.f ? SPLIT_NOT : 0u;
  if (shift == 0) return high - bin;
  for (int i = threadIdx.x; i < n; i += 1024) {
    const KeyWeight e = at(i);
    if (e.key >= floor_key && (high - e.key) >> shift == bin) {
      const uint32_t to = atomicAdd(&s.n, 1u);
      if (to < (uint32_t)SPLIT_RANKED) s.few[to] = e;
    }
  }
  __syncthreads();
  if (s.n > (uint32_t)SPLIT_RANKED) return SPLIT_MANY;
  return ranked_threshold<COUNT>([&](int i) { return s.few[i]; }, (int)s.n, s.rem, -1.f, 0u, s.key);
}

__global__ __launch_bounds__(1024) void split_finish_kernel(SampleArgs p, const SplitRow* ws_rows, const SplitPart* ws_parts, int row0, int G) {
  __shared__ float red[16];
  __shared__ float rv[16];
  __shared__ int ri[16];
  __shared__ RefineLds s;
  __shared__ uint32_t s_sel;
  __shared__ unsigned long long s_rem;
  __shared__ uint2 list[SPLIT_LIST];
  const int rowi = row0 + blockIdx.x, lane = threadIdx.x & 63;
  const SplitRow* ws = ws_rows + blockIdx.x;
  const SplitPart* parts = ws_parts + (long)blockIdx.x * G;
  // everything that may be wanted in one trip (list entries past the counts: nobody's)
  const int each = 1024 / G, from = threadIdx.x / each, slot = threadIdx.x % each;      // of workgroup from's list
  const uint2 entry = parts[min(from, G - 1)].list[slot];
  const bool there = lane < G;
  const float part_max = there ? ws->part_max[lane] : -INFINITY;
  const uint32_t part_n = there ? ws->part_n[lane] : 0u;
  unsigned long long total = there ? ws->total[lane] : 0ull, above = there ? ws->above[lane] : 0ull;
  const uint32_t count_rem = ws->rem;
  const bool counts = ws->counts != 0u;
  ArgMax a{-INFINITY, 0x7fffffff};
  if ((int)threadIdx.x < G) a = ArgMax{ws->part_v[threadIdx.x], ws->part_i[threadIdx.x]};
  const SplitFilter f = split_filter(p, rowi);
  if (!f.greedy && f.mode != MODE_NONE) {
    const float mx = all_max(part_max), zmax = f.k ? mx * f.inv_t : mx;
    const bool all = f.mode == MODE_ALL, weighs = f.tp < 1.f;
    bool alone = __any(part_n > (uint32_t)SPLIT_LIST);
    const uint32_t end = alone ? 0u : scan_add(part_n), n = last_lane(end);
    alone |= n > (uint32_t)SPLIT_LIST;
    unsigned long long target = 1ull;
    if (weighs && !all) {                                // the exact sums say whether the collected bins hold the threshold
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        total += __shfl_xor(total, o, 64);
        above += __shfl_xor(above, o, 64);
      }
      target = (unsigned long long)((double)f.tp * (double)total);
      if (target < 1ull) target = 1ull;
      alone |= !(above < target) || n == 0u;             // (the threshold is among what is drawn from, or nowhere)
      target -= above;
    }
    if (!alone && n > 0u) {
      if (!__any(part_n > (uint32_t)each)) {
        const uint32_t of_n = (uint32_t)__shfl((int)part_n, min(from, 63), 64), of_end = (uint32_t)__shfl((int)end, min(from, 63), 64);
        if (from < G && (uint32_t)slot < of_n) list[of_end - of_n + slot] = entry;
      } else {                                           // longer lists: another trip
        for (uint32_t i = threadIdx.x; i < n; i += 1024) {
          int w = 0;
          uint32_t start = 0u;
          for (int k = 0; k < G; ++k) {
            const uint32_t k_end = (uint32_t)__builtin_amdgcn_readlane((int)end, k);
            if (i >= k_end) { w = k + 1; start = k_end; }
          }
          list[i] = parts[w].list[i - start];
        }
      }
      __syncthreads();
      auto at = [&](int i) {
        const uint32_t key = list[i].x;
        return __uint_as_float((key & 0x80000000u) ? key ^ 0x80000000u : ~key);
      };
      auto counted = [&](int i) { return KeyWeight{list[i].x, 1ull}; };
      auto weighed = [&](int i) { return KeyWeight{list[i].x, fixed_weight(at(i), zmax)}; };
      uint32_t thr = 0u;
      // the list starts with what lies above the cut bin (all) or with that bin
      const float fraction = all ? f.tp : -1.f;
      if (n <= (uint32_t)SPLIT_DIRECT) {
        if (counts) thr = ranked_threshold<true>(counted, (int)n, count_rem, -1.f, 0u, s.key);
        if (weighs) {
          if (threadIdx.x < n) s.few[threadIdx.x] = weighed(threadIdx.x);
          __syncthreads();
          const uint32_t by_weight = ranked_threshold<false>([&](int i) { return s.few[i]; }, (int)n, target, fraction, thr, s.key);
          alone = by_weight == SPLIT_NOT;
          thr = max(thr, by_weight);
        }
      } else {
        if (counts) thr = refined_threshold<true>(counted, (int)n, count_rem, -1.f, 0u, s);
        __syncthreads();
        alone = thr == SPLIT_MANY;
        if (weighs && !alone) {
          const uint32_t by_weight = refined_threshold<false>(weighed, (int)n, target, fraction, thr, s);
          __syncthreads();
          alone = by_weight >= SPLIT_MANY;
          thr = max(thr, by_weight);
        }
      }
      if (!alone) {
        if (f.mp > 0.f) thr = max(thr, fkey(zmax + __logf(f.mp)));
        const uint64_t seed = (uint64_t)(p.seeds ? p.seeds[rowi] : 0);
        for (uint32_t i = threadIdx.x; i < n; i += 1024)
          if (list[i].x >= thr) a = amax2(a, ArgMax{noisy(at((int)i), seed, (int)list[i].y), (int)list[i].y});
      }
    }
    if (alone) {
      sample_row(p, rowi, zmax, true, red, rv, ri, s.hist, &s_sel, &s_rem);
      return;
    }
  }
  a = block_argmax(a, rv, ri);
  if (threadIdx.x == 0) p.out[rowi] = winner(a);
}

// In place: logits masked below the same thresholds the sampler would use (-inf),
// for callers that need the filtered distribution itself (logprobs of the
// processed distribution, rejection sampling).
__global__ __launch_bounds__(1024) void topk_topp_mask_kernel(float* __restrict__ logits,
                                                              const int* __restrict__ top_k,
                                                              const float* __restrict__ top_p,
                                                              const float* __restrict__ min_p, int V, long stride) {
  __shared__ float red[16];
  __shared__ unsigned long long hist[256];
  __shared__ uint32_t s_sel;
  __shared__ unsigned long long s_rem;
  const int rowi = blockIdx.x;
  float* row = logits + (long)rowi * stride;
  float mx = -INFINITY;
  for (int i = threadIdx.x; i < V; i += blockDim.x) mx = fmaxf(mx, row[i]);
  const float zmax = block_max(mx, red);
  uint32_t thr = 0;
  const int k = top_k ? top_k[rowi] : 0;
  const float p = top_p ? top_p[rowi] : 1.f;
  const float mp = min_p ? min_p[rowi] : 0.f;
  auto at = [&](int i) { return row[i]; };
  if (k > 0 && k < V) thr = radix_threshold<true>(at, V, zmax, (float)k, 0ull, 0u, hist, &s_sel, &s_rem);
  if (p < 1.f) thr = max(thr, radix_threshold<false>(at, V, zmax, p, 0ull, thr, hist, &s_sel, &s_rem));
  if (mp > 0.f) thr = max(thr, fkey(zmax + __logf(mp)));
  if (thr == 0) return;
  for (int i = threadIdx.x; i < V; i += blockDim.x)
    if (fkey(row[i]) < thr) row[i] = -INFINITY;
}

// Repetition / frequency / presence penalties on fp32 logits.
// prompt_mask [S, V] (uint8), out_counts [S, V] (int32).
__global__ __launch_bounds__(256) void penalties_kernel(float* __restrict__ logits,
                                                        const uint8_t* __restrict__ prompt_mask,
                                                        const int* __restrict__ out_counts,
                                                        const float* __restrict__ rep, const float* __restrict__ freq,
                                                        const float* __restrict__ pres, int V, long stride) {
  const int rowi = blockIdx.y;
  const float r = rep[rowi], f = freq[rowi], pz = pres[rowi];
  float* row = logits + (long)rowi * stride;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < V; i += gridDim.x * blockDim.x) {
    const int c = out_counts[(long)rowi * V + i];
    const bool seen = c > 0 || prompt_mask[(long)rowi * V + i];
    float x = row[i];
    if (seen) x = x > 0.f ? x / r : x * r;
    x -= f * (float)c;
    if (c > 0) x -= pz;
    row[i] = x;
  }
}

VDA_EXPORT int vda_argmax(const void* logits, long* out, int S, int V, long stride, int dtype, hipStream_t st) {
  if (S == 0) return 0;
  dim3 grid(S), block(1024);
  if (dtype == VDA_F32) hipLaunchKernelGGL(argmax_kernel<float>, grid, block, 0, st, (const float*)logits, out, V, stride);
  else if (dtype == VDA_BF16) hipLaunchKernelGGL(argmax_kernel<bf16_t>, grid, block, 0, st, (const bf16_t*)logits, out, V, stride);
  else if (dtype == VDA_F16) hipLaunchKernelGGL(argmax_kernel<f16_t>, grid, block, 0, st, (const f16_t*)logits, out, V, stride);
  else return -3;
  VDA_CHECK_LAUNCH();
  return 0;
}

// Workgroups of a row: two of 1024 threads per CU and no more (61 rows in nine parts are 549, and the last 37 cost as much as all the
// others), at least a float4 for every thread
static int split_groups(int rows, int V) { return max(1, min(min(SPLIT_ROWS / rows, (V + 4095) / 4096), SPLIT_MAX_G)); }

// bytes of workspace that vda_sample wants for rows of V entries, with top_k or top_p (filtered) or without (0: none)
VDA_EXPORT long vda_sample_workspace(int S, int V, int filtered) {
  if (V < split_min_v(S, filtered)) return 0;
  long parts = 0;
  for (int rows : {min(S, SPLIT_ROWS), S % SPLIT_ROWS})
    if (rows > 0) parts = max(parts, (long)rows * split_groups(rows, V));
  return (long)sizeof(SplitRow) * min(S, SPLIT_ROWS) + (long)sizeof(SplitPart) * (filtered ? 2 : 1) * parts;
}

VDA_EXPORT int vda_sample(const float* logits, long* out, const float* temperature, const int* top_k,
                          const float* top_p, const float* min_p, const long* seeds, int S, int V, long stride,
                          void* workspace, long workspace_bytes, hipStream_t st) {
  if (S == 0) return 0;
  SampleArgs p{logits, out, temperature, top_k, top_p, min_p, seeds, V, stride, false};
  const bool filtered = top_k || top_p;
  if (V < split_min_v(S, filtered)) {
    hipLaunchKernelGGL(sample_kernel, dim3(S), dim3(1024), 0, st, p);
    VDA_CHECK_LAUNCH();
    return 0;
  }
  if (!workspace || workspace_bytes < vda_sample_workspace(S, V, filtered)) return -1;
  SplitRow* ws = (SplitRow*)workspace;
  SplitPart* parts = (SplitPart*)(ws + min(S, SPLIT_ROWS));
  for (int row0 = 0; row0 < S; row0 += SPLIT_ROWS) {
    const int rows = min(S - row0, SPLIT_ROWS), G = split_groups(rows, V);
    int bits = 16;                                       // of a weight: a share's sum fits 32
    while (bits > 0 && (long)split_share(V, G) >> (32 - bits)) --bits;
    const float unit = (float)(1 << bits);
    // With min-p alone its rows need the second launch, and the others join there while the first is a matter of trips only (8 x 32000, all three
    // launches, us: there 14.1, in the first 15.3)
    p.late = !filtered && min_p && split_share(V, G) <= 1024 * SPLIT_HOLDS;
    hipLaunchKernelGGL(split_survey_kernel, dim3(G, rows), dim3(1024), 0, st, p, ws, parts, row0, unit);
    // (the estimate's rounding is half a unit a weight; 2^-32 of every entry and the sums' own are 1e-5 of the total)
    if (filtered || min_p)
      hipLaunchKernelGGL(split_collect_kernel, dim3(G, rows), dim3(1024), 0, st, p, ws, parts, row0, 1.f / unit + 1e-5f);
    hipLaunchKernelGGL(split_finish_kernel, dim3(rows), dim3(1024), 0, st, p, ws, parts, row0, G);
  }
  VDA_CHECK_LAUNCH();
  return 0;
}

VDA_EXPORT int vda_topk_topp_mask(float* logits, const int* top_k, const float* top_p, const float* min_p, int S,
                                  int V, long stride, hipStream_t st) {
  if (S == 0) return 0;
  hipLaunchKernelGGL(topk_topp_mask_kernel, dim3(S), dim3(1024), 0, st, logits, top_k, top_p, min_p, V, stride);
  VDA_CHECK_LAUNCH();
  return 0;
}

VDA_EXPORT int vda_apply_penalties(float* logits, const uint8_t* prompt_mask, const int* out_counts,
                                   const float* rep, const float* freq, const float* pres, int S, int V,
                                   long stride, hipStream_t st) {
  if (S == 0) return 0;
  int gx = (V + 255) / 256;
  if (gx > 64) gx = 64;
  hipLaunchKernelGGL(penalties_kernel, dim3(gx, S), dim3(256), 0, st, logits, prompt_mask, out_counts, rep, freq,
                     pres, V, stride);
  VDA_CHECK_LAUNCH();
  return 0;
}
