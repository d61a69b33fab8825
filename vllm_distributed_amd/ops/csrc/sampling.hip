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
// (at most 1: a conversion to 32 bits and a case for the largest entry; to 64 bits it is ten instructions)
__device__ __forceinline__ unsigned long long fixed_weight(float z, float zmax) {
  const float w = __expf(opaque(opaque(z) - zmax)) * 4294967296.f;
  const uint32_t low = w < 4294967296.f ? (uint32_t)w : 0u;
  return w >= 4294967296.f ? 1ull << 32 : (unsigned long long)low;
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
// workgroups and four launches, 47 us and 15 us (256 rows of 151936 120):
//   stats    the row's maximum and smallest finite value (argmax of a greedy row)
//   bins     counts (top-k) or fixed-point weights (top-p) in SPLIT_BINS bins that are LINEAR between the maximum and the
//            smallest value: neighbouring lanes hit different bins, and a bin holds a few hundred entries
//   collect  draws among the entries above the bin in which the running sum reaches the target, and collects
//            that bin's entries (top-k and top-p together: all entries down to it)
//   finish   the exact threshold key among the collected entries, the draw among them, and the row's winner
// Bound by the noise's 64-bit hash (45 issue slots an entry) where many entries are drawn from, by trips to memory of a
// microsecond each elsewhere.  A fifth and a third less than a form (59 us; 185 for 256 rows of 151936) that let the entries beyond the span meet in
// one bin's atomic (half of the 185), hashed the upper word anew for every entry,
// listed entries with a memory atomic each and always took the radix descent at the end.  Rows without a filter draw in the collecting launch
// alone: half of their entries in the one before gave nothing (61 rows 52.8 / 52.8 us) and cost a single row 2.5 us.  One launch for collect and
// finish, the row's last workgroup finishing it, is no way: the fences it needs took it from 20 to 155 us.
// A row whose bin overflows the list (thousands of equal logits) is done by its finish workgroup alone, the way of the
// short rows.  The result is that of the one-workgroup form: the bins are monotone in the key, sums are integers, and each
// number is rounded alike in every kernel (opaque).
constexpr int SPLIT_BINS = 2048;      // bin 0: the maximum; the last: -inf; the last but one: beyond the span (two per thread)
constexpr int SPLIT_LIST = 4096;      // collected entries of a row
constexpr int SPLIT_MAX_G = 64;
constexpr int SPLIT_MIN_V = 8192;     // shorter rows: the launches cost more than the one-workgroup form's passes
// Without top-k and top-p the one-workgroup form walks a row twice, not ten times, and many rows fill the chip by themselves:
// the launches pay from longer rows on.  Kernel times in us, one workgroup a row / several, draws (greedy rows): 8 x 16384
// 11.9 / 13.0 (5.5 / 8.1), 8 x 32000 19.4 / 13.2 (7.9 / 8.1), 64 x 32000 19.9 / 17.7 (8.1 / 10.2), 256 x 50257 44.7 / 41.9, 600 x 50257
// 82.9 / 99.7 (39.5 / 45.6), 600 x 65536 107 / 106.
static int split_min_v(int S, bool filtered) {
  return filtered ? SPLIT_MIN_V : S <= 32 ? 24576 : S <= 256 ? 40960 : 65536;
}
constexpr int SPLIT_ROWS = 512;       // rows of one set of launches (bounds the workspace)

struct SplitRow {                     // workspace of one row
  unsigned long long hist[SPLIT_BINS];
  uint2 list[SPLIT_LIST];             // (key, token)
  float part_max[SPLIT_MAX_G], part_min[SPLIT_MAX_G], part_v[SPLIT_MAX_G];
  int part_i[SPLIT_MAX_G];
  uint32_t count;                     // of list, also past its end
  uint32_t pad[3];
};

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

// a workgroup's share of the row, walked four entries at a time where the row is aligned
struct SplitChunk { int a, b; bool vec; };
__device__ __forceinline__ SplitChunk split_chunk(const float* row, int V, int G) {
  const int per = ((V + G - 1) / G + 3) & ~3;
  SplitChunk c;
  c.a = min((int)blockIdx.x * per, V);
  c.b = min(c.a + per, V);
  c.vec = (reinterpret_cast<uintptr_t>(row) & 15) == 0;
  return c;
}
// Eight entries a thread are on their way at once; the first of them (``ahead``) since before anything else is known of
// the row: every trip to what another kernel has just written costs about a microsecond.  (Sixteen took the collecting kernel to 86
// registers, which leaves a CU one workgroup of the two that the launch is cut for: 64 rows of 151936 58.5 us, so 50.2; 256 136 / 120.)
constexpr int SPLIT_AHEAD = 2;
struct SplitAhead { f32x4 v[SPLIT_AHEAD]; };
__device__ __forceinline__ SplitAhead split_ahead(const float* row, SplitChunk c, int from) {
  SplitAhead h;
  const int nv = c.a + ((c.b - c.a) & ~3);
#pragma unroll
  for (int u = 0; u < SPLIT_AHEAD; ++u) {
    const int i = from + 4 * (int)threadIdx.x + 4096 * u;
    h.v[u] = c.vec && i < nv ? *reinterpret_cast<const f32x4*>(row + i) : f32x4{0, 0, 0, 0};
  }
  return h;
}
template <typename F>
__device__ __forceinline__ void split_walk(const float* row, SplitChunk c, SplitAhead h, F f) {
  if (c.vec) {
    const int nv = c.a + ((c.b - c.a) & ~3);
    for (int from = c.a; from < nv;) {
#pragma unroll
      for (int u = 0; u < SPLIT_AHEAD; ++u) {
        const int i = from + 4 * (int)threadIdx.x + 4096 * u;
        if (i >= nv) break;
#pragma unroll
        for (int j = 0; j < 4; ++j) f(h.v[u][j], i + j);
      }
      from += 4096 * SPLIT_AHEAD;
      if (from < nv) h = split_ahead(row, c, from);
    }
    for (int i = nv + threadIdx.x; i < c.b; i += 1024) f(row[i], i);
  } else {
    for (int i = c.a + threadIdx.x; i < c.b; i += 1024) f(row[i], i);
  }
}

// the row's maximum and the width of its bins, from the workgroups' partial results; every thread returns the same
struct SplitScale { float zmax, per; };
__device__ __forceinline__ float uniform(float v) { return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v))); }
// (split_parts asks for them)
__device__ __forceinline__ f32x2 split_parts(const SplitRow* ws, int G) {
  const int lane = threadIdx.x & 63;
  return lane < G ? f32x2{ws->part_max[lane], ws->part_min[lane]} : f32x2{-INFINITY, INFINITY};
}
__device__ __forceinline__ SplitScale split_scale(f32x2 parts) {
  float mx = parts[0], mn = parts[1];
  mx = wave_max(mx);
  mn = -wave_max(-mn);
  // weights below 2^-32 of the largest are zero: 22.2; a k-th largest entry further down lands in the last bins
  const float span = fminf(fmaxf(mx - mn, 1e-3f), 24.f);
  return {mx, opaque((float)(SPLIT_BINS - 2) * opaque(__builtin_amdgcn_rcpf(span)))};
}
// functions of the scaled logit that never decrease as it falls
__device__ __forceinline__ float split_place(float z, SplitScale sc) {
  return fmaxf(opaque(opaque(sc.zmax - opaque(z)) * sc.per), 0.f);
}
__device__ __forceinline__ int split_bin(float z, SplitScale sc) {
  if (z == -INFINITY) return SPLIT_BINS - 1;
  return (int)fminf(split_place(z, sc), (float)(SPLIT_BINS - 2));
}

__global__ __launch_bounds__(1024) void split_stats_kernel(SampleArgs p, SplitRow* ws_rows, int row0) {
  __shared__ float red[16];
  __shared__ float rv[16];
  __shared__ int ri[16];
  const int rowi = row0 + blockIdx.y, G = gridDim.x;
  SplitRow* ws = ws_rows + blockIdx.y;
  const float* row = p.logits + (long)rowi * p.stride;
  for (int b = blockIdx.x * 1024 + threadIdx.x; b < SPLIT_BINS; b += G * 1024) ws->hist[b] = 0ull;
  if (blockIdx.x == 0 && threadIdx.x == 0) ws->count = 0u;
  const SplitChunk c = split_chunk(row, p.V, G);
  const SplitAhead ahead = split_ahead(row, c, c.a);
  const SplitFilter f = split_filter(p, rowi);
  if (f.greedy) {
    ArgMax a{-INFINITY, 0x7fffffff};
    split_walk(row, c, ahead, [&](float v, int i) { a = amax2(a, ArgMax{v, i}); });
    a = block_argmax(a, rv, ri);
    if (threadIdx.x == 0) { ws->part_v[blockIdx.x] = a.v; ws->part_i[blockIdx.x] = a.i; }
    return;
  }
  float mx = -INFINITY, mn = INFINITY;
  split_walk(row, c, ahead, [&](float v, int) {
    const float z = v * f.inv_t;
    mx = fmaxf(mx, z);
    if (z > -INFINITY) mn = fminf(mn, z);
  });
  mx = block_max(mx, red);
  mn = -block_max(-mn, red);
  if (threadIdx.x == 0) { ws->part_max[blockIdx.x] = mx; ws->part_min[blockIdx.x] = mn; }
}

// a thread walks its share in order: the first of equals stays
__device__ __forceinline__ void later(ArgMax& a, float v, int i) {
  if (v > a.v) { a.v = v; a.i = i; }
}
// the best of a share's entries that are drawn from without a filter
template <bool SAME>
__device__ __forceinline__ ArgMax split_draw_as(float inv_t, uint32_t floor_key, const float* row, SplitChunk c, const SplitAhead& ahead,
                                                const Noise& n) {
  ArgMax a{-INFINITY, 0x7fffffff};
  if (floor_key) {
    split_walk(row, c, ahead, [&](float v, int i) {
      const float z = v * inv_t;
      if (fkey(z) >= floor_key) later(a, noisy<SAME>(z, n, i), i);
    });
  } else {
    split_walk(row, c, ahead, [&](float v, int i) { later(a, noisy<SAME>(v * inv_t, n, i), i); });
  }
  return a;
}
__device__ __forceinline__ ArgMax split_draw(const SampleArgs& p, const SplitFilter& f, const SplitScale& sc, int rowi, const float* row,
                                             SplitChunk c, const SplitAhead& ahead) {
  const uint32_t floor_key = f.mp > 0.f ? fkey(sc.zmax + __logf(f.mp)) : 0u;
  const Noise n = noise_of((uint64_t)(p.seeds ? p.seeds[rowi] : 0), c.a, c.b);
  return n.same ? split_draw_as<true>(f.inv_t, floor_key, row, c, ahead, n) : split_draw_as<false>(f.inv_t, floor_key, row, c, ahead, n);
}
// Sums in two 32-bit words, each of which 65535 entries cannot overflow: 16 bits of a weight each (the upper one up to 65536,
// and mostly zero).  A 64-bit LDS atomic of a wave costs three times a 32-bit one.
constexpr int SPLIT_SUMMED = 65532;
__global__ __launch_bounds__(1024) void split_bins_kernel(SampleArgs p, SplitRow* ws_rows, int row0) {
  __shared__ uint32_t low[SPLIT_BINS], high[SPLIT_BINS];
  const int rowi = row0 + blockIdx.y;
  SplitRow* ws = ws_rows + blockIdx.y;
  const float* row = p.logits + (long)rowi * p.stride;
  SplitChunk c = split_chunk(row, p.V, gridDim.x);
  SplitAhead ahead = split_ahead(row, c, c.a);
  const f32x2 parts = split_parts(ws, gridDim.x);
  const SplitFilter f = split_filter(p, rowi);
  if (f.greedy || f.mode == MODE_NONE) return;
  const SplitScale sc = split_scale(parts);
  const int end = c.b;
  for (;;) {
#pragma unroll
    for (int b = threadIdx.x; b < SPLIT_BINS; b += 1024) { low[b] = 0u; high[b] = 0u; }
    __syncthreads();
    c.b = min(c.a + SPLIT_SUMMED, end);
    if (f.k) {
      // most of a row far below its maximum, or masked, is one bin: lanes that meet there wait for each other
      uint32_t beyond = 0u, masked = 0u;
      split_walk(row, c, ahead, [&](float v, int) {
        const int b = split_bin(v * f.inv_t, sc);
        beyond += b == SPLIT_BINS - 2;
        masked += b == SPLIT_BINS - 1;
        if (b < SPLIT_BINS - 2) atomicAdd(&low[b], 1u);
      });
      if (beyond) atomicAdd(&low[SPLIT_BINS - 2], beyond);
      if (masked) atomicAdd(&low[SPLIT_BINS - 1], masked);
    } else {
      split_walk(row, c, ahead, [&](float v, int) {
        const float z = v * f.inv_t;
        const unsigned long long w = fixed_weight(z, sc.zmax);
        const int b = split_bin(z, sc);
        const uint32_t lo = (uint32_t)w & 0xffffu, hi = (uint32_t)(w >> 16);
        if (lo) atomicAdd(&low[b], lo);
        if (hi) atomicAdd(&high[b], hi);
      });
    }
    __syncthreads();
#pragma unroll
    for (int b = threadIdx.x; b < SPLIT_BINS; b += 1024) {
      const unsigned long long sum = ((unsigned long long)high[b] << 16) + low[b];
      if (sum) atomicAdd(&ws->hist[b], sum);
    }
    c.a = c.b;
    if (c.a >= end) return;
    ahead = split_ahead(row, SplitChunk{c.a, min(c.a + SPLIT_SUMMED, end), c.vec}, c.a);
    __syncthreads();
  }
}

// Where the running sum over the bins reaches the target: the bin, what is left of the target there, and (counts)
// how many entries it and all before it hold.  bin -1: no weight at all, nothing is filtered.
struct SplitCut { int bin; unsigned long long rem, upto; };
// w: the sums of the two bins that are this thread's.
typedef unsigned long long u64x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ SplitCut split_cut(u64x2 w, const SplitFilter& f, unsigned long long* s_wave /*[16]*/,
                                              SplitCut* s_cut) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  unsigned long long cum = w[0] + w[1];
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const unsigned long long up = __shfl_up(cum, o, 64);
    if (lane >= o) cum += up;
  }
  if (lane == 63) s_wave[wid] = cum;
  if (threadIdx.x == 0) *s_cut = SplitCut{-1, 0ull, 0ull};
  __syncthreads();
  unsigned long long total = 0ull;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    if (i < wid) cum += s_wave[i];
    total += s_wave[i];
  }
  unsigned long long remaining;
  if (f.k) remaining = (unsigned long long)f.k;
  else {
    remaining = (unsigned long long)((double)f.tp * (double)total);
    if (remaining < 1ull) remaining = 1ull;
  }
  const unsigned long long before = cum - w[0] - w[1];
  if (w[0] > 0ull && before < remaining && before + w[0] >= remaining)
    *s_cut = SplitCut{2 * (int)threadIdx.x, remaining - before, before + w[0]};
  else if (w[1] > 0ull && before + w[0] < remaining && cum >= remaining)
    *s_cut = SplitCut{2 * (int)threadIdx.x + 1, remaining - before - w[0], cum};
  __syncthreads();
  return *s_cut;
}

// Rows that one workgroup finishes by itself: counts that say before collecting that the list is too short
// (top-k and top-p together list everything down to the cut, without the -inf entries), and rows of nothing but -inf.
__device__ __forceinline__ bool split_alone(const SplitFilter& f, const SplitCut& cut, const SplitScale& sc) {
  if (sc.zmax == -INFINITY) return true;
  if (f.mode != MODE_ALL) return false;
  const unsigned long long n = cut.bin == SPLIT_BINS - 1 ? (unsigned long long)f.k - cut.rem : cut.upto;
  return n > (unsigned long long)SPLIT_LIST;
}

// The same threshold as radix_threshold over a list of 256 at most, in one go: four threads an entry sum what lies above it.
// The key is the lowest of those above which less than the target lies (0 where there is no weight at all).
template <bool COUNT>
__device__ uint32_t ranked_threshold(const uint2* list, const unsigned long long* weight, int n, unsigned long long target,
                                     float fraction, uint32_t floor_key, uint32_t* s_key) {
  const int i = threadIdx.x >> 2;
  if (threadIdx.x == 0) *s_key = 0xffffffffu;
  const uint32_t key = i < n ? list[i].x : 0u;
  unsigned long long above = 0ull, total = 0ull;
  if (i < n) {
#pragma unroll 4
    for (int j = threadIdx.x & 3; j < n; j += 4) {
      const uint32_t k = list[j].x;
      const unsigned long long w = COUNT ? 1ull : weight[j];
      above += k > key ? w : 0ull;
      if (!COUNT) total += k >= floor_key ? w : 0ull;
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
  const bool in = i < n && key >= floor_key && above < target && (COUNT || weight[i] > 0ull);
  uint32_t lowest = in ? key : 0xffffffffu;
#pragma unroll
  for (int o = 4; o < 64; o <<= 1) lowest = min(lowest, (uint32_t)__shfl_xor((int)lowest, o, 64));
  __syncthreads();
  if ((threadIdx.x & 63) == 0 && lowest != 0xffffffffu) atomicMin(s_key, lowest);
  __syncthreads();
  const uint32_t found = *s_key;
  __syncthreads();
  return found == 0xffffffffu ? 0u : found;
}

__global__ __launch_bounds__(1024) void split_collect_kernel(SampleArgs p, SplitRow* ws_rows, int row0) {
  __shared__ float rv[16];
  __shared__ int ri[16];
  __shared__ unsigned long long s_wave[16];
  __shared__ SplitCut s_cut;
  __shared__ uint32_t s_count, s_base;
  __shared__ uint2 list[SPLIT_LIST];
  const int rowi = row0 + blockIdx.y;
  SplitRow* ws = ws_rows + blockIdx.y;
  const float* row = p.logits + (long)rowi * p.stride;
  const SplitChunk c = split_chunk(row, p.V, gridDim.x);
  const SplitAhead ahead = split_ahead(row, c, c.a);
  const f32x2 parts = split_parts(ws, gridDim.x);
  const u64x2 bin_sum = reinterpret_cast<const u64x2*>(ws->hist)[threadIdx.x];
  const SplitFilter f = split_filter(p, rowi);
  if (f.greedy) return;
  SplitScale sc = split_scale(parts);                     // (64 registers, two workgroups a CU: what is the row's own is in scalar ones)
  sc = SplitScale{uniform(sc.zmax), uniform(sc.per)};
  ArgMax a{-INFINITY, 0x7fffffff};
  if (f.mode == MODE_NONE) {
    a = split_draw(p, f, sc, rowi, row, c, ahead);
  } else {
    if (threadIdx.x == 0) s_count = 0u;
    SplitCut cut = split_cut(bin_sum, f, s_wave, &s_cut);
    cut.bin = __builtin_amdgcn_readfirstlane(cut.bin);
    const bool all = f.mode == MODE_ALL;
    // a count that reaches the -inf entries keeps every other one: none of them needs to be listed
    const bool keeps_all = cut.bin < 0 || cut.bin == SPLIT_BINS - 1;
    // Bins below draw_to are drawn from here, bins list_from .. list_to are collected: in places between bins, as split_bin has
    // them ahead of its rounding down (-inf entries and those beyond the span share the place at infinity)
    const float draw_to = all ? 0.f : keeps_all ? INFINITY : (float)cut.bin;
    const float list_from = all ? 0.f : keeps_all ? NAN : (float)cut.bin;
    const bool beyond = cut.bin >= SPLIT_BINS - 2;
    const float list_end = beyond ? INFINITY : (float)(cut.bin + 1);
    const uint32_t floor_key = f.mp > 0.f ? fkey(sc.zmax + __logf(f.mp)) : 0u;
    const Noise noise = noise_of((uint64_t)(p.seeds ? p.seeds[rowi] : 0), c.a, c.b);
    auto walk = [&](auto same) {
      split_walk(row, c, ahead, [&](float v, int i) {
        const float z = v * f.inv_t, at = split_place(z, sc);
        if (at < draw_to) {
          if (!floor_key || fkey(z) >= floor_key) later(a, noisy<decltype(same)::value>(z, noise, i), i);
        } else if (at >= list_from && (at < list_end || (beyond && z != -INFINITY))) {
          const uint32_t to = atomicAdd(&s_count, 1u);
          if (to < (uint32_t)SPLIT_LIST) list[to] = make_uint2(fkey(z), (uint32_t)i);
        }
      });
    };
    if (!split_alone(f, cut, sc)) {
      if (noise.same) walk(std::true_type());
      else walk(std::false_type());
      // this share's entries behind those of others: one atomic on the row's count
      __syncthreads();
      const uint32_t n = s_count;
      if (n > 0u) {
        if (threadIdx.x == 0) s_base = atomicAdd(&ws->count, n);
        __syncthreads();
        const uint32_t base = s_base;
        for (uint32_t i = threadIdx.x; i < n && base + i < (uint32_t)SPLIT_LIST; i += 1024) ws->list[base + i] = list[i];
      }
    }
  }
  a = block_argmax(a, rv, ri);
  if (threadIdx.x == 0) { ws->part_v[blockIdx.x] = a.v; ws->part_i[blockIdx.x] = a.i; }
}

constexpr int SPLIT_RANKED = 256;     // entries; more take the radix descent (its LDS histogram holds the weights of these)
__global__ __launch_bounds__(1024) void split_finish_kernel(SampleArgs p, SplitRow* ws_rows, int row0, int G) {
  __shared__ float red[16];
  __shared__ float rv[16];
  __shared__ int ri[16];
  __shared__ unsigned long long hist[256];
  __shared__ uint32_t s_sel;
  __shared__ unsigned long long s_rem, s_wave[16];
  __shared__ SplitCut s_cut;
  __shared__ uint2 list[SPLIT_LIST];
  const int rowi = row0 + blockIdx.x;
  SplitRow* ws = ws_rows + blockIdx.x;
  // everything that may be wanted in one trip (list entries past the count: nobody's)
  const f32x2 parts = split_parts(ws, G);
  const u64x2 bin_sum = reinterpret_cast<const u64x2*>(ws->hist)[threadIdx.x];
  const uint2 entry = ws->list[threadIdx.x];
  const uint32_t n = ws->count;
  ArgMax a{-INFINITY, 0x7fffffff};
  if ((int)threadIdx.x < G) a = ArgMax{ws->part_v[threadIdx.x], ws->part_i[threadIdx.x]};
  const SplitFilter f = split_filter(p, rowi);
  if (!f.greedy) {
    const SplitScale sc = split_scale(parts);
    SplitCut cut{-1, 0ull, 0ull};
    if (f.mode != MODE_NONE) cut = split_cut(bin_sum, f, s_wave, &s_cut);
    const bool all = f.mode == MODE_ALL;
    if (n > (uint32_t)SPLIT_LIST || split_alone(f, cut, sc)) {
      sample_row(p, rowi, sc.zmax, true, red, rv, ri, hist, &s_sel, &s_rem);
      return;
    }
    if (n > 0u) {
      list[threadIdx.x] = entry;
      for (uint32_t i = threadIdx.x + 1024; i < n; i += 1024) list[i] = ws->list[i];
      __syncthreads();
      auto at = [&](int i) {
        const uint32_t key = list[i].x;
        return __uint_as_float((key & 0x80000000u) ? key ^ 0x80000000u : ~key);
      };
      uint32_t thr = 0;
      // the list starts with what lies above the cut bin (all) or with that bin
      const bool counts = f.k && cut.bin != SPLIT_BINS - 1, weighs = f.tp < 1.f;
      if (n <= (uint32_t)SPLIT_RANKED) {
        if (weighs && threadIdx.x < n) hist[threadIdx.x] = fixed_weight(at(threadIdx.x), sc.zmax);
        __syncthreads();
        if (counts) thr = ranked_threshold<true>(list, hist, (int)n, all ? (unsigned long long)f.k : cut.rem, -1.f, 0u, &s_sel);
        if (weighs) thr = max(thr, ranked_threshold<false>(list, hist, (int)n, cut.rem, all ? f.tp : -1.f, thr, &s_sel));
      } else {
        if (counts) thr = radix_threshold<true>(at, (int)n, sc.zmax, all ? (float)f.k : (float)cut.rem, 0ull, 0u, hist, &s_sel, &s_rem);
        if (weighs)
          thr = max(thr, radix_threshold<false>(at, (int)n, sc.zmax, f.tp, all ? 0ull : cut.rem, thr, hist, &s_sel, &s_rem));
      }
      if (f.mp > 0.f) thr = max(thr, fkey(sc.zmax + __logf(f.mp)));
      const uint64_t seed = (uint64_t)(p.seeds ? p.seeds[rowi] : 0);
      for (uint32_t i = threadIdx.x; i < n; i += 1024)
        if (list[i].x >= thr) a = amax2(a, ArgMax{noisy(at((int)i), seed, (int)list[i].y), (int)list[i].y});
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

// bytes of workspace that vda_sample wants for rows of V entries, with top_k or top_p (filtered) or without (0: none)
VDA_EXPORT long vda_sample_workspace(int S, int V, int filtered) {
  return V < split_min_v(S, filtered) ? 0 : (long)sizeof(SplitRow) * (S < SPLIT_ROWS ? S : SPLIT_ROWS);
}

VDA_EXPORT int vda_sample(const float* logits, long* out, const float* temperature, const int* top_k,
                          const float* top_p, const float* min_p, const long* seeds, int S, int V, long stride,
                          void* workspace, long workspace_bytes, hipStream_t st) {
  if (S == 0) return 0;
  const SampleArgs p{logits, out, temperature, top_k, top_p, min_p, seeds, V, stride};
  const bool filtered = top_k || top_p;
  if (V < split_min_v(S, filtered)) {
    hipLaunchKernelGGL(sample_kernel, dim3(S), dim3(1024), 0, st, p);
    VDA_CHECK_LAUNCH();
    return 0;
  }
  if (!workspace || workspace_bytes < vda_sample_workspace(S, V, filtered)) return -1;
  SplitRow* ws = (SplitRow*)workspace;
  for (int row0 = 0; row0 < S; row0 += SPLIT_ROWS) {
    const int rows = min(S - row0, SPLIT_ROWS);
    // two workgroups of 1024 threads per CU and no more (61 rows in nine parts are 549, and the last 37 cost as much as all the
    // others), at least a float4 for every thread
    const int G = max(1, min(min(512 / rows, (V + 4095) / 4096), SPLIT_MAX_G));
    hipLaunchKernelGGL(split_stats_kernel, dim3(G, rows), dim3(1024), 0, st, p, ws, row0);
    if (filtered) hipLaunchKernelGGL(split_bins_kernel, dim3(G, rows), dim3(1024), 0, st, p, ws, row0);
    hipLaunchKernelGGL(split_collect_kernel, dim3(G, rows), dim3(1024), 0, st, p, ws, row0);
    hipLaunchKernelGGL(split_finish_kernel, dim3(rows), dim3(1024), 0, st, p, ws, row0, G);
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
