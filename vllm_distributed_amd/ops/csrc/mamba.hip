// State-space (Mamba / Mamba-2) kernels over a ragged batch with per-request state slots.
//
// Both kernels take the same batch description as the attention kernels:
//   qsl[S+1]       first token row of every sequence in the flat [T, ...] inputs
//   seq_lens[S]    tokens of the sequence after this step (0 = padded graph row: skipped)
//   block_table    row s, column 0 holds the state slot of sequence s
// A sequence carries state in from earlier steps when seq_len - new_tokens > 0, so chunked
// prefill, decode and mixed batches are one code path.
// Role of the reference's csrc/mamba/mamba_ssm/selective_scan_fwd.cu and
// csrc/mamba/causal_conv1d/causal_conv1d.cu (varlen forward + single-token update).
#include "common.h"

__device__ __forceinline__ float silu_f(float v) { return v / (1.f + __expf(-v)); }
constexpr float LOG2E = 1.4426950408889634f, LOG2E_LO = 1.925963033500e-8f, LN2 = 0.6931471805599453f;
// log(1 + e^v) = max(v, 0) + log(1 + e^-|v|).  The exponential's argument keeps its rounding error (e^v alone loses 1e-6 of
// a step size at v = -15), and log(1 + e) the part of e that 1 + e rounds away (Kahan's correction, (e - d) / u).  About
// 25 instructions where log1pf takes over 60; relative error at most 2.6e-7 between -87 and 80 (two million v in each of six
// ranges, with correctly rounded exponential, logarithm and reciprocal; log1pf of e^v: 1e-6), zero below, where e^v is subnormal.
__device__ __forceinline__ float softplus_f(float v) {
  const float t = fmaxf(-fabsf(v), -100.f);
  float p = t * LOG2E;
  asm("" : "+v"(p));                                    // (the statements keep roundings that are subtracted below from
  const float lo = fmaf(t, LOG2E_LO, fmaf(t, LOG2E, -p));       //  being simplified away)
  float e = __builtin_amdgcn_exp2f(p);
  e = fmaf(e, lo * LN2, e);
  float u = 1.f + e;
  asm("" : "+v"(u));
  float d = u - 1.f;
  asm("" : "+v"(d));
  const float l = fmaf(e - d, __builtin_amdgcn_rcpf(u), __builtin_amdgcn_logf(u) * LN2);
  return v != v ? v : fmaxf(v, 0.f) + l;
}
// sum over aligned groups of n lanes (n a power of two), in every lane: exchanges inside 16 lanes are modifiers of the addition
template <int CTRL> __device__ __forceinline__ float add_dpp(float v) {
  return v + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, true));
}
template <int n> __device__ __forceinline__ float group_sum(float v) {
  if (n > 1) v = add_dpp<0xb1>(v);                      // lanes 1, 0, 3, 2 of every four
  if (n > 2) v = add_dpp<0x4e>(v);                      // lanes 2, 3, 0, 1
  if (n > 4) v = add_dpp<0x141>(v);                     // eight lanes mirrored (all of a four hold the same)
  if (n > 8) v = add_dpp<0x140>(v);                     // sixteen mirrored
  if (n > 16) v += __shfl_xor(v, 16, 64);
  if (n > 32) v += __shfl_xor(v, 32, 64);
  return v;
}

// ---- depthwise causal convolution ----------------------------------------------------------------
// V neighbouring channels per thread (the coalesced dimension of x and out) and a chunk of tokens, eight of them in flight.
// The W-1 inputs before a chunk come from x itself or, at the start of the step, from conv_state.  The first chunk's
// threads, which alone read conv_state, also roll it forward, from the last inputs of the sequence: one launch.
// Memory bound: 3325 tokens x 8192 channels in bf16 is 24 us of traffic at the copy rate; one channel a thread and a second
// launch for the state took 57 us, this form 29.
// Few new tokens a sequence are a trip to the state and back, which wants threads: one channel each, and up to four tokens one
// token at a time.  Kernel times, four channels and eight tokens a thread -> this: 8192 channels, 256 single tokens 19.6 -> 10.7 us,
// 64 sequences of four 7.9 -> 5.3, eight of thirty 10.4 -> 5.9.
template <typename T, int W, int V, int U>
__global__ __launch_bounds__(256) void causal_conv1d_kernel(
    T* __restrict__ out, const T* __restrict__ x, const T* __restrict__ weight, const T* __restrict__ bias,
    T* __restrict__ conv_state, const int* __restrict__ qsl, const int* __restrict__ seq_lens,
    const int* __restrict__ block_table, long bt_stride, int C, long x_stride, long o_stride, int act, int chunk) {
  typedef T vec_t __attribute__((ext_vector_type(V)));
  const int s = blockIdx.y, c = (blockIdx.x * 256 + threadIdx.x) * V;
  if (c >= C) return;
  const int sl = seq_lens[s];
  if (sl <= 0) return;
  const int t0 = qsl[s], L = qsl[s + 1] - t0;
  const bool has_init = sl - L > 0;
  // (the grid is sized by what the caller says is the longest: its last chunk takes all that is left)
  const int cs = blockIdx.z * chunk, ce = blockIdx.z + 1 < gridDim.z ? min(L, cs + chunk) : L;
  if (cs > 0 && cs >= L) return;
  T* st = conv_state + ((long)block_table[s * bt_stride] * C + c) * (W - 1);
  auto load = [&](int t) { return *reinterpret_cast<const vec_t*>(x + (long)(t0 + t) * x_stride + c); };
  float w[V][W], win[V][W - 1], b[V];
#pragma unroll
  for (int v = 0; v < V; ++v) {
#pragma unroll
    for (int j = 0; j < W; ++j) w[v][j] = (float)weight[(long)(c + v) * W + j];
    b[v] = bias ? (float)bias[c + v] : 0.f;
  }
#pragma unroll
  for (int j = 0; j < W - 1; ++j) {
    const int p = cs - (W - 1) + j;
    if (p >= 0) {
      const vec_t q = load(p);
#pragma unroll
      for (int v = 0; v < V; ++v) win[v][j] = (float)q[v];
    } else {
#pragma unroll
      for (int v = 0; v < V; ++v) win[v][j] = has_init ? (float)st[v * (W - 1) + W - 1 + p] : 0.f;
    }
  }
  const bool whole = cs == 0 && ce == L;                // the window that the walk ends with is the state
  if (cs == 0 && !whole) {
    // the state after this step: input L - (W - 1) + j, from before the step where that is negative
#pragma unroll
    for (int j = 0; j < W - 1; ++j) {
      const int p = L - (W - 1) + j;
      if (p >= 0) {
        const vec_t q = load(p);
#pragma unroll
        for (int v = 0; v < V; ++v) st[v * (W - 1) + j] = q[v];
      } else {
#pragma unroll
        for (int v = 0; v < V; ++v) {
          float o = 0.f;
#pragma unroll
          for (int k = 0; k < W - 1; ++k)
            if (k == W - 1 + p) o = win[v][k];
          st[v * (W - 1) + j] = (T)o;
        }
      }
    }
  }
  for (int t = cs; t < ce; t += U) {
    vec_t cur[U];
#pragma unroll
    for (int k = 0; k < U; ++k) cur[k] = load(min(t + k, ce - 1));
#pragma unroll
    for (int k = 0; k < U; ++k) {
      if (t + k >= ce) break;
      vec_t o;
#pragma unroll
      for (int v = 0; v < V; ++v) {
        float acc = b[v] + w[v][W - 1] * (float)cur[k][v];
#pragma unroll
        for (int j = 0; j < W - 1; ++j) acc += w[v][j] * win[v][j];
#pragma unroll
        for (int j = 0; j < W - 2; ++j) win[v][j] = win[v][j + 1];
        win[v][W - 2] = (float)cur[k][v];
        o[v] = (T)(act ? silu_f(acc) : acc);
      }
      *reinterpret_cast<vec_t*>(out + (long)(t0 + t + k) * o_stride + c) = o;
    }
  }
  if (whole) {
#pragma unroll
    for (int v = 0; v < V; ++v)
#pragma unroll
      for (int j = 0; j < W - 1; ++j) st[v * (W - 1) + j] = (T)win[v][j];
  }
}

VDA_EXPORT int vda_causal_conv1d(void* out, const void* x, const void* weight, const void* bias, void* conv_state,
                                 const int* qsl, const int* seq_lens, const int* block_table, long bt_stride, int S,
                                 int C, int W, int max_q, long x_stride, long o_stride, int act, int dtype,
                                 hipStream_t st) {
  if (S <= 0 || C <= 0) return 0;
  if (W < 2 || W > 8) return -1;
  const int chunk = 32;
  const int nz = max(1, (max_q + chunk - 1) / chunk);
  // four channels a thread where every row starts on such a boundary and there are tokens to walk (more than one chunk)
  const int eb = dtype == VDA_F32 ? 4 : 2;
  const bool one = max_q <= 4, few = max_q <= chunk, vec = !few && C % 4 == 0 && x_stride % 4 == 0 && o_stride % 4 == 0 && (uintptr_t)x % (4 * eb) == 0 && (uintptr_t)out % (4 * eb) == 0;
  dim3 block(256), grid(vec ? (C / 4 + 255) / 256 : (C + 255) / 256, S, nz);
#define L(TT, WW, VV, UU) hipLaunchKernelGGL((causal_conv1d_kernel<TT, WW, VV, UU>), grid, block, 0, st, (TT*)out, (const TT*)x, \
    (const TT*)weight, (const TT*)bias, (TT*)conv_state, qsl, seq_lens, block_table, bt_stride, C, x_stride, o_stride,   \
    act, chunk)
#define BYW(TT, VV, UU) do { switch (W) { case 2: L(TT, 2, VV, UU); break; case 3: L(TT, 3, VV, UU); break; \
    case 4: L(TT, 4, VV, UU); break; case 5: L(TT, 5, VV, UU); break; case 6: L(TT, 6, VV, UU); break;         \
    case 7: L(TT, 7, VV, UU); break; default: L(TT, 8, VV, UU); break; } } while (0)
#define RUN(TT) do { if (one) BYW(TT, 1, 1); else if (vec) BYW(TT, 4, 8); else BYW(TT, 1, 8); } while (0)
  if (dtype == VDA_BF16) RUN(bf16_t);
  else if (dtype == VDA_F16) RUN(f16_t);
  else if (dtype == VDA_F32) RUN(float);
  else return -3;
#undef RUN
#undef BYW
#undef L
  VDA_CHECK_LAUNCH();
  return 0;
}

// ---- selective scan ----------------------------------------------------------------------------
// h[c, n] <- exp(dt * A[c, n]) * h[c, n] + dt * B[t, n] * u[t, c];  y[t, c] = sum_n C[t, n] h[c, n] + D[c] u[t, c]
// NL = N / 16 lanes share one channel (16 states each, y summed with shuffles), so Mamba (N = 16) uses one
// lane per channel and Mamba-2 (N = 128) eight.
//   dt_div      channels per dt / A / D entry (1: per channel; head_dim for Mamba-2 heads)
//   a_scalar    A holds one value per dt entry instead of [C, N]
//   group_ch    channels per B / C group (B, C are [T, groups * N])
// MODE 0  whole sequences in one pass (decode, short chunks): tokens walked in order, state read and written.
// Long prefills are cut into chunks of `chunk` tokens (grid.z) and run in three passes, since the
// recurrence is linear in h:  h_end = P * h_start + H_loc  with P = prod exp(dt A), H_loc = chunk result from 0.
// MODE 1  per chunk: P and H_loc into the workspace (no output)
//         (then scan_combine_kernel walks the chunks of a sequence: start state of every chunk, final state)
// MODE 2  per chunk: outputs, starting from the chunk's start state in the workspace
template <typename T, int N, int MODE>
__global__ __launch_bounds__(256) void selective_scan_kernel(
    T* __restrict__ out, const T* __restrict__ u, const T* __restrict__ delta, const float* __restrict__ A,
    const T* __restrict__ Bm, const T* __restrict__ Cm, const float* __restrict__ D, const T* __restrict__ z,
    const float* __restrict__ delta_bias, float* __restrict__ ssm_state, const int* __restrict__ qsl,
    const int* __restrict__ seq_lens, const int* __restrict__ block_table, long bt_stride, int C, long u_stride,
    long d_stride, long b_stride, long c_stride, long z_stride, long o_stride, int dt_div, int a_scalar,
    int group_ch, int softplus, int chunk, float* __restrict__ ws_p, float* __restrict__ ws_h) {
  constexpr int NL = N / 16;
  const int s = blockIdx.y;
  const int gid = blockIdx.x * 256 + threadIdx.x;
  const int c = gid / NL, part = gid % NL;
  if (c >= C) return;       // NL divides 64, so the lanes of one channel leave together
  const int sl = seq_lens[s];
  if (sl <= 0) return;
  const int t0 = qsl[s], L = qsl[s + 1] - t0;
  const bool has_init = sl - L > 0;
  int ta = t0, tb = t0 + L;
  long ws_off = 0;
  if (MODE != 0) {
    ta = t0 + blockIdx.z * chunk;
    if (ta >= tb) return;
    if (blockIdx.z + 1 < gridDim.z) tb = min(tb, ta + chunk);      // (the last chunk of the grid takes all that is left)
    ws_off = ((((long)s * gridDim.z + blockIdx.z) * C + c) * N) + part * 16;
  }
  float* hp = ssm_state + ((long)block_table[s * bt_stride] * C + c) * N + part * 16;
  const int e = c / dt_div;
  float a[16], h[16], pr[16];
#pragma unroll
  for (int n = 0; n < 16; ++n) {
    a[n] = a_scalar ? A[e] : A[(long)c * N + part * 16 + n];
    if (MODE == 0) h[n] = has_init ? hp[n] : 0.f;
    else if (MODE == 1) h[n] = 0.f;
    else h[n] = ws_p[ws_off + n];            // start state left there by the combine pass
    pr[n] = 1.f;
  }
  const float dv = D ? D[e] : 0.f;
  const float db = delta_bias ? delta_bias[e] : 0.f;
  const long bc_off = (long)(c / group_ch) * N + part * 16;
  // the next token's inputs are on their way while this one's are worked on (past the end: the last token's again)
  T nd, nu, nz = (T)0.f, nb[16], nc[16];
  auto fetch = [&](int t) {
    nd = delta[(long)t * d_stride + e];
    nu = u[(long)t * u_stride + c];
    if (MODE != 1 && z) nz = z[(long)t * z_stride + c];
#pragma unroll
    for (int n = 0; n < 16; ++n) nb[n] = Bm[(long)t * b_stride + bc_off + n];
    if (MODE != 1) {
#pragma unroll
      for (int n = 0; n < 16; ++n) nc[n] = Cm[(long)t * c_stride + bc_off + n];
    }
  };
  if (ta < tb) fetch(ta);
  for (int t = ta; t < tb; ++t) {
    float dt = (float)nd + db;
    const float x = (float)nu, zt = (float)nz;
    T bt[16], ct[16];
#pragma unroll
    for (int n = 0; n < 16; ++n) { bt[n] = nb[n]; if (MODE != 1) ct[n] = nc[n]; }
    fetch(min(t + 1, tb - 1));
    if (softplus) dt = softplus_f(dt);
    const float dx = dt * x;
    float y = 0.f;
#pragma unroll
    for (int n = 0; n < 16; ++n) {
      const float dec = __expf(dt * a[n]);
      h[n] = dec * h[n] + dx * (float)bt[n];
      if (MODE == 1) pr[n] *= dec;
      else y += (float)ct[n] * h[n];
    }
    if (MODE != 1) {
#pragma unroll
      for (int o = NL / 2; o > 0; o >>= 1) y += __shfl_xor(y, o, 64);
      if (part == 0) {
        y += dv * x;
        if (z) y *= silu_f(zt);
        out[(long)t * o_stride + c] = (T)y;
      }
    }
  }
  if (MODE == 0) {
#pragma unroll
    for (int n = 0; n < 16; ++n) hp[n] = h[n];
  } else if (MODE == 1) {
#pragma unroll
    for (int n = 0; n < 16; ++n) { ws_p[ws_off + n] = pr[n]; ws_h[ws_off + n] = h[n]; }
  }
}

// One thread per (sequence, channel, state): walk the sequence's chunks, replace every chunk's P by the
// state the chunk starts from, and leave the final state in the request's slot.
__global__ __launch_bounds__(256) void scan_combine_kernel(float* __restrict__ ws_p, const float* __restrict__ ws_h,
                                                           float* __restrict__ ssm_state,
                                                           const int* __restrict__ qsl,
                                                           const int* __restrict__ seq_lens,
                                                           const int* __restrict__ block_table, long bt_stride,
                                                           long CN, int chunk, int nchunks) {
  const int s = blockIdx.y;
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= CN) return;
  const int sl = seq_lens[s];
  if (sl <= 0) return;
  const int L = qsl[s + 1] - qsl[s];
  float* hp = ssm_state + (long)block_table[s * bt_stride] * CN + i;
  float h = (sl - L > 0) ? *hp : 0.f;
  const int nc = min((L + chunk - 1) / chunk, nchunks);
  for (int k = 0; k < nc; ++k) {
    const long off = ((long)s * nchunks + k) * CN + i;
    const float p = ws_p[off];
    ws_p[off] = h;
    h = p * h + ws_h[off];
  }
  *hp = h;
}

// ---- selective scan, channels in pairs ----------------------------------------------------------------------------------
// The form above loads B and C of every token once per lane, two bytes a load, which is most of its time.  Here a workgroup
// stages them in LDS (fp32) for a tile of tokens, and a lane owns a pair of neighbouring channels, so that one LDS read of four
// states' B and C serves eight updates.  NL = N / 16 lanes share the states of a pair, lane q of them the groups of four
// q, q + NL, q + 2 NL, q + 3 NL: their state accesses are contiguous.
// A chunk's product of decays is exp2(a * sum of dt): the workspace holds the sum, not the product.
// The output pass of several chunks reads its start states from the workspace alone: the last chunk leaves its end state in
// the request's slot while the first one may not have begun, so the carry kernel puts the slot's state aside first.
// Bound by vector issue: per state and token exp2 (4 slots), its argument, two for the state and one for y.
// 3325 tokens of 8192 channels x 16 states, three sequences: both passes 637 -> 320 us;
// 1100 tokens of 64 heads x 64 x 128 states: 990 -> 283 with the convolution.  (The two forms below take most of what this one
// took: it keeps 32-bit inputs, rows off their boundaries, few tokens of many sequences.)
struct ScanArgs {
  void* out;
  const void *u, *delta;
  const float* A;
  const void *B, *C;
  const float* D;
  const void* z;
  const float* delta_bias;
  float* state;
  const int *qsl, *seq_lens, *block_table;
  long bt_stride, u_stride, d_stride, b_stride, c_stride, z_stride, o_stride;
  int Ch, dt_div, group_ch, softplus, chunk, tile;      // tile: tokens staged at a time
  // [S, chunks, Ch] sums of dt; [S, chunks, Ch, N] states: of a sequence's chunks but the last their end states, in the last
  // one's place the state that the sequence starts from
  float *ws_dt, *ws_h;
};
constexpr int SCAN_LDS = 8192;                          // floats of staged B and C

// MODE 0: whole sequences; 1: a chunk's end state from zero and its sum of dt (from the request's state for the first chunk);
// 2: a chunk's outputs from its start state, the last chunk also leaves the request's state.  ASC: one decay rate per dt.
template <typename T, int N, int MODE, bool ASC>
__global__ __launch_bounds__(256) void scan_pairs_kernel(ScanArgs p) {
  typedef T pair_t __attribute__((ext_vector_type(2)));
  constexpr int NL = N / 16, WGCH = 512 / NL;
  __shared__ __attribute__((aligned(16))) float bc[SCAN_LDS];
  const int s = blockIdx.y;
  const int sl = p.seq_lens[s];
  if (sl <= 0) return;
  const int t0 = p.qsl[s], L = p.qsl[s + 1] - t0;
  const int nch = MODE == 0 ? 1 : min((L + p.chunk - 1) / p.chunk, (int)gridDim.z), kch = MODE == 0 ? 0 : blockIdx.z;
  if (kch >= nch || (MODE == 1 && kch == nch - 1)) return;       // (the last chunk's end state falls out of its output pass)
  // (the grid is sized by what the caller says is the longest: a sequence's last chunk takes all that is left)
  const bool last = kch == nch - 1;
  const int ta = MODE == 0 ? 0 : kch * p.chunk, tb = last ? L : ta + p.chunk;
  const bool from_state = sl - L > 0 && kch == 0;
  const int cw = blockIdx.x * WGCH, g0 = cw / p.group_ch;
  const int span = (min(cw + WGCH, p.Ch) - 1) / p.group_ch - g0 + 1;       // B / C groups of this workgroup's channels
  const int part = threadIdx.x % NL;
  const int c = min(cw + 2 * (int)(threadIdx.x / NL), p.Ch - 2);
  const bool mine = cw + 2 * (int)(threadIdx.x / NL) < p.Ch;
  const int e0 = c / p.dt_div, e1 = (c + 1) / p.dt_div;
  const int grp = c / p.group_ch - g0;
  float* hp = p.state + ((long)p.block_table[s * p.bt_stride] * p.Ch + c) * N + 4 * part;
  const long wc = ((long)s * gridDim.z + kch) * p.Ch + c;

  f32x4 a[2][4], h[2][4];
  float as[2] = {ASC ? p.A[e0] * LOG2E : 0.f, ASC ? p.A[e1] * LOG2E : 0.f}, sdt[2] = {0.f, 0.f};
#pragma unroll
  for (int v = 0; v < 2; ++v)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int at = v * N + 4 * j * NL;
      if (!ASC) a[v][j] = *reinterpret_cast<const f32x4*>(p.A + (long)c * N + 4 * part + at) * LOG2E;
      if (MODE == 2 && kch > 0) h[v][j] = *reinterpret_cast<const f32x4*>(p.ws_h + (wc - p.Ch) * N + 4 * part + at);
      else if (MODE == 2 && from_state && nch > 1)
        h[v][j] = *reinterpret_cast<const f32x4*>(p.ws_h + (wc + (long)(nch - 1) * p.Ch) * N + 4 * part + at);
      else h[v][j] = from_state ? *reinterpret_cast<const f32x4*>(hp + at) : f32x4{0, 0, 0, 0};
    }
  const float dv[2] = {p.D ? p.D[e0] : 0.f, p.D ? p.D[e1] : 0.f};
  const float db[2] = {p.delta_bias ? p.delta_bias[e0] : 0.f, p.delta_bias ? p.delta_bias[e1] : 0.f};
  const T* U = (const T*)p.u + (long)t0 * p.u_stride + c;
  const T* Dt = (const T*)p.delta + (long)t0 * p.d_stride;
  const T* Z = p.z ? (const T*)p.z + (long)t0 * p.z_stride + c : nullptr;
  T* O = (T*)p.out + (long)t0 * p.o_stride + c;

  // TB tokens at a time; lane q of a pair's NL works out the step sizes and finishes the outputs of tokens q, q + NL, ...
  constexpr int TB = NL < 2 ? 2 : NL, OWN = TB / NL;
  // the next block's inputs (past the end: the last token's again)
  pair_t nu[TB], nz[OWN];
  float nd[OWN][2];
  auto fetch = [&](int t) {
#pragma unroll
    for (int o = 0; o < OWN; ++o) {
      const long at_t = min(t + part + o * NL, tb - 1);
      if (p.dt_div == 1) {
        const pair_t d = *reinterpret_cast<const pair_t*>(Dt + at_t * p.d_stride + c);
        nd[o][0] = (float)d[0];
        nd[o][1] = (float)d[1];
      } else {
        nd[o][0] = (float)Dt[at_t * p.d_stride + e0];
        nd[o][1] = 0.f;
      }
      if (MODE != 1 && Z) nz[o] = *reinterpret_cast<const pair_t*>(Z + at_t * p.z_stride);
      else nz[o] = pair_t{(T)0.f, (T)0.f};
    }
#pragma unroll
    for (int k = 0; k < TB; ++k) nu[k] = *reinterpret_cast<const pair_t*>(U + (long)min(t + k, tb - 1) * p.u_stride);
  };
  if (ta < tb) fetch(ta);

  const int per = 2 * N * span;                         // staged floats per token: [span][B, C][N]
  for (int tt = ta; tt < tb; tt += p.tile) {
    const int nt = min(p.tile, tb - tt);
    __syncthreads();
    for (int i = threadIdx.x; i < nt * per; i += 256) {
      const int t = i / per, k = i - t * per, g = k / (2 * N), n = k % (2 * N);
      const long at = (long)(g0 + g) * N + n % N;
      bc[i] = n < N ? (float)((const T*)p.B)[(long)(t0 + tt + t) * p.b_stride + at]
                    : (float)((const T*)p.C)[(long)(t0 + tt + t) * p.c_stride + at];
    }
    __syncthreads();
    for (int tk = 0; tk < nt; tk += TB) {
      pair_t uu[TB], zz[OWN];
      float my_dt[OWN][2], my_dec[OWN][2];
#pragma unroll
      for (int k = 0; k < TB; ++k) uu[k] = nu[k];
#pragma unroll
      for (int o = 0; o < OWN; ++o) { zz[o] = nz[o]; my_dt[o][0] = nd[o][0]; my_dt[o][1] = nd[o][1]; }
      // under this block's arithmetic (a tile that ends inside a block leaves the rest of it to the next)
      fetch(tt + min(tk + TB, nt));
#pragma unroll
      for (int o = 0; o < OWN; ++o)
#pragma unroll
        for (int v = 0; v < 2; ++v) {
          if (v == 1 && p.dt_div > 1) { my_dt[o][1] = my_dt[o][0]; my_dec[o][1] = my_dec[o][0]; continue; }
          my_dt[o][v] += db[v];
          if (p.softplus) my_dt[o][v] = softplus_f(my_dt[o][v]);
          if (tk + part + o * NL >= nt) my_dt[o][v] = 0.f;       // no token: the state stays as it is
          my_dec[o][v] = ASC ? __builtin_amdgcn_exp2f(my_dt[o][v] * as[v]) : 0.f;
        }
      float y[OWN][2];
#pragma unroll
      for (int k = 0; k < TB; ++k) {
        const f32x4* bp = reinterpret_cast<const f32x4*>(bc + min(tk + k, nt - 1) * per + grp * 2 * N) + part;
        float dt[2], dx[2], dec[2], yk[2] = {0.f, 0.f};
        const int from = (threadIdx.x & 63 & ~(NL - 1)) + k % NL;
#pragma unroll
        for (int v = 0; v < 2; ++v) {
          dt[v] = NL == 1 ? my_dt[k / NL][v] : v == 1 && p.dt_div > 1 ? dt[0] : __shfl(my_dt[k / NL][v], from, 64);
          dec[v] = !ASC || NL == 1 ? my_dec[k / NL][v] : v == 1 && p.dt_div > 1 ? dec[0] : __shfl(my_dec[k / NL][v], from, 64);
          dx[v] = dt[v] * (float)uu[k][v];
          if (MODE == 1) sdt[v] += dt[v];
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const f32x4 b = bp[j * NL];
          const f32x4 cc = MODE != 1 ? bp[N / 4 + j * NL] : b;
#pragma unroll
          for (int v = 0; v < 2; ++v)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const float d = ASC ? dec[v] : __builtin_amdgcn_exp2f(dt[v] * a[v][j][i]);
              h[v][j][i] = fmaf(d, h[v][j][i], dx[v] * b[i]);
              if (MODE != 1) yk[v] = fmaf(cc[i], h[v][j][i], yk[v]);
            }
        }
        if (MODE != 1) {
#pragma unroll
          for (int v = 0; v < 2; ++v) {
            yk[v] = group_sum<NL>(yk[v]) + dv[v] * (float)uu[k][v];
            if (k % NL == 0 || k % NL == part) y[k / NL][v] = yk[v];
          }
        }
        __builtin_amdgcn_sched_barrier(0);               // token by token: their operands together do not fit
      }
      if (MODE != 1 && mine) {
#pragma unroll
        for (int q = 0; q < OWN; ++q) {
          const int t = tk + part + q * NL;
          if (t >= nt) break;
          pair_t o;
#pragma unroll
          for (int v = 0; v < 2; ++v) o[v] = (T)(Z ? y[q][v] * silu_f((float)zz[q][v]) : y[q][v]);
          *reinterpret_cast<pair_t*>(O + (long)(tt + t) * p.o_stride) = o;
        }
      }
    }
  }
  if (!mine) return;
  if (MODE == 1 && part == 0) { p.ws_dt[wc] = sdt[0]; p.ws_dt[wc + 1] = sdt[1]; }
  float* to = MODE == 1 ? p.ws_h + wc * N + 4 * part : hp;
  if (MODE == 1 || last) {
#pragma unroll
    for (int v = 0; v < 2; ++v)
#pragma unroll
      for (int j = 0; j < 4; ++j) *reinterpret_cast<f32x4*>(to + v * N + 4 * j * NL) = h[v][j];
  }
}

// The sequence of workgroups blockIdx.y == at of a pass over whole sequences: the longest ones' start first (up to 64 of them).  What waits for a place
// on the chip at its end is short then, and of the waves of a SIMD the first to start is the first to issue, so the longest one does not
// walk its last tokens alone, when only every eighth cycle issues.  us, convolution and scan, in the batch's order -> this: 16 states, 8192 channels, three of
// 1558, 1043 and 724 tokens 215 -> 207, 16 of some 180 162 -> 156, two of some 1400 305 -> 294; 128 states, 4096 channels, these three 276 -> 261, 16 of some
// 180 231 -> 224.  (With s_setprio by length as well: 209, 159, 296, 263, 227.)  Called by whole waves.
__device__ __forceinline__ int by_length(const int* qsl, int S, int at) {
  if (S > 64) return at;
  const int lane = threadIdx.x & 63;
  const int len = lane < S ? qsl[lane + 1] - qsl[lane] : -1;
  int before = 0;
  for (int i = 0; i < S; ++i) {
    const int other = __builtin_amdgcn_readlane(len, i);
    before += other > len || (other == len && i < lane);
  }
  return __builtin_amdgcn_readfirstlane((int)__builtin_ctzll(__ballot(before == at && lane < S)));
}
// ---- selective scan, two states a lane ---------------------------------------------------------------------------------
// 16 states with decay rates of their own (Mamba): eight lanes share a channel, two states each, so that three prompts of 8192
// channels are 3072 waves and walk their tokens in one pass where the pairs above took two.  A SIMD issues at its full rate from
// two waves on (one alone: every 8 cycles instead of 4, measured), which is what chunks are still made for where sequences
// and channels are few.
// Everything that a (token, channel) needs once is done while a tile of 32 tokens x 32 channels is staged: a thread takes four
// channels of a token, applies the softplus and leaves (dt, dt * u) in LDS; the gate and D join when the tile's sums come
// back through LDS.  The recurrence itself then reads two LDS words a token, B and C of its two states beside each other.
// The sums over a channel's eight lanes are transposed ones: of eight tokens' partial sums each lane sends the half that its
// partner finishes, 21 instructions for eight tokens instead of 24 additions and eight selections, and lane k ends with token k's.
// Per state and token: exp2 (two issue slots), its argument, two for the state, one for y: 69 us for 3325 tokens of 8192 channels
// x 16 states at the full rate, with the sums and the staging about twice that: 298 (pairs) -> 163 us; 16 sequences of 323 tokens
// at most 291 -> 126; one of 1609 169 -> 119, with 4096 channels 105 -> 70.
constexpr int LN_TT = 32, LN_CH = 32, LN_YS = 40;       // tokens and channels of a tile; floats between two tokens' sums
template <typename T> __device__ __forceinline__ void load_few(const T* p, float (&v)[4], bool vec, int last) {
  typedef T v4_t __attribute__((ext_vector_type(4)));
  if (vec) {
    const v4_t q = *reinterpret_cast<const v4_t*>(p);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = (float)q[i];
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = (float)p[min(i, last)];
  }
}
// The first of the four channels that a staging thread reads.  Threads past the last channel (their values are dropped) read the
// last four again where four are read at once, which begin where theirs would: C is a multiple of four there.
__host__ __device__ __forceinline__ int lane_channel(int at, int C, int vec) {
  const int most = C - (vec ? 4 : 1);
  return at < most ? at : most;
}
// (for the test of its bounds, which runs on the host)
VDA_EXPORT int vda_scan_lane_channel(int at, int C, int vec) { return lane_channel(at, C, vec); }
// a chunk's MODE, as in the pairs above; vec: rows of four channels may be read and written at once
template <typename T, int MODE>
__global__ __launch_bounds__(256) void scan_lanes_kernel(ScanArgs p, int vec) {
  constexpr int N = 16;
  typedef T v4_t __attribute__((ext_vector_type(4)));
  __shared__ __attribute__((aligned(16))) float dd[LN_TT][LN_CH][2], bc[LN_TT][8][4], ys[LN_TT][LN_YS];
  const int s = MODE == 0 ? by_length(p.qsl, gridDim.y, blockIdx.y) : blockIdx.y;
  const int sl = p.seq_lens[s];
  if (sl <= 0) return;
  const int t0 = p.qsl[s], L = p.qsl[s + 1] - t0;
  const int nch = MODE == 0 ? 1 : min((L + p.chunk - 1) / p.chunk, (int)gridDim.z), kch = MODE == 0 ? 0 : blockIdx.z;
  if (kch >= nch || (MODE == 1 && kch == nch - 1)) return;
  const bool last = kch == nch - 1;
  const int ta = MODE == 0 ? 0 : kch * p.chunk, tb = last ? L : ta + p.chunk;
  if (ta >= tb) return;
  const bool from_state = sl - L > 0 && kch == 0;
  // neighbouring workgroups share lines of 128 bytes: they go to one XCD (workgroups are dealt to the eight in turn)
  const int nb = gridDim.x, cb = nb % 8 ? (int)blockIdx.x : (int)(blockIdx.x % 8) * (nb / 8) + (int)(blockIdx.x / 8);
  const int cw = cb * LN_CH;
  const int lane = threadIdx.x & 63, q = lane & 7, mych = (threadIdx.x >> 6) * 8 + (lane >> 3);
  const int c = min(cw + mych, p.Ch - 1);
  const bool mine = cw + mych < p.Ch;
  float* hp = p.state + ((long)p.block_table[s * p.bt_stride] * p.Ch + c) * N + 2 * q;
  const long wc = ((long)s * gridDim.z + kch) * p.Ch + c;
  f32x2 a = *reinterpret_cast<const f32x2*>(p.A + (long)c * N + 2 * q), h = {0, 0};
  a[0] *= LOG2E;
  a[1] *= LOG2E;
  if (MODE == 2 && kch > 0) h = *reinterpret_cast<const f32x2*>(p.ws_h + (wc - p.Ch) * N + 2 * q);
  else if (MODE == 2 && from_state && nch > 1) h = *reinterpret_cast<const f32x2*>(p.ws_h + (wc + (long)(nch - 1) * p.Ch) * N + 2 * q);
  else if (from_state) h = *reinterpret_cast<const f32x2*>(hp);

  // staging: this thread's token of a tile, its four channels, and its two states' B and C
  const int st = threadIdx.x >> 3, sc = 4 * (threadIdx.x & 7), c4 = lane_channel(cw + sc, p.Ch, vec), left = p.Ch - 1 - c4;
  const long g = (long)(cw / p.group_ch) * N + 2 * (threadIdx.x & 7);
  const T* U = (const T*)p.u + (long)t0 * p.u_stride + c4;
  const T* Dt = (const T*)p.delta + (long)t0 * p.d_stride + c4;
  const T* Z = p.z ? (const T*)p.z + (long)t0 * p.z_stride + c4 : nullptr;
  const T* B = (const T*)p.B + (long)t0 * p.b_stride + g;
  const T* C = (const T*)p.C + (long)t0 * p.c_stride + g;
  T* O = (T*)p.out + (long)t0 * p.o_stride + c4;
  float dv[4], db[4], nd[4], nu[4], nz[4] = {0, 0, 0, 0}, nbc[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    dv[i] = p.D ? p.D[c4 + min(i, left)] : 0.f;
    db[i] = p.delta_bias ? p.delta_bias[c4 + min(i, left)] : 0.f;
  }
  auto fetch = [&](int tt) {
    const long t = tt + st;
    if (t >= tb) return;
    load_few(Dt + t * p.d_stride, nd, vec, left);
    load_few(U + t * p.u_stride, nu, vec, left);
    if (MODE != 1 && Z) load_few(Z + t * p.z_stride, nz, vec, left);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      nbc[i] = (float)B[t * p.b_stride + i];
      nbc[2 + i] = MODE != 1 ? (float)C[t * p.c_stride + i] : 0.f;
    }
  };
  fetch(ta);
  float sdt[4] = {0, 0, 0, 0};
  for (int tt = ta; tt < tb; tt += LN_TT) {
    const bool there = tt + st < tb;                    // no token: the state stays as it is
    float cu[4], cz[4];
    f32x4 w[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}}, wb = {0, 0, 0, 0};
    if (there) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float dt = nd[i] + db[i];
        if (p.softplus) dt = softplus_f(dt);
        if (MODE == 1) sdt[i] += dt;
        cu[i] = nu[i];
        cz[i] = nz[i];
        w[i >> 1][2 * (i & 1)] = dt;
        w[i >> 1][2 * (i & 1) + 1] = dt * nu[i];
        wb[i] = nbc[i];
      }
    }
    *reinterpret_cast<f32x4*>(&dd[st][sc][0]) = w[0];
    *reinterpret_cast<f32x4*>(&dd[st][sc + 2][0]) = w[1];
    *reinterpret_cast<f32x4*>(&bc[st][threadIdx.x & 7][0]) = wb;
    __syncthreads();
    if (tt + LN_TT < tb) fetch(tt + LN_TT);             // under this tile's arithmetic
    const int nt = min(LN_TT, tb - tt);
    for (int tk = 0; tk < nt; tk += 8) {
      float y[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const f32x2 d = *reinterpret_cast<const f32x2*>(&dd[tk + k][mych][0]);
        const f32x4 b = *reinterpret_cast<const f32x4*>(&bc[tk + k][q][0]);
        h[0] = fmaf(__builtin_amdgcn_exp2f(d[0] * a[0]), h[0], d[1] * b[0]);
        h[1] = fmaf(__builtin_amdgcn_exp2f(d[0] * a[1]), h[1], d[1] * b[1]);
        y[k] = fmaf(b[3], h[1], b[2] * h[0]);
      }
      if (MODE != 1) {
        auto meet = [](float keep, float send, auto ctrl) {
          return keep + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(send), decltype(ctrl)::value, 0xf, 0xf, true));
        };
        const bool b2 = q & 4, b1 = q & 2, b0 = q & 1;
        float y4[4], y2[2];
#pragma unroll
        for (int k = 0; k < 4; ++k) y4[k] = meet(b2 ? y[k + 4] : y[k], b2 ? y[k] : y[k + 4], std::integral_constant<int, 0x141>());
#pragma unroll
        for (int k = 0; k < 2; ++k) y2[k] = meet(b1 ? y4[k + 2] : y4[k], b1 ? y4[k] : y4[k + 2], std::integral_constant<int, 0x1b>());
        ys[tk + q][mych] = meet(b0 ? y2[1] : y2[0], b0 ? y2[0] : y2[1], std::integral_constant<int, 0xb1>());
      }
    }
    __syncthreads();
    if (MODE != 1 && there && cw + sc < p.Ch) {
      const f32x4 y = *reinterpret_cast<const f32x4*>(&ys[st][sc]);
      v4_t o;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float v = fmaf(dv[i], cu[i], y[i]);
        o[i] = (T)(Z ? v * silu_f(cz[i]) : v);
      }
      T* to = O + (long)(tt + st) * p.o_stride;
      if (vec) *reinterpret_cast<v4_t*>(to) = o;
      else
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (i <= left) to[i] = o[i];
    }
  }
  if (MODE == 1) {                                      // a channel's sum of dt: over the 32 threads that staged its tokens
    __syncthreads();
    *reinterpret_cast<f32x4*>(&ys[st][sc]) = f32x4{sdt[0], sdt[1], sdt[2], sdt[3]};
    __syncthreads();
    if (threadIdx.x < LN_CH && cw + (int)threadIdx.x < p.Ch) {
      float sum = 0.f;
      for (int t = 0; t < LN_TT; ++t) sum += ys[t][threadIdx.x];
      p.ws_dt[((long)s * gridDim.z + kch) * p.Ch + cw + threadIdx.x] = sum;
    }
  }
  if (mine && (MODE == 1 || last)) *reinterpret_cast<f32x2*>(MODE == 1 ? p.ws_h + wc * N + 2 * q : hp) = h;
}

// ---- selective scan, one decay a head: eight states a lane --------------------------------------------------------------
// Mamba-2: a step size and a decay rate per head, 64 states and more.  A workgroup takes 64 / Q channels of one head, its 4 Q lane
// groups eight states each (Q lanes of every wave share a channel): three prompts of 64 heads x 64 are 3072 waves, which walk their
// tokens in one pass.  Step size, decay and dt * u are worked out while a tile of 16 tokens is staged, and the gate and D join
// when its sums come back, as above; the recurrence reads a pair and 16 values of B and C a token from LDS and does three
// instructions a state.  A channel's sums go over its Q lanes transposed (Q tokens at a time) and over the waves through LDS.
// Bound by the reads of B and C from LDS (32 cycles of a CU a wave and token beside 30 instructions).  us, pairs -> this, 4096 x 128
// states: 3325 tokens of three 598 -> 254, one of 1609 337 -> 192, 16 of 173 at most 226 -> 118.
constexpr int GR_TT = 16;
template <typename T, int N, int MODE>
__global__ __launch_bounds__(256) void scan_groups_kernel(ScanArgs p) {
  typedef T v8_t __attribute__((ext_vector_type(8)));
  constexpr int Q = N / 32, CH = 64 / Q;                // lanes of a wave per channel, channels of a workgroup
  constexpr int PER = N / 4;                            // 16-byte pieces (8 values) of B and C of a tile
  constexpr int STEPS = GR_TT * PER / 256 > 0 ? GR_TT * PER / 256 : 1;
  __shared__ __attribute__((aligned(16))) float bc[GR_TT][2][N], dd[GR_TT][CH][2], ys[4][GR_TT][CH];
  __shared__ float head_dt[GR_TT][2];
  const int s = MODE == 0 ? by_length(p.qsl, gridDim.y, blockIdx.y) : blockIdx.y;
  const int sl = p.seq_lens[s];
  if (sl <= 0) return;
  const int t0 = p.qsl[s], L = p.qsl[s + 1] - t0;
  const int nch = MODE == 0 ? 1 : min((L + p.chunk - 1) / p.chunk, (int)gridDim.z), kch = MODE == 0 ? 0 : blockIdx.z;
  if (kch >= nch || (MODE == 1 && kch == nch - 1)) return;
  const bool last = kch == nch - 1;
  const int ta = MODE == 0 ? 0 : kch * p.chunk, tb = last ? L : ta + p.chunk;
  if (ta >= tb) return;
  const bool from_state = sl - L > 0 && kch == 0;
  const int nb = gridDim.x, cb = nb % 8 ? (int)blockIdx.x : (int)(blockIdx.x % 8) * (nb / 8) + (int)(blockIdx.x / 8);
  const int cw = cb * CH, e = cw / p.dt_div;            // (a workgroup's channels are one head's)
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, q = lane % Q, mych = lane / Q, c = cw + mych;
  const int n0 = 8 * (wave * Q + q);
  float* hp = p.state + ((long)p.block_table[s * p.bt_stride] * p.Ch + c) * N + n0;
  const long wc = ((long)s * gridDim.z + kch) * p.Ch + c;
  const float rate = p.A[e] * LOG2E, dbias = p.delta_bias ? p.delta_bias[e] : 0.f, dv = p.D ? p.D[e] : 0.f;
  f32x4 h[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
  {
    const float* from = MODE == 2 && kch > 0 ? p.ws_h + (wc - p.Ch) * N + n0
                        : MODE == 2 && from_state && nch > 1 ? p.ws_h + (wc + (long)(nch - 1) * p.Ch) * N + n0
                        : from_state ? hp : nullptr;
    if (from) { h[0] = reinterpret_cast<const f32x4*>(from)[0]; h[1] = reinterpret_cast<const f32x4*>(from)[1]; }
  }
  const long g = (long)(cw / p.group_ch) * N;
  const T* U = (const T*)p.u + (long)t0 * p.u_stride + cw;
  const T* Dt = (const T*)p.delta + (long)t0 * p.d_stride + e;
  const T* Z = p.z ? (const T*)p.z + (long)t0 * p.z_stride + cw : nullptr;
  const T* B = (const T*)p.B + (long)t0 * p.b_stride + g;
  const T* C = (const T*)p.C + (long)t0 * p.c_stride + g;
  T* O = (T*)p.out + (long)t0 * p.o_stride + cw;
  // staging: pieces of B and C, one value of u and z for each of GR_TT * CH / 256 tokens, a token's step size
  constexpr int UV = (GR_TT * CH + 255) / 256;
  v8_t nbc[STEPS];
  float nu[UV], nz[UV], nd = 0.f;
  auto fetch = [&](int tt) {                            // (past the end: the last token's again)
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {
      const int pi = tid + 256 * i, t = pi / PER, k = pi % PER;
      const long at = min(tt + min(t, GR_TT - 1), tb - 1);
      nbc[i] = k < PER / 2 ? *reinterpret_cast<const v8_t*>(B + at * p.b_stride + 8 * k)
                           : *reinterpret_cast<const v8_t*>(C + at * p.c_stride + 8 * (k - PER / 2));
    }
#pragma unroll
    for (int i = 0; i < UV; ++i) {
      const int vi = tid + 256 * i, t = min(vi / CH, GR_TT - 1), ch = vi % CH;
      const long at = min(tt + t, tb - 1);
      nu[i] = (float)U[at * p.u_stride + ch];
      nz[i] = MODE != 1 && Z ? (float)Z[at * p.z_stride + ch] : 0.f;
    }
    if (tid < GR_TT) nd = (float)Dt[(long)min(tt + tid, tb - 1) * p.d_stride];
  };
  fetch(ta);
  float sdt = 0.f;
  for (int tt = ta; tt < tb; tt += GR_TT) {
    if (tid < GR_TT) {
      float dt = nd + dbias;
      if (p.softplus) dt = softplus_f(dt);
      if (tt + tid >= tb) dt = 0.f;                     // no token: the state stays as it is
      sdt += dt;
      head_dt[tid][0] = __builtin_amdgcn_exp2f(dt * rate);
      head_dt[tid][1] = dt;
    }
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {
      const int pi = tid + 256 * i, t = pi / PER, k = pi % PER;
      if (GR_TT * PER % 256 && t >= GR_TT) break;
      float* to = &bc[t][0][0] + 8 * k;                 // (B's values, then C's)
#pragma unroll
      for (int v = 0; v < 2; ++v) {
        f32x4 w;
#pragma unroll
        for (int j = 0; j < 4; ++j) w[j] = tt + t < tb ? (float)nbc[i][4 * v + j] : 0.f;
        reinterpret_cast<f32x4*>(to)[v] = w;
      }
    }
    float cu[UV], cz[UV];
#pragma unroll
    for (int i = 0; i < UV; ++i) { cu[i] = nu[i]; cz[i] = nz[i]; }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < UV; ++i) {
      const int vi = tid + 256 * i, t = vi / CH, ch = vi % CH;
      if (GR_TT * CH % 256 && t >= GR_TT) break;
      const float dt = head_dt[t][1];
      *reinterpret_cast<f32x2*>(&dd[t][ch][0]) = f32x2{head_dt[t][0], tt + t < tb ? dt * cu[i] : 0.f};
    }
    __syncthreads();
    if (tt + GR_TT < tb) fetch(tt + GR_TT);             // under this tile's arithmetic
    const int nt = min(GR_TT, tb - tt);
    for (int tk = 0; tk < nt; tk += 8) {
      float y[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const f32x2 d = *reinterpret_cast<const f32x2*>(&dd[tk + k][mych][0]);
        const f32x4* b = reinterpret_cast<const f32x4*>(&bc[tk + k][0][n0]);
        const f32x4* cc = reinterpret_cast<const f32x4*>(&bc[tk + k][1][n0]);
        y[k] = 0.f;
#pragma unroll
        for (int v = 0; v < 2; ++v) {
          const f32x4 bv = b[v], cv = MODE != 1 ? cc[v] : f32x4{0, 0, 0, 0};
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            h[v][j] = fmaf(d[0], h[v][j], d[1] * bv[j]);
            if (MODE != 1) y[k] = fmaf(cv[j], h[v][j], y[k]);
          }
        }
      }
      if (MODE != 1) {                                  // lane q of a channel's Q ends with tokens q, q + Q, ...
        auto meet = [](float keep, float send, auto ctrl) {
          return keep + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(send), decltype(ctrl)::value, 0xf, 0xf, true));
        };
        if constexpr (Q == 8) {
          const bool b2 = q & 4;
#pragma unroll
          for (int k = 0; k < 4; ++k) y[k] = meet(b2 ? y[k + 4] : y[k], b2 ? y[k] : y[k + 4], std::integral_constant<int, 0x141>());
        }
        constexpr int K4 = Q == 8 ? 4 : 8;              // values left: of every four, two and one
        if constexpr (Q >= 4) {
          const bool b1 = q & 2;
#pragma unroll
          for (int j = 0; j < K4; j += 4)
#pragma unroll
            for (int k = 0; k < 2; ++k)
              y[j / 2 + k] = meet(b1 ? y[j + k + 2] : y[j + k], b1 ? y[j + k] : y[j + k + 2], std::integral_constant<int, 0x1b>());
        }
        constexpr int K2 = Q == 8 ? 2 : Q == 4 ? 4 : 8;
        if constexpr (Q >= 2) {
          const bool b0 = q & 1;
#pragma unroll
          for (int j = 0; j < K2; j += 2) y[j / 2] = meet(b0 ? y[j + 1] : y[j], b0 ? y[j] : y[j + 1], std::integral_constant<int, 0xb1>());
        }
#pragma unroll
        for (int j = 0; j < 8 / Q; ++j) ys[wave][tk + Q * j + q][mych] = y[j];
      }
    }
    __syncthreads();
    if (MODE != 1)
#pragma unroll
      for (int i = 0; i < UV; ++i) {
        const int vi = tid + 256 * i, t = vi / CH, ch = vi % CH;
        if (t >= nt) break;
        float v = fmaf(dv, cu[i], (ys[0][t][ch] + ys[1][t][ch]) + (ys[2][t][ch] + ys[3][t][ch]));
        if (Z) v *= silu_f(cz[i]);
        O[(long)(tt + t) * p.o_stride + ch] = (T)v;
      }
  }
  if (MODE == 1 && wave == 0) {                         // the sum of dt, for every channel of the workgroup
    sdt = lane < GR_TT ? sdt : 0.f;
    sdt = group_sum<16>(sdt);
    sdt = __shfl(sdt, 0, 64);
    if (lane < CH) p.ws_dt[((long)s * gridDim.z + kch) * p.Ch + cw + lane] = sdt;
  }
  if (MODE == 1 || last) {
    float* to = MODE == 1 ? p.ws_h + wc * N + n0 : hp;
    reinterpret_cast<f32x4*>(to)[0] = h[0];
    reinterpret_cast<f32x4*>(to)[1] = h[1];
  }
}

// One thread per (sequence, channel, four states): walk the chunks, leaving in chunk k's place its TRUE end state, which is
// where chunk k + 1 starts.  (The first chunk's is true already.)  The last chunk's place, which has no end state yet, takes
// the state that the sequence continues from.
template <bool ASC>
__global__ __launch_bounds__(256) void scan_carry_kernel(ScanArgs p, int N, int nchunks) {
  const int s = blockIdx.y;
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  const int c = (int)(i / (N / 4)), n = (int)(i % (N / 4)) * 4;
  const int sl = p.seq_lens[s];
  if (c >= p.Ch || sl <= 0) return;
  const int L = p.qsl[s + 1] - p.qsl[s], nc = min((L + p.chunk - 1) / p.chunk, nchunks);
  f32x4 a;
  if (ASC) { const float v = p.A[c / p.dt_div] * LOG2E; a = f32x4{v, v, v, v}; }
  else a = *reinterpret_cast<const f32x4*>(p.A + (long)c * N + n) * LOG2E;
  f32x4 h = {0, 0, 0, 0};
  const long w0 = (long)s * nchunks * p.Ch + c;
  if (nc > 1 && sl - L > 0)
    *reinterpret_cast<f32x4*>(p.ws_h + (w0 + (long)(nc - 1) * p.Ch) * N + n) =
        *reinterpret_cast<const f32x4*>(p.state + ((long)p.block_table[s * p.bt_stride] * p.Ch + c) * N + n);
  constexpr int U = 8;                                  // chunks in flight
  for (int k0 = 0; k0 < nc - 1; k0 += U) {
    f32x4 loc[U];
    float dt[U];
#pragma unroll
    for (int k = 0; k < U; ++k) {
      const long w = w0 + (long)min(k0 + k, nc - 2) * p.Ch;
      loc[k] = *reinterpret_cast<const f32x4*>(p.ws_h + w * N + n);
      dt[k] = p.ws_dt[w];
    }
#pragma unroll
    for (int k = 0; k < U; ++k) {
      if (k0 + k >= nc - 1) break;
      if (k0 + k == 0) { h = loc[k]; continue; }
#pragma unroll
      for (int j = 0; j < 4; ++j) h[j] = fmaf(__builtin_amdgcn_exp2f(dt[k] * a[j]), h[j], loc[k][j]);
      *reinterpret_cast<f32x4*>(p.ws_h + (w0 + (long)(k0 + k) * p.Ch) * N + n) = h;
    }
  }
}

// One token per sequence (or few): the state read and written is all there is (118 sequences of
// 4096 x 128 states, 495 MB, with the convolution: 118 us).  A lane owns four states, a wave one contiguous KB of them, and
// K of those are in flight: eight where the states are many.  Few are a chain of trips to memory, so there two are taken by a wave
// and all their inputs are asked for before the first store, which the compiler moves no load across (one sequence of
// 4096 x 16 states 8.3 us with eight, 6.2 in the plain form; SCAN_FEW says how many are few).
template <typename T, int N, bool ASC, int K>
__global__ __launch_bounds__(256) void scan_step_kernel(ScanArgs p) {
  constexpr int Q = N / 4, CW = 64 / Q;                 // lanes per channel, channels per KB
  constexpr bool AHEAD = K <= 2;
  const int s = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int sl = p.seq_lens[s];
  if (sl <= 0) return;
  const int t0 = p.qsl[s], L = p.qsl[s + 1] - t0;
  if (L <= 0) return;
  const bool has_init = sl - L > 0;
  const int q = lane % Q, c0 = (blockIdx.x * 4 + wave) * (CW * K) + lane / Q;
  float* hp = p.state + (long)p.block_table[s * p.bt_stride] * p.Ch * N + 4 * q;
  f32x4 h[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int c = c0 + k * CW;
    h[k] = has_init && c < p.Ch ? *reinterpret_cast<const f32x4*>(hp + (long)c * N) : f32x4{0, 0, 0, 0};
  }
  // one channel's inputs of a token, and what is done with them (whole channels: the lanes of one come here together)
  struct In { T delta, u, z, b[4], c[4]; float bias, d; f32x4 a; };
  auto load = [&](int t, int c) {
    In in;
    const int e = c / p.dt_div;
    in.delta = ((const T*)p.delta)[(long)t * p.d_stride + e];
    in.u = ((const T*)p.u)[(long)t * p.u_stride + c];
    in.z = p.z ? ((const T*)p.z)[(long)t * p.z_stride + c] : (T)0.f;
    in.bias = p.delta_bias ? p.delta_bias[e] : 0.f;
    in.d = p.D ? p.D[e] : 0.f;
    const long g = (long)(c / p.group_ch) * N + 4 * q;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      in.b[i] = ((const T*)p.B)[(long)t * p.b_stride + g + i];
      in.c[i] = ((const T*)p.C)[(long)t * p.c_stride + g + i];
    }
    if (ASC) { const float v = p.A[e]; in.a = f32x4{v, v, v, v}; }
    else in.a = *reinterpret_cast<const f32x4*>(p.A + (long)c * N + 4 * q);
    return in;
  };
  auto token = [&](int t, int c, f32x4 hk, const In& in) {
    float dt = (float)in.delta + in.bias;
    if (p.softplus) dt = softplus_f(dt);
    const float x = (float)in.u, dx = dt * x;
    float y = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      hk[i] = fmaf(__builtin_amdgcn_exp2f(dt * (in.a[i] * LOG2E)), hk[i], dx * (float)in.b[i]);
      y = fmaf((float)in.c[i], hk[i], y);
    }
    *reinterpret_cast<f32x4*>(hp + (long)c * N) = hk;
    y = group_sum<Q>(y);
    if (q == 0) {
      y += in.d * x;
      if (p.z) y *= silu_f((float)in.z);
      ((T*)p.out)[(long)t * p.o_stride + c] = (T)y;
    }
  };
  In in[K];
#pragma unroll
  for (int k = 0; k < K; ++k)
    if (AHEAD) in[k] = load(t0, min(c0 + k * CW, p.Ch - 1));
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int c = c0 + k * CW;
    if (c >= p.Ch) break;
    token(t0, c, h[k], AHEAD ? in[k] : load(t0, c));
  }
  // further tokens of a sequence, rare here: each lane's own states again from memory
#pragma unroll 1
  for (int i = K; i < K * L; ++i) {
    const int c = c0 + i % K * CW;
    if (c < p.Ch) token(t0 + i / K, c, *reinterpret_cast<const f32x4*>(hp + (long)c * N), load(t0 + i / K, c));
  }
}

constexpr long SCAN_FEW = 5L << 20;                     // states of a one-token step (20 MB)

// form 1: the sequences have one new token each (none and several are right too); 2: two states a lane (16 of them, a rate each, a step size per
// channel, 32 channels on a boundary of 32 share B and C); 3: eight states a lane (64 of them and more, a rate per head); 0: channels in pairs (the caller checks that pairs share B, C and are aligned).  nchunks > 1: ws_dt [S, nchunks, C] and ws_h [S, nchunks, C, N].
VDA_EXPORT int vda_selective_scan_pairs(void* out, const void* u, const void* delta, const float* A, const void* Bm,
                                        const void* Cm, const float* D, const void* z, const float* delta_bias,
                                        float* ssm_state, const int* qsl, const int* seq_lens, const int* block_table,
                                        long bt_stride, int S, int C, int N, long u_stride, long d_stride, long b_stride,
                                        long c_stride, long z_stride, long o_stride, int dt_div, int a_scalar,
                                        int group_ch, int softplus, int form, int chunk, int nchunks, float* ws_dt,
                                        float* ws_h, int dtype, hipStream_t st) {
  if (S <= 0 || C <= 0) return 0;
  if (N != 16 && N != 32 && N != 64 && N != 128 && N != 256) return -1;
  if (dt_div < 1 || group_ch < 1) return -2;
  const bool step = form == 1, lanes = form == 2, groups = form == 3;
  // (a workgroup's channels: of one head and one group, rows of B and C in pieces of 16 bytes)
  if (groups && ((N != 64 && N != 128 && N != 256) || !a_scalar || C % (2048 / N) || dt_div % (2048 / N) || group_ch % (2048 / N) || b_stride % 8 ||
                 c_stride % 8 || dtype == VDA_F32 || (uintptr_t)Bm % 16 || (uintptr_t)Cm % 16)) return -4;
  if (lanes && (N != 16 || a_scalar || dt_div != 1 || (group_ch < C && group_ch % LN_CH))) return -4;
  const int nl = N / 16, wgch = 512 / nl;
  const int span = min((wgch + group_ch - 1) / group_ch + 1, (C + group_ch - 1) / group_ch);
  if (form == 0 && ((C & 1) || (group_ch & 1) || (dt_div > 1 && (dt_div & 1)) || 2 * N * span > SCAN_LDS)) return -4;
  if (nchunks > 1 && (!ws_dt || !ws_h || chunk < 1)) return -4;
  ScanArgs p{out, u, delta, A, Bm, Cm, D, z, delta_bias, ssm_state, qsl, seq_lens, block_table, bt_stride, u_stride, d_stride,
             b_stride, c_stride, z_stride, o_stride, C, dt_div, group_ch, softplus, chunk, 0, ws_dt, ws_h};
  p.tile = SCAN_LDS / (2 * N * span);
  p.tile = p.tile > 64 ? 64 : p.tile > nl ? p.tile / nl * nl : p.tile;     // (whole blocks of tokens where they fit)
  const dim3 block(256), grid((C + wgch - 1) / wgch, S, nchunks > 1 ? nchunks : 1);
  const bool few = (long)S * C * N < SCAN_FEW;
  const int step_ch = 4 * (few ? 2 : 8) * (256 / N);
  const dim3 grid_step((C + step_ch - 1) / step_ch, S);
  const dim3 grid_carry((unsigned)(((long)C * (N / 4) + 255) / 256), S);
  const long eb = dtype == VDA_F32 ? 4 : 2;
  const auto apart = [&](const void* at, long stride) { return stride % 4 == 0 && (uintptr_t)at % (4 * eb) == 0; };
  const int vec = C % 4 == 0 && apart(u, u_stride) && apart(delta, d_stride) && (!z || apart(z, z_stride)) && apart(out, o_stride);
  const dim3 grid_lanes((C + LN_CH - 1) / LN_CH, S, nchunks > 1 ? nchunks : 1);
#define K2(TT) do {                                                                                                     \
    if (nchunks <= 1) hipLaunchKernelGGL((scan_lanes_kernel<TT, 0>), grid_lanes, block, 0, st, p, vec);                  \
    else {                                                                                                                 \
      hipLaunchKernelGGL((scan_lanes_kernel<TT, 1>), grid_lanes, block, 0, st, p, vec);                                    \
      hipLaunchKernelGGL((scan_carry_kernel<false>), grid_carry, block, 0, st, p, N, nchunks);                             \
      hipLaunchKernelGGL((scan_lanes_kernel<TT, 2>), grid_lanes, block, 0, st, p, vec);                                    \
    } } while (0)
#define K(TT, NN, AA) do {                                                                                              \
    if (step && few) hipLaunchKernelGGL((scan_step_kernel<TT, NN, AA, 2>), grid_step, block, 0, st, p);                    \
    else if (step) hipLaunchKernelGGL((scan_step_kernel<TT, NN, AA, 8>), grid_step, block, 0, st, p);                      \
    else if (nchunks <= 1) hipLaunchKernelGGL((scan_pairs_kernel<TT, NN, 0, AA>), grid, block, 0, st, p);                  \
    else {                                                                                                                 \
      hipLaunchKernelGGL((scan_pairs_kernel<TT, NN, 1, AA>), grid, block, 0, st, p);                                       \
      hipLaunchKernelGGL((scan_carry_kernel<AA>), grid_carry, block, 0, st, p, NN, nchunks);                               \
      hipLaunchKernelGGL((scan_pairs_kernel<TT, NN, 2, AA>), grid, block, 0, st, p);                                       \
    } } while (0)
#define K3(TT, NN) do {                                                                                                    \
    const dim3 grid_groups(C / (2048 / NN), S, nchunks > 1 ? nchunks : 1);                                                 \
    if (nchunks <= 1) hipLaunchKernelGGL((scan_groups_kernel<TT, NN, 0>), grid_groups, block, 0, st, p);                  \
    else {                                                                                                                 \
      hipLaunchKernelGGL((scan_groups_kernel<TT, NN, 1>), grid_groups, block, 0, st, p);                                   \
      hipLaunchKernelGGL((scan_carry_kernel<true>), grid_carry, block, 0, st, p, N, nchunks);                              \
      hipLaunchKernelGGL((scan_groups_kernel<TT, NN, 2>), grid_groups, block, 0, st, p);                                   \
    } } while (0)
#define BYG(TT) do { if (N == 64) K3(TT, 64); else if (N == 128) K3(TT, 128); else K3(TT, 256); } while (0)
  if (groups) {
    if (dtype == VDA_BF16) BYG(bf16_t);
    else BYG(f16_t);
    VDA_CHECK_LAUNCH();
    return 0;
  }
#undef BYG
#undef K3
#define BYA(TT, NN) do { if (a_scalar) K(TT, NN, true); else K(TT, NN, false); } while (0)
#define RUN(TT) do { if (lanes) K2(TT); else if (N == 16) BYA(TT, 16); else if (N == 32) BYA(TT, 32); else if (N == 64) BYA(TT, 64); \
                     else if (N == 128) BYA(TT, 128); else BYA(TT, 256); } while (0)
  if (dtype == VDA_BF16) RUN(bf16_t);
  else if (dtype == VDA_F16) RUN(f16_t);
  else if (dtype == VDA_F32) RUN(float);
  else return -3;
#undef RUN
#undef BYA
#undef K
#undef K2
  VDA_CHECK_LAUNCH();
  return 0;
}

VDA_EXPORT int vda_selective_scan(void* out, const void* u, const void* delta, const float* A, const void* Bm,
                                  const void* Cm, const float* D, const void* z, const float* delta_bias,
                                  float* ssm_state, const int* qsl, const int* seq_lens, const int* block_table,
                                  long bt_stride, int S, int C, int N, long u_stride, long d_stride, long b_stride,
                                  long c_stride, long z_stride, long o_stride, int dt_div, int a_scalar, int group_ch,
                                  int softplus, int chunk, int nchunks, float* ws_p, float* ws_h, int dtype,
                                  hipStream_t st) {
  if (S <= 0 || C <= 0) return 0;
  if (N != 16 && N != 32 && N != 64 && N != 128 && N != 256) return -1;
  if (dt_div < 1 || group_ch < 1) return -2;
  const bool chunked = nchunks > 1;
  if (chunked && (!ws_p || !ws_h || chunk < 1)) return -4;
  const long threads = (long)C * (N / 16);
  dim3 block(256), grid((unsigned)((threads + 255) / 256), S, chunked ? nchunks : 1);
#define L(TT, NN, MODE) hipLaunchKernelGGL((selective_scan_kernel<TT, NN, MODE>), grid, block, 0, st, (TT*)out,             (const TT*)u, (const TT*)delta, A, (const TT*)Bm, (const TT*)Cm, D, (const TT*)z, delta_bias, ssm_state, qsl,           seq_lens, block_table, bt_stride, C, u_stride, d_stride, b_stride, c_stride, z_stride, o_stride, dt_div, a_scalar,      group_ch, softplus, chunk, ws_p, ws_h)
#define BYN(TT, MODE) do { if (N == 16) L(TT, 16, MODE); else if (N == 32) L(TT, 32, MODE);                                    else if (N == 64) L(TT, 64, MODE); else if (N == 128) L(TT, 128, MODE);                             else L(TT, 256, MODE); } while (0)
#define RUN(TT) do {                                                                                                   \
    if (!chunked) { BYN(TT, 0); }                                                                                      \
    else {                                                                                                             \
      BYN(TT, 1);                                                                                                      \
      const long CN = (long)C * N;                                                                                     \
      hipLaunchKernelGGL(scan_combine_kernel, dim3((unsigned)((CN + 255) / 256), S), block, 0, st, ws_p, ws_h,         \
                         ssm_state, qsl, seq_lens, block_table, bt_stride, CN, chunk, nchunks);                        \
      BYN(TT, 2);                                                                                                      \
    } } while (0)
  if (dtype == VDA_BF16) RUN(bf16_t);
  else if (dtype == VDA_F16) RUN(f16_t);
  else if (dtype == VDA_F32) RUN(float);
  else return -3;
#undef RUN
#undef BYN
#undef L
  VDA_CHECK_LAUNCH();
  return 0;
}
