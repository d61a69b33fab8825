// Paged attention for gfx950: decode (split-KV, the 4 waves of a workgroup share
// the query columns and split the keys) and varlen prefill / chunked prefill
// (each wave owns its own query columns) on one MFMA data flow.
//
// Covers what the reference spreads over csrc/rocm/attention.cu (MFMA decode),
// csrc/attention/paged_attention_v{1,2}.cu, the Triton unified_attention kernel
// (vllm/attention/ops/triton_unified_attention.py) and
// csrc/attention/merge_attn_states.cu.
//
// Cache layout (chosen for MFMA operands, see sched/kv_cache_interface.py):
//   K: [num_blocks, kv_heads, BS, D]    a token row is D contiguous elements
//   V: [num_blocks, kv_heads, D, BS]    a d-row is BS contiguous tokens
//
// Data flow per 32-key step, per wave (lane l: r = l&15, g = l>>4):
//   S^T = K . Q^T    A = K rows (token on the MFMA row), B = Q^T (query column r)
//                    -> the lane owns scores of column r for keys 8g..8g+7 of the
//                       step (the two 16-key tiles interleave keys so that this
//                       holds), i.e. softmax statistics are per-lane scalars;
//   O^T += V^T . P^T A = V^T rows (d on the MFMA row, 8 contiguous keys per lane
//                       = one 16-byte load from the V layout above), B = P^T which
//                       is exactly the 8 probabilities the lane already holds.
// Nothing goes through LDS except the final cross-wave merge of the decode form.
#include "attention.h"

// Which sequence and query tokens a prompt's workgroup owns: tiles of sequence s lie in [qsl[s] / q_tile + s, qsl[s + 1] / q_tile
// + s + 1).  The lanes look at 64 sequences at once and hand out what they have read: one trip to memory where a binary
// search makes one for each of its steps and two more.
struct QueryTile { int seq, q0, qs, q_len, seq_len; };
__device__ __forceinline__ QueryTile query_tile(const AttnParams& p, int tile) {
  QueryTile t{0, 0, 0, 0, 0};
  if (p.num_seqs == 1) {             // nothing to look for, and scalar loads are the shorter trip (17 tokens, 32 / 8 heads of 64 6.0 -> 5.8 us)
    t.qs = p.q_start_loc[0];
    t.q_len = p.q_start_loc[1] - t.qs;
    t.seq_len = p.seq_lens[0];
    t.q0 = (tile - t.qs / p.q_tile) * p.q_tile;
    return t;
  }
  const int lane = threadIdx.x & 63;
  for (int base = 0; base < p.num_seqs; base += 64) {
    const int i = min(base + lane, p.num_seqs - 1);
    const int start = p.q_start_loc[i], end = p.q_start_loc[i + 1], len = p.seq_lens[i];
    const int n = __popcll(__ballot(base + lane < p.num_seqs && start / p.q_tile + i <= tile));
    if (n > 0) {
      t.seq = base + n - 1;
      t.qs = __builtin_amdgcn_readlane(start, n - 1);
      t.q_len = __builtin_amdgcn_readlane(end, n - 1) - t.qs;
      t.seq_len = __builtin_amdgcn_readlane(len, n - 1);
    }
    if (n < 64) break;
  }
  t.q0 = (tile - (t.qs / p.q_tile + t.seq)) * p.q_tile;
  return t;
}

// Prompts whose query tiles do not fill the chip: one part of a tile's 32-key steps (vda_prefill_parts says how many there are), whose results attn_reduce_kernel merges.
__device__ __forceinline__ void key_part(const AttnParams& p, int part, int& step_lo, int& step_hi) {
  if (p.nsplit <= 1) return;
  const int per = (max(step_hi - step_lo, 0) + p.nsplit - 1) / p.nsplit;
  step_lo += part * per;
  step_hi = min(step_hi, step_lo + per);
}
// a lane's values 16 n + 4 g of one (token, head), as that part's row and its log2-domain weight
template <int D>
__device__ __forceinline__ void store_part(const AttnParams& p, int part, long tok, int head, int g, const f32x4 (&acc)[D / 16],
                                           float inv, float m, float l) {
  const long at = (tok * p.Hq + head) * p.nsplit + part;
  if (l != 0.f) {                                         // (a part without keys is left out by its weight; one that is NaN is not)
    float* po = p.part_out + at * D + 4 * g;
#pragma unroll
    for (int n = 0; n < D / 16; ++n) *reinterpret_cast<f32x4*>(po + 16 * n) = acc[n] * inv;
  }
  if (g == 0) p.part_lse[at] = l != 0.f ? m + log2f(l) : -INFINITY;
}

template <typename T, int D, int BS, int NCT, bool F8>
__global__ __launch_bounds__(256) void paged_attn_kernel(AttnParams p) {
  using V8 = typename Vec<T>::v8;
  using CT = typename KVElem<T, F8>::type;
  using V4 = typename Vec<T>::v4;
  constexpr int KS = D / 32;       // MFMA k-steps over the head dimension
  constexpr int NT = D / 16;       // 16-wide d tiles of the output
  constexpr int DQ = D / 4;        // d elements owned by one lane group in QK^T
  constexpr int COLS = 16 * NCT;   // query columns per wave
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int kvh = blockIdx.y;
  const int G = p.Hq / p.Hkv;

  const QueryTile own = query_tile(p, blockIdx.x);
  const int seq = own.seq, q0 = own.q0, qs = own.qs, q_len = own.q_len, seq_len = own.seq_len;
  if (q0 >= q_len) return;
  const int ctx = seq_len - q_len;        // keys that precede the first query token
  const int* bt = p.block_table + (long)seq * p.max_blocks;
  const int nblk_valid = (seq_len + BS - 1) / BS;

  // ---- per-lane query columns -------------------------------------------------
  // column c of the workgroup -> (query token c / G, head c % G)
  int limit[NCT], lower[NCT];
  long col_off[NCT];           // element offset of (token, head) in q / out
  float slope[NCT], sink_m[NCT], bfar2[NCT];
  const float* bias_col[NCT];
  V8 qf[NCT][KS];
  int wave_hi = 0, wave_lo = 0x7fffffff;
#pragma unroll
  for (int ct = 0; ct < NCT; ++ct) {
    const int c = wave * COLS + ct * 16 + r;
    const int ti = c / G, h = c % G;
    const int qt = q0 + ti;
    const bool valid = qt < min(q_len, q0 + p.q_tile);
    limit[ct] = valid ? (p.causal ? ctx + qt + 1 : seq_len) : 0;
    lower[ct] = (valid && p.window > 0) ? max(0, limit[ct] - p.window) : 0;
    if (valid && p.chunk > 0) lower[ct] = max(lower[ct], (limit[ct] - 1) / p.chunk * p.chunk);
    const int head = kvh * G + h;
    slope[ct] = (p.alibi && valid) ? p.alibi[head] : 0.f;
    bias_col[ct] = p.dist_bias ? dist_row(p, head) : nullptr;
    bfar2[ct] = (p.dist_bias && valid) ? bias_col[ct][p.dist_far] * 1.4426950408889634f : 0.f;
    // a sink is a score without key or value: the running maximum starts there and the sum with its weight of one
    // (once per column: in the lane group that holds the sum's first part)
    sink_m[ct] = (p.sink && valid) ? p.sink[head] * 1.4426950408889634f : -INFINITY;
    const T* qp = (const T*)p.q + (long)(qs + (valid ? qt : q0)) * p.q_stride + (long)head * D + g * DQ;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      qf[ct][s] = valid ? ld16<V8>(qp + 8 * s) : V8{};
    }
    col_off[ct] = valid ? (long)(qs + qt) : -1;   // token index; -1 = padding column
    if (valid) { wave_hi = max(wave_hi, limit[ct]); wave_lo = min(wave_lo, lower[ct]); }
  }
  // wave-uniform key range
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    wave_hi = max(wave_hi, __shfl_xor(wave_hi, o, 64));
    wave_lo = min(wave_lo, __shfl_xor(wave_lo, o, 64));
  }
  int step_lo = wave_hi > 0 ? wave_lo / 32 : 0, step_hi = (wave_hi + 31) / 32;
  key_part(p, blockIdx.z, step_lo, step_hi);

  float m[NCT], l[NCT];
  f32x4 acc[NCT][NT];
#pragma unroll
  for (int ct = 0; ct < NCT; ++ct) {
    if (blockIdx.z > 0) sink_m[ct] = -INFINITY;           // (a sink joins once)
    m[ct] = sink_m[ct]; l[ct] = (sink_m[ct] != -INFINITY && g == 0) ? 1.f : 0.f;
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[ct][n] = f32x4{0, 0, 0, 0};
  }

  const CT* kc = (const CT*)p.k_cache;
  const CT* vc = (const CT*)p.v_cache;
  const int hkv_v = p.Hkv >> p.v_shift, kvh_v = kvh >> p.v_shift;      // the value head behind this key head
  // K row of this lane inside a step: tile u, row r  <->  key 8*(r>>2) + 4u + (r&3)
  const int krow0 = 8 * (r >> 2) + (r & 3);

  auto load_k = [&](int step, V8 (&kf)[2][KS]) {
    const int tb = step * 32;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int tok = tb + krow0 + 4 * u;
      const int bi = max(min(tok / BS, nblk_valid - 1), 0);
      const long blk = bt[bi];
      const CT* kp = kc + ((blk * p.Hkv + kvh) * BS + (tok % BS)) * (long)D + g * DQ;
#pragma unroll
      for (int s = 0; s < KS; ++s) kf[u][s] = KVLoad<T, F8>::ld(kp + 8 * s);
    }
  };
  auto load_v = [&](int step, V8 (&vf)[NT]) {
    const int tok = step * 32 + 8 * g;
    const int bi = max(min(tok / BS, nblk_valid - 1), 0);
    const long blk = bt[bi];
    const CT* vp = vc + ((blk * hkv_v + kvh_v) * (long)D + r) * BS + (tok % BS);
#pragma unroll
    for (int n = 0; n < NT; ++n) vf[n] = KVLoad<T, F8>::ld(vp + (long)n * 16 * BS);
  };

  V8 kf[2][KS], kn[2][KS], vf[NT];
  if (step_lo < step_hi) load_k(step_lo, kf);
  for (int step = step_lo; step < step_hi; ++step) {
    load_v(step, vf);
    const int nxt = step + 1;
    if (nxt < step_hi) load_k(nxt, kn);
    const int tb = step * 32 + 8 * g;   // first key of this lane's 8
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct) {
      f32x4 s0 = {0, 0, 0, 0}, s1 = {0, 0, 0, 0};
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        s0 = mfma16(kf[0][s], qf[ct][s], s0);
        s1 = mfma16(kf[1][s], qf[ct][s], s1);
      }
      float sv[8] = {s0[0], s0[1], s0[2], s0[3], s1[0], s1[1], s1[2], s1[3]};
      float mx = -INFINITY;
      float bj[8] = {0, 0, 0, 0, 0, 0, 0, 0};         // key tb + j sits limit - 1 - tb - j behind the query
      if (p.dist_bias) {
        const int d_lo = limit[ct] - 1 - (tb + 7);
        const f32x4 b0 = dist_bias4(bias_col[ct], d_lo, p.dist_far), b1 = dist_bias4(bias_col[ct], d_lo + 4, p.dist_far);
        bj[7] = b0[0]; bj[6] = b0[1]; bj[5] = b0[2]; bj[4] = b0[3];
        bj[3] = b1[0]; bj[2] = b1[1]; bj[1] = b1[2]; bj[0] = b1[3];
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int tok = tb + j;
        float x = sv[j] * p.scale;
        if (p.softcap > 0.f) x = p.softcap * fast_tanh(x / p.softcap);
        x += slope[ct] * (float)(tok - (limit[ct] - 1));
        x += bj[j];
        x *= 1.4426950408889634f;
        x = (tok < limit[ct] && tok >= lower[ct]) ? x : -INFINITY;
        sv[j] = x;
        mx = fmaxf(mx, x);
      }
      mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      const float m_new = fmaxf(m[ct], mx);
      const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
      const float alpha = fexp2(m[ct] - m_use);
      m[ct] = m_new;
      float ps = 0.f;
      V8 pb;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float e = fexp2(sv[j] - m_use);
        ps += e;
        pb[j] = (T)e;
      }
      l[ct] = l[ct] * alpha + ps;
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        acc[ct][n] *= alpha;
        acc[ct][n] = mfma16(vf[n], pb, acc[ct][n]);
      }
    }
    if (nxt < step_hi) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int s = 0; s < KS; ++s) kf[u][s] = kn[u][s];
    }
  }

  // lane-partial row sums -> full sums
#pragma unroll
  for (int ct = 0; ct < NCT; ++ct) {
    l[ct] += __shfl_xor(l[ct], 16, 64);
    l[ct] += __shfl_xor(l[ct], 32, 64);
  }

#pragma unroll
  for (int ct = 0; ct < NCT; ++ct) {
    if (col_off[ct] < 0) continue;
    const int c = wave * COLS + ct * 16 + r;
    const int head = kvh * G + c % G;
    const float inv = l[ct] > 0.f ? p.v_scale / l[ct] : 0.f;
    if (p.nsplit > 1) {
      store_part<D>(p, blockIdx.z, col_off[ct], head, g, acc[ct], inv, m[ct], l[ct]);
      continue;
    }
    T* op = (T*)p.out + col_off[ct] * p.out_stride + (long)head * D + 4 * g;
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      V4 o;
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = (T)(acc[ct][n][i] * inv);
      *reinterpret_cast<V4*>(op + 16 * n) = o;
    }
    if (p.lse_out && g == 0)
      p.lse_out[(long)head * p.num_tokens + col_off[ct]] =
          l[ct] > 0.f ? (m[ct] + log2f(l[ct])) * 0.6931471805599453f : -INFINITY;
  }
}

// a product that is rounded by itself
__device__ __forceinline__ float rounded(float v) {
  asm("" : "+v"(v));
  return v;
}

// Decode: a workgroup per (sequence, kv head, part of the keys); its waves share the query columns and split the keys.
//
// Memory is all there is to do: each key and value byte is read once, so what counts is bytes in flight.  A step is as many
// keys as give every lane 16 bytes of a value row: 32 of a 16-bit cache, 64 of an e4m3 one (RUN keys in a row per lane group;
// the 16-key MFMA tiles take keys RUN g + 4 u + i, so that the products' operands are what the lane loaded).  Rows stay raw in
// registers until the product takes them: the next step's keys are requested as soon as the scores have used this step's, its
// values as soon as the outputs have, and page numbers a step before that, so that no load waits for another.  Few short sequences are a
// chain of trips instead: in one part and without a window the first steps' pages are asked for together with the lengths, and eight
// waves hold two steps each.
//
// What it measured (us, before -> after): 183 sequences of 525 .. 3675 keys, 64 / 8 heads of 128, e4m3 cache 257 -> 148 (5.3 TB/s),
// 16-bit 310 -> 271; 256 of 1100, 64 / 8 heads, e4m3 160 -> 113, 16-bit 206 -> 200 (5.8 TB/s), of 300 keys 70 -> 64; 64 of
// 500 .. 3500, 16 / 8 heads of 256 308 -> 203.  Before the pages came ahead and the waves' sums met in one step -> since, attention alone in
// a graph: 256 of some 40 keys, 32 / 8 heads, 22.4 -> 16.4, of 300 64.7 -> 58.8, 40 of 900 32.5 -> 31.6, four tokens each of 16 on 1000 24.4 -> 22.6; ten of 46, 16 / 8
// heads of 256, 7.6 -> 6.4, 64 of 2000 198.5 -> 195.6 (193 with four lanes' pieces of a key row one behind another, whose products add in
// another order: results keep their bits instead).  A CU takes in 31 bytes a cycle at
// most: 675 keys of one head are 11000 cycles of the launch's 24000.  Of the first, 203 without the order of sequences below; held to the 168 registers of three
// waves per SIMD it spills 15 and takes 177.  Non-temporal loads: e4m3 rows 6 % faster, 16-bit ones, of which a lane's pieces share
// lines, up to 60 % slower.
constexpr unsigned DECODE_RANKED = 512;    // two workgroups per CU are resident
constexpr int DECODE_APART = 256;          // keys
// WAVES: four, or eight where few sequences of few keys are asked for in two parts of four waves: the waves of one workgroup
// do what the parts would, and their sums meet in LDS instead of in memory and another launch.  Five of some 390 keys, 32 / 8 heads of
// 128, with rotation and cache write: 20.0 -> 16.5 us as single calls when it came; of 96 values 12.5 -> 10.8 in a graph, e4m3 14.4 -> 12.2.  Three
// and four parts in eight waves: 15.2 -> 17.0 and 14.8 -> 18.8 in a graph.
template <typename T, int D, int BS, int NCT, bool F8, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void paged_decode_kernel(AttnParams p) {
  using V8 = typename Vec<T>::v8;
  using CT = typename KVElem<T, F8>::type;
  using V4 = typename Vec<T>::v4;
  constexpr int KS = D / 32;       // MFMA k-steps over the head dimension
  constexpr int NT = D / 16;       // 16-wide d tiles of the output
  constexpr int PIECE = 16 / (int)sizeof(CT);        // d elements of 16 bytes
  constexpr int HS = F8 ? 2 : 1;   // 32-key halves of a step
  constexpr int RUN = 8 * HS, KEYS = 32 * HS;
  constexpr int DQ = D / 4;        // d elements owned by one lane group in QK^T
  constexpr int KB = D / (4 * PIECE);                // pieces of a key row per lane
  constexpr int COLS = 16 * NCT;   // query columns
  constexpr int DEPTH = WAVES == 8 && D <= 128 ? 2 : 1;      // steps whose rows a wave holds (registers of two waves a SIMD)
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  // Workgroup -> (sequence, part, kv head), heads fastest.  A grid larger than the chip holds takes its sequences longest
  // first: a long one that starts last would run alone.  Every wave finds its own, the blockIdx.z-th largest of the lengths,
  // bit by bit: no barrier, and no more than some 25 dependent counts before the first key (counting ranks over LDS took
  // 256 of 300 keys, 64 / 8 heads, from 70 to 90 us).  Lengths within an eighth or 256 keys of the first one's stay in their order: a
  // workgroup of few keys costs less than looking for it (250 of 12 .. 87 keys, 32 / 8 heads, 31.5 us in order of length, 28.4 in the
  // batch's; e4m3 33.4 / 30.2).
  const int kvh = blockIdx.x, part = blockIdx.y;
  int seq = blockIdx.z;
  // (the pages of the first steps, asked for in the same trip; load_k and load_v below read them)
  int page_k[DEPTH], page_v[DEPTH];
  auto pages_ahead = [&] {
    if (p.table_cols <= 0) return;
    const int* row = p.block_table + (long)seq * p.max_blocks;
#pragma unroll
    for (int i = 0; i < DEPTH; ++i) {
      const int st = wave + i * WAVES;
      page_k[i] = row[min((st * KEYS + RUN * (r >> 2)) / BS, p.table_cols - 1)];
      page_v[i] = row[min((st * KEYS + RUN * g) / BS, p.table_cols - 1)];
    }
  };
  int qs = p.q_start_loc[seq], q_end = p.q_start_loc[seq + 1], seq_len = p.seq_lens[seq];
  pages_ahead();
  if (gridDim.x * gridDim.y * gridDim.z > DECODE_RANKED && p.num_seqs <= 256) {
    const int base = p.seq_lens[0], bits = min(32 - __clz(p.max_blocks * BS), 22);
    int key[4];                                         // length, then the first of the batch; no two alike
    bool differs = false;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int at = lane + 64 * i, len = p.seq_lens[min(at, p.num_seqs - 1)];
      differs |= abs(len - base) > max(base >> 3, DECODE_APART);
      key[i] = at < p.num_seqs ? min(max(len, 0), (1 << bits) - 1) << 8 | (255 - at) : -1;
    }
    if (__any(differs)) {
      int found = 0;                                    // the largest number that more than blockIdx.z keys reach
      for (int bit = bits + 7; bit >= 0; --bit) {
        const int next = found | 1 << bit;
        int reach = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) reach += __popcll(__ballot(key[i] >= next));
        if (reach > (int)blockIdx.z) found = next;
      }
      seq = 255 - (found & 255);
      qs = p.q_start_loc[seq]; q_end = p.q_start_loc[seq + 1]; seq_len = p.seq_lens[seq];
      pages_ahead();
    }
  }
  const int G = p.Hq / p.Hkv;
  const int q_len = q_end - qs;
  if (q_len <= 0) return;
  const int ctx = seq_len - q_len;        // keys that precede the first query token
  const int* bt = p.block_table + (long)seq * p.max_blocks;

  // ---- per-lane query columns: column c -> (query token c / G, head c % G) ----
  int limit[NCT], lower[NCT];
  long col_off[NCT];           // token index, -1 = padding column
  float slope[NCT], sink_m[NCT];
  const float* bias_col[NCT];
  V8 qf[NCT][KS];
  int wave_hi = 0, wave_lo = 0x7fffffff, full_hi = 0x7fffffff, full_lo = 0;
#pragma unroll
  for (int ct = 0; ct < NCT; ++ct) {
    const int c = ct * 16 + r, ti = c / G, h = c % G;
    const bool valid = ti < q_len && c < COLS;
    limit[ct] = valid ? (p.causal ? ctx + ti + 1 : seq_len) : 0;
    lower[ct] = (valid && p.window > 0) ? max(0, limit[ct] - p.window) : 0;
    if (valid && p.chunk > 0) lower[ct] = max(lower[ct], (limit[ct] - 1) / p.chunk * p.chunk);
    const int head = kvh * G + h;
    slope[ct] = (p.alibi && valid) ? p.alibi[head] : 0.f;
    bias_col[ct] = p.dist_bias ? dist_row(p, head) : nullptr;
    // a sink is a score without key or value: the running maximum starts there and the sum with its weight of one, once
    // per column: in one lane group of one wave of one part
    sink_m[ct] = (p.sink && valid && wave == 0 && part == 0) ? p.sink[head] * 1.4426950408889634f : -INFINITY;
    const T* qp = (const T*)p.q + (long)(qs + (valid ? ti : 0)) * p.q_stride + (long)head * D + g * DQ;
#pragma unroll
    for (int s = 0; s < KS; ++s) qf[ct][s] = valid ? ld16<V8>(qp + 8 * s) : V8{};
    col_off[ct] = valid ? (long)(qs + ti) : -1;
    if (valid) {
      wave_hi = max(wave_hi, limit[ct]); wave_lo = min(wave_lo, lower[ct]);
      full_hi = min(full_hi, limit[ct]); full_lo = max(full_lo, lower[ct]);
    }
  }
  if (q_len > 1) {                                      // (the columns of one token see the same keys)
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) {
      wave_hi = max(wave_hi, __shfl_xor(wave_hi, o, 64));
      wave_lo = min(wave_lo, __shfl_xor(wave_lo, o, 64));
      full_hi = min(full_hi, __shfl_xor(full_hi, o, 64));
      full_lo = max(full_lo, __shfl_xor(full_lo, o, 64));
    }
  }
  wave_hi = __builtin_amdgcn_readfirstlane(wave_hi);
  wave_lo = __builtin_amdgcn_readfirstlane(wave_lo);
  full_hi = __builtin_amdgcn_readfirstlane(full_hi);
  full_lo = __builtin_amdgcn_readfirstlane(full_lo);
  // the parts of the steps over gridDim.z, a part's steps dealt to the waves
  int step = wave_hi > 0 ? wave_lo / KEYS : 0, step_hi = (wave_hi + KEYS - 1) / KEYS;
  {
    const int per = (step_hi - step + p.nsplit - 1) / p.nsplit;
    step += part * per;
    step_hi = min(step_hi, step + per);
    step += __builtin_amdgcn_readfirstlane(wave);
  }

  float m[NCT], l[NCT];
  f32x4 acc[NCT][NT];
#pragma unroll
  for (int ct = 0; ct < NCT; ++ct) {
    m[ct] = sink_m[ct]; l[ct] = (sink_m[ct] != -INFINITY && g == 0) ? 1.f : 0.f;
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[ct][n] = f32x4{0, 0, 0, 0};
  }

  const CT* kc = (const CT*)p.k_cache;
  const CT* vc = (const CT*)p.v_cache;
  const int hkv_v = p.Hkv >> p.v_shift, kvh_v = kvh >> p.v_shift;      // the value head behind this key head
  const int page_lo = wave_lo / BS, page_hi = max((seq_len + BS - 1) / BS - 1, 0);
  u32x4 kr[DEPTH][HS][2][KB], vr[DEPTH][NT];
  int knext, vnext;                                     // pages of the step that is asked for next
  auto page_at = [&](int tok) { return bt[max(min(tok / BS, page_hi), page_lo)]; };
  auto load_k = [&](int i, int st, int page) {          // half h, tile u, row r: key RUN (r / 4) + 8 h + 4 u + r % 4 of the step
    const int tok = st * KEYS + RUN * (r >> 2) + (r & 3);
    const CT* kp = kc + (((long)page * p.Hkv + kvh) * BS + tok % BS) * (long)D + g * DQ;
#pragma unroll
    for (int h = 0; h < HS; ++h)
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int b = 0; b < KB; ++b)
          kr[i][h][u][b] = *reinterpret_cast<const u32x4*>(kp + (8 * h + 4 * u) * D + b * PIECE);
  };
  auto load_v = [&](int i, int st, int page) {
    const int tok = st * KEYS + RUN * g;
    const CT* vp = vc + (((long)page * hkv_v + kvh_v) * (long)D + r) * BS + tok % BS;
#pragma unroll
    for (int n = 0; n < NT; ++n) vr[i][n] = *reinterpret_cast<const u32x4*>(vp + n * 16 * BS);
  };
  auto operand = [](const u32x4& raw, int half) {      // 8 values: all of a 16-bit piece, one half of an e4m3 piece
    if constexpr (F8) return KVLoad<T, true>::widen(u32x2{raw[2 * half], raw[2 * half + 1]});
    else return __builtin_bit_cast(V8, raw);
  };

  const bool plain = !(p.softcap > 0.f) && p.alibi == nullptr && p.dist_bias == nullptr;
  const float sl2 = p.scale * 1.4426950408889634f;
  auto pages = [&](int st) {
    knext = page_at(st * KEYS + RUN * (r >> 2));
    vnext = page_at(st * KEYS + RUN * g);
  };
#pragma unroll
  for (int i = 0; i < DEPTH; ++i) {
    const int st = step + i * WAVES;
    if (st >= step_hi) break;
    if (p.table_cols > 0) {
      // What was read past the sequence's last page is nobody's: those keys, which are masked, are read in the step's first page
      const int k0 = __builtin_amdgcn_readlane(page_k[i], 0), v0 = __builtin_amdgcn_readlane(page_v[i], 0);
      knext = (st * KEYS + RUN * (r >> 2)) / BS <= page_hi ? page_k[i] : k0;
      vnext = (st * KEYS + RUN * g) / BS <= page_hi ? page_v[i] : v0;
    } else {
      pages(st);
    }
    load_k(i, st, knext);
    load_v(i, st, vnext);
  }
  if (step + DEPTH * WAVES < step_hi) pages(step + DEPTH * WAVES);
  auto work = [&](int i, int step) {
    f32x4 s[NCT][HS][2];
#pragma unroll
    for (int h = 0; h < HS; ++h)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
#pragma unroll
        for (int ct = 0; ct < NCT; ++ct) s[ct][h][u] = f32x4{0, 0, 0, 0};
#pragma unroll
        for (int k = 0; k < KS; ++k) {
          const V8 a = operand(kr[i][h][u][k / HS], k % HS);
#pragma unroll
          for (int ct = 0; ct < NCT; ++ct) s[ct][h][u] = mfma16(a, qf[ct][k], s[ct][h][u]);
        }
      }
    const int ahead = step + DEPTH * WAVES;             // takes this step's place
    int vpage = vnext;
    if (ahead < step_hi) {
      load_k(i, ahead, knext);
      if (ahead + WAVES < step_hi) pages(ahead + WAVES);
    }
    __builtin_amdgcn_sched_barrier(0);
    const int tb = step * KEYS + RUN * g;               // first key of this lane's
    const bool whole = plain && step * KEYS + KEYS <= full_hi && step * KEYS >= full_lo;
    V8 pb[NCT][HS];
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct) {
      float mx = -INFINITY;
      if (whole) {
#pragma unroll
        for (int j = 0; j < RUN; ++j) {
          const float x = s[ct][j >> 3][(j >> 2) & 1][j & 3] * sl2;
          s[ct][j >> 3][(j >> 2) & 1][j & 3] = x;
          mx = fmaxf(mx, x);
        }
      } else {
#pragma unroll
        for (int h = 0; h < HS; ++h) {
          float bj[8] = {0, 0, 0, 0, 0, 0, 0, 0};      // key tb + 8 h + j sits limit - 1 - tb - 8 h - j behind the query
          if (p.dist_bias) {
            const int d_lo = limit[ct] - 1 - (tb + 8 * h + 7);
            const f32x4 b0 = dist_bias4(bias_col[ct], d_lo, p.dist_far), b1 = dist_bias4(bias_col[ct], d_lo + 4, p.dist_far);
            bj[7] = b0[0]; bj[6] = b0[1]; bj[5] = b0[2]; bj[4] = b0[3];
            bj[3] = b1[0]; bj[2] = b1[1]; bj[1] = b1[2]; bj[0] = b1[3];
          }
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const int tok = tb + 8 * h + j;
            float x = s[ct][h][j >> 2][j & 3] * p.scale;
            if (p.softcap > 0.f) x = p.softcap * fast_tanh(x / p.softcap);
            x += slope[ct] * (float)(tok - (limit[ct] - 1));
            x += bj[j];
            x *= 1.4426950408889634f;
            x = (tok < limit[ct] && tok >= lower[ct]) ? x : -INFINITY;
            s[ct][h][j >> 2][j & 3] = x;
            mx = fmaxf(mx, x);
          }
        }
      }
      mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      const float m_new = fmaxf(m[ct], mx);
      const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
      const float alpha = fexp2(m[ct] - m_use);
      m[ct] = m_new;
      float ps = 0.f;
#pragma unroll
      for (int j = 0; j < RUN; ++j) {
        const float e = fexp2(s[ct][j >> 3][(j >> 2) & 1][j & 3] - m_use);
        ps += e;
        pb[ct][j >> 3][j & 7] = (T)e;
      }
      l[ct] = l[ct] * alpha + ps;
      if (__any(alpha != 1.f)) {
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[ct][n] *= alpha;
      }
    }
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int h = 0; h < HS; ++h) {
        const V8 a = operand(vr[i][n], h);
#pragma unroll
        for (int ct = 0; ct < NCT; ++ct) acc[ct][n] = mfma16(a, pb[ct][h], acc[ct][n]);
      }
    __builtin_amdgcn_sched_barrier(0);
    if (ahead < step_hi) load_v(i, ahead, vpage);
  };
  for (; step < step_hi; step += DEPTH * WAVES) {
    work(0, step);
    if constexpr (DEPTH == 2)
      if (step + WAVES < step_hi) work(1, step + WAVES);
  }

  // lane-partial row sums -> full sums
#pragma unroll
  for (int ct = 0; ct < NCT; ++ct) {
    l[ct] += __shfl_xor(l[ct], 16, 64);
    l[ct] += __shfl_xor(l[ct], 32, 64);
  }
  // ---- merge the waves: their sums meet in LDS, and every thread joins four values of a column over the waves --------
  // (rows of D + 4: a lane's 16 bytes lie a bank group beside its neighbours'.  They add as a tree over halves of the waves, each level of
  // which was two barriers; which product is rounded and which joins the sum unrounded is part of the result's bits)
  constexpr int ROW = D + 4;
  __shared__ __attribute__((aligned(16))) float s_acc[WAVES][COLS][ROW];
  __shared__ float s_m[COLS][WAVES], s_l[COLS][WAVES];
#pragma unroll
  for (int ct = 0; ct < NCT; ++ct) {
    if (col_off[ct] < 0) continue;
    const int c = ct * 16 + r;
#pragma unroll
    for (int n = 0; n < NT; ++n) *reinterpret_cast<f32x4*>(&s_acc[wave][c][16 * n + 4 * g]) = acc[ct][n];
    if (g == 0) { s_m[c][wave] = m[ct]; s_l[c][wave] = l[ct]; }
  }
  __syncthreads();
  const int columns = min(q_len * G, COLS);
  for (int item = threadIdx.x; item < columns * (D / 4); item += 64 * WAVES) {
    const int c = item / (D / 4), d = 4 * (item % (D / 4));
    float ms[WAVES], ls[WAVES];
    f32x4 os[WAVES];
#pragma unroll
    for (int w = 0; w < WAVES; ++w) { ms[w] = s_m[c][w]; ls[w] = s_l[c][w]; os[w] = *reinterpret_cast<const f32x4*>(&s_acc[w][c][d]); }
#pragma unroll
    for (int cnt = WAVES / 2; cnt > 0; cnt >>= 1)
#pragma unroll
      for (int w = 0; w < cnt; ++w) {
        const float M = fmaxf(ms[w], ms[w + cnt]), Mu = (M == -INFINITY) ? 0.f : M;
        const float f1 = fexp2(ms[w] - Mu), f2 = fexp2(ms[w + cnt] - Mu);
        ls[w] = fmaf(ls[w], f1, rounded(ls[w + cnt] * f2));
        ms[w] = M;
#pragma unroll
        for (int j = 0; j < 4; ++j) os[w][j] = fmaf(os[w + cnt][j], f2, rounded(os[w][j] * f1));
      }
    const float L = ls[0], Mu = ms[0] == -INFINITY ? 0.f : ms[0];
    f32x4 o = os[0];
    o *= L > 0.f ? p.v_scale / L : 0.f;
    const int head = kvh * G + c % G;
    const long token = qs + c / G;
    if (p.nsplit == 1) {
      V4 to;
#pragma unroll
      for (int i = 0; i < 4; ++i) to[i] = (T)o[i];
      *reinterpret_cast<V4*>((T*)p.out + token * p.out_stride + (long)head * D + d) = to;
    } else {
      const long pi = (token * p.Hq + head) * p.nsplit + part;
      *reinterpret_cast<f32x4*>(p.part_out + pi * D + d) = o;
      if (d == 0) p.part_lse[pi] = L > 0.f ? Mu + log2f(L) : -INFINITY;
    }
  }
}

// Prefill form with K/V staged through LDS.  The direct-to-register form above (head groups of more queries than a workgroup has columns here) makes every wave of a
// workgroup fetch the same keys from L2 (4x the traffic) and is L2-bandwidth bound in prefill; here the
// 256 threads copy each 32-key K tile and V tile once (fully coalesced 16-byte pieces, fp8 caches are
// widened on the way in), double-buffered so that the next tile's global loads fly during the MFMAs, and
// every wave then reads its MFMA operands from LDS.  16-byte pieces are XOR-swizzled so that the eight
// lanes served per LDS cycle hit eight different bank groups for both the row-per-lane K reads and the
// d-row-per-lane V reads.
#ifndef PREFILL_WGS_PER_CU
#define PREFILL_WGS_PER_CU 2
#endif
//
// SPARSE: vertical-slash selection for very long prompts.  A workgroup serves 128 query rows of ONE head (the
// selection is per head, so the rows of a GQA group no longer share their keys) and visits only the 32-key steps that
// hold a selected key position or that a selected diagonal crosses inside its rows; it marks them in an LDS bitmap
// built from the two lists when it starts (no index arrays in memory: the reference's block_offset / column_index,
// csrc/attention/vertical_slash_index.cu:26-150, grow with rows x list length) and walks the set bits in order.
// Inside a visited step every key is seen (subject to the causal limit), so the pattern is a superset of the exact
// lines at 32-key granularity.
constexpr int SPARSE_BM_WORDS = 4096;        // 4096 x 32 steps x 32 keys = 4 Mi keys per table
// Query columns of a workgroup: 32 a wave, or 16 where the outputs and the queries of more would not fit the registers of two
// workgroups a CU.  Heads of 96, 192 and 256 values took the direct form before: us, eight prompts of some 1000, 16 / 8 heads of 256 535 -> 308,
// 24 / 8 of 96 255 -> 196; four of 300 78 -> 54 and 49 -> 41.
template <int D> constexpr int PREFILL_COLS = D <= 128 ? 128 : 64;
template <typename T, int D, int BS, bool F8, bool SPARSE = false>
__global__ __launch_bounds__(256, PREFILL_WGS_PER_CU) void paged_prefill_lds_kernel(AttnParams p, SparseSel sp) {
  using V8 = typename Vec<T>::v8;
  using V4 = typename Vec<T>::v4;
  using CT = typename KVElem<T, F8>::type;
  constexpr int KS = D / 32, NT = D / 16, DQ = D / 4, NCT = PREFILL_COLS<D> / 64, COLS = 16 * NCT;
  constexpr int KCH = D / 8;          // 16-byte pieces per K row
  constexpr bool XOR = (KCH & (KCH - 1)) == 0;
  constexpr int KROW = XOR ? KCH : KCH + 1;     // pieces between two rows: swizzled ones, or an odd number
  constexpr int KP = 32 * KCH;        // K pieces per 32-key step
  constexpr int VP = D * 4;           // V pieces per step (D rows x 4 groups of 8 keys)
  constexpr int KPT = (KP + 255) / 256, VPT = (VP + 255) / 256;
  static_assert(D % 32 == 0, "head sizes are multiples of an MFMA step");
  __shared__ V8 sK[2][32 * KROW];
  __shared__ V8 sV[2][VP];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int G = SPARSE ? 1 : p.Hq / p.Hkv;
  // The tiles of one kv head's part read the same keys: neighbouring items of one XCD (workgroups are dealt to the eight in
  // turn), whose L2 then serves them, the longest tiles of a prompt first (us, tiles over all XCDs -> this: eight prompts of some
  // 1000, 16 / 8 heads of 256 308 -> 268, 24 / 8 of 96 196 -> 167, 32 / 8 of 64 141 -> 128; 25 new tokens on 3000 of two, 64 / 8 of
  // 128, 70 -> 45).  Four groups of few prompts share their two XCDs tile by tile (28 / 4 heads of 128, one of 4000 275 -> 186, three of 1500
  // 127 -> 108, 16 / 4 of 192 293 -> 180); many prompts, few tiles and fewer groups are even enough in runs, and stay in their L2 (eight of
  // 1000, dealt by tiles 118 -> 131, two groups 85 -> 116; one of 300, 17 tiles, 21.9 -> 22.6).
  int tile = blockIdx.x, part = 0, kvh = SPARSE ? blockIdx.y / (p.Hq / p.Hkv) : blockIdx.y;
  if constexpr (!SPARSE) {
    const int tiles = gridDim.x, groups = gridDim.y * gridDim.z, n = tiles * groups;
    const int id = blockIdx.x + tiles * (blockIdx.y + gridDim.y * blockIdx.z), x = id & 7;
    int group, at;
    if (groups == 4 && p.num_seqs <= 3 && tiles >= 48) {  // two XCDs a group: its tiles in turn, or one of them has all of the longest
      group = x & 3;
      at = (id >> 3) * 2 + (x >> 2);
    } else {
      const int more = n & 7, item = x * (n >> 3) + min(x, more) + (id >> 3);
      group = item / tiles;
      at = item - group * tiles;
    }
    tile = tiles - 1 - at;
    kvh = group % (int)gridDim.y;
    part = group / (int)gridDim.y;
  }
  const int head0 = SPARSE ? blockIdx.y : kvh * G;        // first query head of this workgroup's columns

  const QueryTile own = query_tile(p, tile);
  const int seq = own.seq, q0 = own.q0, qs = own.qs, q_len = own.q_len, seq_len = own.seq_len;
  if (q0 >= q_len) return;                  // uniform over the workgroup
  const int ctx = seq_len - q_len;
  const int* bt = p.block_table + (long)seq * p.max_blocks;
  const int nblk_valid = (seq_len + BS - 1) / BS;
  const int qt_end = min(q_len, q0 + p.q_tile);

  int limit[NCT], lower[NCT];
  long col_off[NCT];
  float slope[NCT], sink_m[NCT], bfar2[NCT];
  const float* bias_col[NCT];
  V8 qf[NCT][KS];
  int wave_hi = 0, wave_lo = 0x7fffffff;
#pragma unroll
  for (int ct = 0; ct < NCT; ++ct) {
    const int c = wave * COLS + ct * 16 + r;
    const int ti = c / G, h = c % G;
    const int qt = q0 + ti;
    const bool valid = qt < qt_end;
    limit[ct] = valid ? (p.causal ? ctx + qt + 1 : seq_len) : 0;
    lower[ct] = (valid && p.window > 0) ? max(0, limit[ct] - p.window) : 0;
    if (valid && p.chunk > 0) lower[ct] = max(lower[ct], (limit[ct] - 1) / p.chunk * p.chunk);
    const int head = head0 + h;
    slope[ct] = (p.alibi && valid) ? p.alibi[head] : 0.f;
    bias_col[ct] = p.dist_bias ? dist_row(p, head) : nullptr;
    bfar2[ct] = (p.dist_bias && valid) ? bias_col[ct][p.dist_far] * 1.4426950408889634f : 0.f;
    sink_m[ct] = (p.sink && valid) ? p.sink[head] * 1.4426950408889634f : -INFINITY;
    const T* qp = (const T*)p.q + (long)(qs + (valid ? qt : q0)) * p.q_stride + (long)head * D + g * DQ;
#pragma unroll
    for (int s = 0; s < KS; ++s) qf[ct][s] = valid ? ld16<V8>(qp + 8 * s) : V8{};
    col_off[ct] = valid ? (long)(qs + qt) : -1;
    if (valid) { wave_hi = max(wave_hi, limit[ct]); wave_lo = min(wave_lo, lower[ct]); }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    wave_hi = max(wave_hi, __shfl_xor(wave_hi, o, 64));
    wave_lo = min(wave_lo, __shfl_xor(wave_lo, o, 64));
  }
  // workgroup-uniform key range (all waves take part in every tile copy)
  const int wg_hi = p.causal ? ctx + qt_end : seq_len;
  int wg_lo = p.window > 0 ? max(0, ctx + q0 + 1 - p.window) : 0;
  if (p.chunk > 0 && p.causal) wg_lo = max(wg_lo, (ctx + q0) / p.chunk * p.chunk);
  int step_lo = wg_lo / 32, step_hi = (wg_hi + 31) / 32;
  if constexpr (!SPARSE) {
    key_part(p, part, step_lo, step_hi);
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct) sink_m[ct] = part > 0 ? -INFINITY : sink_m[ct];   // (a sink joins once)
  }

  __shared__ unsigned bm[SPARSE ? SPARSE_BM_WORDS : 1];
  if constexpr (SPARSE) {
    const int nwords = (step_hi + 31) >> 5;
    for (int i = tid; i < nwords; i += 256) bm[i] = 0u;
    __syncthreads();
    auto mark = [&](int a, int b) {            // steps of the keys a..b of this table (clipped to what is visible)
      a = max(a, 0); b = min(b, wg_hi - 1);
      for (int s = a >> 5; a <= b && s <= (b >> 5); ++s) atomicOr(&bm[s >> 5], 1u << (s & 31));
    };
    const long sh = (long)seq * p.Hq + head0;
    const int kb = sp.key_base[seq];
    const int qa0 = sp.q_base[seq] + q0 - kb, qa1 = sp.q_base[seq] + qt_end - 1 - kb;
    const int nv = min(sp.vcount[sh], sp.NV), ns = min(sp.scount[sh], sp.NS);
    for (int i = tid; i < nv; i += 256) { const int k = sp.vert[sh * sp.NV + i] - kb; mark(k, k); }
    for (int i = tid; i < ns; i += 256) { const int d = sp.slash[sh * sp.NS + i]; if (d >= 0) mark(qa0 - d, qa1 - d); }
    if (p.causal && tid == 0) mark(qa0, qa1);              // a row always sees itself
    __syncthreads();
  }
  // first step >= from that is to be visited (step_hi: none)
  auto next_step = [&](int from) -> int {
    if constexpr (!SPARSE) return from;
    if (from >= step_hi) return step_hi;
    int w = from >> 5;
    const int nwords = (step_hi + 31) >> 5;
    unsigned x = bm[w] & (~0u << (from & 31));
    while (!x) { if (++w >= nwords) return step_hi; x = bm[w]; }
    return min(step_hi, (w << 5) + __ffs(x) - 1);
  };

  float m[NCT], l[NCT];
  f32x4 acc[NCT][NT];
#pragma unroll
  for (int ct = 0; ct < NCT; ++ct) {
    m[ct] = sink_m[ct]; l[ct] = (sink_m[ct] != -INFINITY && g == 0) ? 1.f : 0.f;
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[ct][n] = f32x4{0, 0, 0, 0};
  }
  const CT* kc = (const CT*)p.k_cache;
  const CT* vc = (const CT*)p.v_cache;

  V8 rk[KPT], rv[VPT];
  unsigned pk[KPT], pv[VPT];                    // page numbers, asked for a tile before what lies in the pages
  // Address arithmetic kept in 32 bits except for the one block-number x block-stride product (a single
  // v_mad_u64_u32): offsets inside a block fit 32 bits by construction.
  const unsigned blk_stride = (unsigned)p.Hkv * BS * D;          // elements per K cache block
  const unsigned v_blk_stride = (unsigned)(p.Hkv >> p.v_shift) * D * BS;     // per V cache block (fewer heads when shared)
  const unsigned k_head = (unsigned)kvh * BS * D, v_head = (unsigned)(kvh >> p.v_shift) * D * BS;
  auto pages = [&](int step) {
    const int tb = step * 32;
#pragma unroll
    for (int i = 0; i < KPT; ++i) pk[i] = (unsigned)bt[max(min((tb + (tid + 256 * i) / KCH) / BS, nblk_valid - 1), 0)];
#pragma unroll
    for (int i = 0; i < VPT; ++i) pv[i] = (unsigned)bt[max(min((tb + 8 * ((tid + 256 * i) & 3)) / BS, nblk_valid - 1), 0)];
  };
  // (the last of a thread's pieces may be past a step's)
  auto gload = [&](int step) {
    const int tb = step * 32;
#pragma unroll
    for (int i = 0; i < KPT; ++i) {
      const int pi = tid + 256 * i;
      if (KP % 256 && pi >= KP) break;
      const int key = pi / KCH, ch = pi % KCH;
      const int tok = tb + key;
      const unsigned off = k_head + (unsigned)(tok % BS) * D + ch * 8;
      rk[i] = KVLoad<T, F8>::ld(kc + (size_t)pk[i] * blk_stride + off);
    }
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      const int pi = tid + 256 * i;
      if (VP % 256 && pi >= VP) break;
      const int d = pi >> 2, c = pi & 3;
      const int tok = tb + 8 * c;
      const unsigned off = v_head + (unsigned)d * BS + (tok % BS);
      rv[i] = KVLoad<T, F8>::ld(vc + (size_t)pv[i] * v_blk_stride + off);
    }
  };
  // XOR swizzle of the 16-byte pieces of a K row.  ds_read_b128 serves lanes {0-3,12-15,20-27},
  // {4-11,16-19,28-31} (and the same in the upper half) together; with the key a lane reads (krow0 + 4u
  // below) these masks put the sixteen lanes of every such group on sixteen different pieces, where the
  // earlier three-bit mask left them two-way (one extra LDS cycle per group on every K operand read).
  auto kswz = [](int key) { return !XOR ? 0 : KCH >= 16 ? (key & 15) : (((key & 3) << 1) | ((key >> 3) & 1)); };
  auto sstore = [&](int buf) {
#pragma unroll
    for (int i = 0; i < KPT; ++i) {
      const int pi = tid + 256 * i;
      if (KP % 256 && pi >= KP) break;
      const int key = pi / KCH, ch = pi % KCH;
      sK[buf][key * KROW + (ch ^ kswz(key))] = rk[i];
    }
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      const int pi = tid + 256 * i;
      if (VP % 256 && pi >= VP) break;
      const int d = pi >> 2, c = pi & 3;
      sV[buf][d * 4 + (c ^ ((d >> 1) & 3))] = rv[i];
    }
  };

  const int krow0 = 8 * (r >> 2) + (r & 3);
  // Tiles strictly below every column's causal limit and above every window edge need no masking; with no
  // soft-cap and no ALiBi the score transform is then a single multiply.  Both tests are wave-uniform.
  int full_hi = 0x7fffffff, full_lo = 0;
#pragma unroll
  for (int ct = 0; ct < NCT; ++ct) {
    if (col_off[ct] >= 0) { full_hi = min(full_hi, limit[ct]); full_lo = max(full_lo, lower[ct]); }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    full_hi = min(full_hi, __shfl_xor(full_hi, o, 64));
    full_lo = max(full_lo, __shfl_xor(full_lo, o, 64));
  }
  const bool plain = !(p.softcap > 0.f) && p.alibi == nullptr;
  const float sl2 = p.scale * 1.4426950408889634f;
  auto compute = [&](int step, int buf) {
    const int tb0 = step * 32;
    if (!(tb0 < wave_hi && tb0 + 32 > wave_lo)) return;   // wave-uniform: tile outside this wave's causal range
    const bool far_tile = p.dist_bias != nullptr && tb0 + 32 <= full_hi - p.dist_far;
    const bool fast = plain && tb0 + 32 <= full_hi && tb0 >= full_lo && (p.dist_bias == nullptr || far_tile);
    // read once for all of a wave's column tiles, or where they are multiplied
    auto k_piece = [&](int u, int s) {
      const int key = krow0 + 4 * u;
      return sK[buf][key * KROW + ((g * KS + s) ^ kswz(key))];
    };
    auto v_piece = [&](int n) {
      const int d = 16 * n + r;
      return sV[buf][d * 4 + (g ^ ((d >> 1) & 3))];
    };
    V8 kf[2][KS], vf[NT];
    if constexpr (NCT > 1) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int s = 0; s < KS; ++s) kf[u][s] = k_piece(u, s);
#pragma unroll
      for (int n = 0; n < NT; ++n) vf[n] = v_piece(n);
    }
    const int tb = tb0 + 8 * g;
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct) {
      f32x4 s0 = {0, 0, 0, 0}, s1 = {0, 0, 0, 0};
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        s0 = mfma16(NCT > 1 ? kf[0][s] : k_piece(0, s), qf[ct][s], s0);
        s1 = mfma16(NCT > 1 ? kf[1][s] : k_piece(1, s), qf[ct][s], s1);
      }
      float sv[8] = {s0[0], s0[1], s0[2], s0[3], s1[0], s1[1], s1[2], s1[3]};
      float mx = -INFINITY;
      if (fast) {
        // raw scores: the scale (positive) is applied to the maximum once and folded into the fma that
        // feeds the exponential, so a score costs max + fma + exp + add
#pragma unroll
        for (int j = 0; j < 8; ++j) mx = fmaxf(mx, sv[j]);
        mx = fmaf(mx, sl2, bfar2[ct]);
      } else {
        // a tile at least dist_far behind every column of the wave takes the table's last value throughout
        float bj[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) bj[j] = bfar2[ct];
        if (p.dist_bias && !far_tile) {
          const int d_lo = limit[ct] - 1 - (tb + 7);
          const f32x4 b0 = dist_bias4(bias_col[ct], d_lo, p.dist_far) * 1.4426950408889634f;
          const f32x4 b1 = dist_bias4(bias_col[ct], d_lo + 4, p.dist_far) * 1.4426950408889634f;
          bj[7] = b0[0]; bj[6] = b0[1]; bj[5] = b0[2]; bj[4] = b0[3];
          bj[3] = b1[0]; bj[2] = b1[1]; bj[1] = b1[2]; bj[0] = b1[3];
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const int tok = tb + j;
          float x = sv[j] * p.scale;
          if (p.softcap > 0.f) x = p.softcap * fast_tanh(x / p.softcap);
          x += slope[ct] * (float)(tok - (limit[ct] - 1));
          x = fmaf(x, 1.4426950408889634f, bj[j]);
          x = (tok < limit[ct] && tok >= lower[ct]) ? x : -INFINITY;
          sv[j] = x;
          mx = fmaxf(mx, x);
        }
      }
      mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      const float m_new = fmaxf(m[ct], mx);
      const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
      const float alpha = fexp2(m[ct] - m_use);
      m[ct] = m_new;
      float ps = 0.f;
      V8 pb;
      const float mul = fast ? sl2 : 1.f;
      const float off = (fast ? bfar2[ct] : 0.f) - m_use;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float e = fexp2(fmaf(sv[j], mul, off));
        ps += e;
        pb[j] = (T)e;
      }
      l[ct] = l[ct] * alpha + ps;
      if (__any(alpha != 1.f)) {          // the running maximum settles early: most tiles need no rescale
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[ct][n] *= alpha;
      }
#pragma unroll
      for (int n = 0; n < NT; ++n) acc[ct][n] = mfma16(NCT > 1 ? vf[n] : v_piece(n), pb, acc[ct][n]);
    }
  };

  // One register stage (two workgroups fit a CU, so one wave's global-load and softmax latency is covered by the other wave of
  // its SIMD rather than by a deeper software pipeline).  Tile t+1 sits in registers while tile t is consumed, then moves to
  // the other LDS buffer and tile t+2 is requested from the pages that were looked up an iteration before (looked up only then,
  // two prompts of 500, 32 / 32 heads, take 74 us, so 67).
  int s0 = next_step(step_lo), s1 = next_step(s0 + 1), s2 = next_step(s1 + 1);
  if (s0 < step_hi) {
    pages(s0);
    gload(s0);
    pages(s1);
    sstore(0);
    if (s1 < step_hi) gload(s1);
    pages(s2);
  }
  __syncthreads();
  for (int buf = 0; s0 < step_hi; buf ^= 1) {
    compute(s0, buf);
    if (s1 < step_hi) sstore(buf ^ 1);
    if (s2 < step_hi) gload(s2);
    s0 = s1; s1 = s2; s2 = next_step(s2 + 1);
    if (s2 < step_hi) pages(s2);
    __syncthreads();
  }

#pragma unroll
  for (int ct = 0; ct < NCT; ++ct) {
    l[ct] += __shfl_xor(l[ct], 16, 64);
    l[ct] += __shfl_xor(l[ct], 32, 64);
  }
#pragma unroll
  for (int ct = 0; ct < NCT; ++ct) {
    if (col_off[ct] < 0) continue;
    const int c = wave * COLS + ct * 16 + r;
    const int head = head0 + c % G;
    const float inv = l[ct] > 0.f ? p.v_scale / l[ct] : 0.f;
    if (p.nsplit > 1) {
      store_part<D>(p, part, col_off[ct], head, g, acc[ct], inv, m[ct], l[ct]);
      continue;
    }
    T* op = (T*)p.out + col_off[ct] * p.out_stride + (long)head * D + 4 * g;
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      V4 o;
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = (T)(acc[ct][n][i] * inv);
      *reinterpret_cast<V4*>(op + 16 * n) = o;
    }
    if (p.lse_out && g == 0)
      p.lse_out[(long)head * p.num_tokens + col_off[ct]] =
          l[ct] > 0.f ? (m[ct] + log2f(l[ct])) * 0.6931471805599453f : -INFINITY;
  }
}

// Merge split-KV partials: W waves per (token, head).  There is little to read and a chain of trips to memory to read it
// through, so the trips are what counts: a row of a partition takes D / 4 lanes of 16 bytes, the other lanes take other
// partitions, and all rows of a lane are asked for at once, beside the partitions' weights and not after them (rows of
// partitions without keys, which nobody wrote, are read and left out).  Up to eight partitions take one wave, which then
// reads four rows a lane at most (heads of 128), more take four.
// One wave that walked the partitions four rows at a time, a branch on each one's weight ahead of its load, took (us, before
// -> after): 28 heads x 64 partitions 19.7 -> 3.6, 128 of 64 values x 32 12.2 -> 4.1, 48 of 256 values x 42 42.4 -> 4.2,
// 640 x 12 9.8 -> 4.2, 160 x 2 4.0 -> 3.2.
constexpr int REDUCE_ONE_WAVE = 8;                      // partitions
template <typename T, int D, int W>
__global__ __launch_bounds__(64 * W) void attn_reduce_kernel(T* out, const float* part_out, const float* part_lse,
                                                             int Hq, int nsplit, long out_stride, const int* q_start_loc,
                                                             int num_seqs) {
  constexpr int LANES = D / 4, ROWS = 64 * W / LANES, MAXP = W == 1 ? REDUCE_ONE_WAVE : 64, U = (MAXP + ROWS - 1) / ROWS;
  __shared__ __attribute__((aligned(16))) float sum[ROWS][D];
  const long th = blockIdx.x;          // token * Hq + head
  // (prompts: rows that belong to no sequence have no parts and stay as they are)
  if (q_start_loc && (th / Hq < q_start_loc[0] || th / Hq >= q_start_loc[num_seqs])) return;
  const int lane = threadIdx.x & 63, col = 4 * ((int)threadIdx.x % LANES), row = threadIdx.x / LANES;
  f32x4 v[U];
#pragma unroll
  for (int k = 0; k < U; ++k)
    v[k] = *reinterpret_cast<const f32x4*>(part_out + (th * nsplit + min(row + k * ROWS, nsplit - 1)) * D + col);
  // lane s of every wave holds partition s (nsplit <= 64); partitions without keys (short sequences under a split factor
  // fixed at graph capture) carry -inf
  const float mine = lane < nsplit ? part_lse[th * nsplit + lane] : -INFINITY;
  float M = mine;
#pragma unroll
  for (int o_ = 32; o_ > 0; o_ >>= 1) M = fmaxf(M, __shfl_xor(M, o_, 64));
  const float Mu = (M == -INFINITY) ? 0.f : M;
  const float w_mine = (mine == -INFINITY) ? 0.f : fexp2(mine - Mu);
  float total = w_mine;
#pragma unroll
  for (int o_ = 32; o_ > 0; o_ >>= 1) total += __shfl_xor(total, o_, 64);
  f32x4 o = {0, 0, 0, 0};
#pragma unroll
  for (int k = 0; k < U; ++k) {
    const int s = row + k * ROWS;
    const float w = __shfl(w_mine, min(s, 63), 64);
    if (s < nsplit && w != 0.f) o += w * v[k];
  }
  if (row < ROWS) *reinterpret_cast<f32x4*>(&sum[row][col]) = o;
  __syncthreads();
  if (row > 0) return;
#pragma unroll
  for (int k = 1; k < ROWS; ++k) o += *reinterpret_cast<const f32x4*>(&sum[k][col]);
  const float inv = total > 0.f ? 1.f / total : 0.f;
  T* to = out + th / Hq * out_stride + th % Hq * D + col;
#pragma unroll
  for (int i = 0; i < 4; ++i) to[i] = (T)(o[i] * inv);
}

// LSE-weighted merge of two partial attention outputs (cascade / prefix+suffix).
// out, prefix, suffix: [T, H, D]; lse: [H, T] natural-log domain.
template <typename T>
__global__ void merge_attn_states_kernel(T* out, float* out_lse, const T* pre, const float* pre_lse,
                                         const T* suf, const float* suf_lse, int Tn, int H, int D) {
  const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;   // over T*H*D/8
  const int per = D / 8;
  if (idx >= (long)Tn * H * per) return;
  const int d8 = (idx % per) * 8;
  const long th = idx / per;
  const int h = th % H;
  const long t = th / H;
  float a = pre_lse[(long)h * Tn + t], b = suf_lse[(long)h * Tn + t];
  a = isinf(a) && a > 0 ? -INFINITY : a;
  b = isinf(b) && b > 0 ? -INFINITY : b;
  const float mx = fmaxf(a, b);
  const float mu = (mx == -INFINITY) ? 0.f : mx;
  const float ea = expf(a - mu), eb = expf(b - mu);
  const float den = ea + eb;
  const float wa = den > 0.f ? ea / den : 0.f, wb = den > 0.f ? eb / den : 0.f;
  using V8 = typename Vec<T>::v8;
  const V8 x = ld16<V8>(pre + th * D + d8), y = ld16<V8>(suf + th * D + d8);
  V8 o;
#pragma unroll
  for (int i = 0; i < 8; ++i) o[i] = (T)((float)x[i] * wa + (float)y[i] * wb);
  st16<V8>(out + th * D + d8, o);
  if (out_lse && d8 == 0) out_lse[(long)h * Tn + t] = den > 0.f ? mu + logf(den) : -INFINITY;
}

// ---------------------------------------------------------------------------
// host-side dispatch
// ---------------------------------------------------------------------------
template <typename T, int D, int BS, bool F8>
static int launch_attn(const AttnParams& p, int form, int grid_x, hipStream_t st, int waves) {
  // form 0: decode (split over waves, NCT=1, up to 16 query columns per kv head)
  // form 1: decode with up to 32 columns; form 2: prefill (NCT=2)
  dim3 block(256);
  if (form == 0 || form == 1) {
    for (int s0 = 0; s0 < grid_x; s0 += 65535) {       // (the most that a grid's third dimension takes)
      AttnParams c = p;
      c.num_seqs = min(grid_x - s0, 65535);
      c.q_start_loc += s0; c.seq_lens += s0; c.block_table += (long)s0 * p.max_blocks;
      const dim3 grid(p.Hkv, p.nsplit, c.num_seqs);
      if (waves == 8) {
        if constexpr (D <= 192) hipLaunchKernelGGL((paged_decode_kernel<T, D, BS, 1, F8, 8>), grid, dim3(512), 0, st, c);
        else return -6;
      } else if (form == 0) hipLaunchKernelGGL((paged_decode_kernel<T, D, BS, 1, F8, 4>), grid, block, 0, st, c);
      else hipLaunchKernelGGL((paged_decode_kernel<T, D, BS, 2, F8, 4>), grid, block, 0, st, c);
    }
  } else if (form == 3) {
    dim3 grid(grid_x, p.Hkv, p.nsplit);
    hipLaunchKernelGGL((paged_prefill_lds_kernel<T, D, BS, F8>), grid, block, 0, st, p, SparseSel{});
  } else {
    dim3 grid(grid_x, p.Hkv, p.nsplit);
    hipLaunchKernelGGL((paged_attn_kernel<T, D, BS, 2, F8>), grid, block, 0, st, p);
  }
  VDA_CHECK_LAUNCH();
  return 0;
}

template <typename T, int D, bool F8>
static int dispatch_bs(const AttnParams& p, int bs, int form, int grid_x, hipStream_t st, int waves) {
  switch (bs) {
    case 16: return launch_attn<T, D, 16, F8>(p, form, grid_x, st, waves);
    case 32: return launch_attn<T, D, 32, F8>(p, form, grid_x, st, waves);
    case 64: return launch_attn<T, D, 64, F8>(p, form, grid_x, st, waves);
  }
  return -2;
}

// Head sizes: any multiple of 32 fits the kernels (a lane group owns D / 4 values in MFMA steps of 8); built are
// 64, 96, 128, 192 and 256, so heads of 80 / 96 run in 96-value rows and 160 / 192 in 192-value rows instead of
// the next power of two (reference head sizes: csrc/attention/paged_attention_v1.cu:150-188).
template <typename T, bool F8>
static int dispatch_d8(const AttnParams& p, int d, int bs, int form, int grid_x, hipStream_t st, int waves) {
  switch (d) {
    case 64: return dispatch_bs<T, 64, F8>(p, bs, form, grid_x, st, waves);
    case 128: return dispatch_bs<T, 128, F8>(p, bs, form, grid_x, st, waves);
  }
  if constexpr (!F8) {
    switch (d) {
      case 96: return dispatch_bs<T, 96, F8>(p, bs, form, grid_x, st, waves);
      case 192: return dispatch_bs<T, 192, F8>(p, bs, form, grid_x, st, waves);
      case 256: return dispatch_bs<T, 256, F8>(p, bs, form, grid_x, st, waves);
    }
  }
  return -3;
}

template <typename T>
static int dispatch_d(const AttnParams& p, int d, int bs, int form, int grid_x, hipStream_t st, int kv_fp8, int waves = 4) {
  // fp8 caches: head sizes 64 / 128 (the common ones) to bound the number of kernel variants
  if (kv_fp8) return dispatch_d8<T, true>(p, d, bs, form, grid_x, st, waves);
  return dispatch_d8<T, false>(p, d, bs, form, grid_x, st, waves);
}

static void launch_reduce(const AttnParams& p, int dtype, int D, int num_tokens, const int* q_start_loc, hipStream_t st) {
  const long n = (long)num_tokens * p.Hq;
#define RED(TT, DD) do {                                                                                              \
    if (p.nsplit <= REDUCE_ONE_WAVE)                                                                                     \
      hipLaunchKernelGGL((attn_reduce_kernel<TT, DD, 1>), dim3(n), dim3(64), 0, st, (TT*)p.out, p.part_out, p.part_lse, \
                         p.Hq, p.nsplit, p.out_stride, q_start_loc, p.num_seqs);                                         \
    else                                                                                                                 \
      hipLaunchKernelGGL((attn_reduce_kernel<TT, DD, 4>), dim3(n), dim3(256), 0, st, (TT*)p.out, p.part_out, p.part_lse, \
                         p.Hq, p.nsplit, p.out_stride, q_start_loc, p.num_seqs); } while (0)
  if (dtype == VDA_BF16) {
    if (D == 64) RED(bf16_t, 64); else if (D == 96) RED(bf16_t, 96); else if (D == 128) RED(bf16_t, 128);
    else if (D == 192) RED(bf16_t, 192); else RED(bf16_t, 256);
  } else {
    if (D == 64) RED(f16_t, 64); else if (D == 96) RED(f16_t, 96); else if (D == 128) RED(f16_t, 128);
    else if (D == 192) RED(f16_t, 192); else RED(f16_t, 256);
  }
#undef RED
}

// Decode / speculative-verify attention.  Every sequence contributes
// q_len = q_start_loc[s+1]-q_start_loc[s] query tokens with q_len * (Hq/Hkv) <= 32.  Two parts without a workspace (16 columns and
// 192 values at most) are eight waves of one workgroup.
// num_tokens is only needed to size the split-KV reduce.
VDA_EXPORT int vda_paged_attention_decode(
    void* out, const void* q, const void* k_cache, const void* v_cache, const int* block_table,
    const int* seq_lens, const int* q_start_loc, const float* alibi, float* part_out, float* part_lse,
    int num_seqs, int num_tokens, int Hq, int Hkv, int D, int block_size, int max_blocks, int nsplit,
    int max_q_len, long q_stride, long out_stride, float scale, float softcap, int window, int dtype,
    int kv_fp8, float k_scale, float v_scale, const float* sink, int chunk, int v_shift, const float* dist_bias,
    int dist_far, int table_cols, hipStream_t st) {
  if (Hq % Hkv) return -1;
  if (chunk < 0 || v_shift < 0 || (Hkv >> v_shift) << v_shift != Hkv || (dist_bias && dist_far < 0)) return -7;
  if (nsplit < 1 || nsplit > 64) return -6;      // the reduce kernel keeps one partition per lane
  const int cols = max_q_len * (Hq / Hkv);
  if (cols > 32 || (cols > 16 && D > 128)) return -4;
  AttnParams p{q, k_cache, v_cache, out, part_out, part_lse, block_table, seq_lens, q_start_loc, alibi,
               num_seqs, Hq, Hkv, max_blocks, nsplit, q_stride, out_stride, scale * (kv_fp8 ? k_scale : 1.f), softcap,
               kv_fp8 ? v_scale : 1.f, window, 0, 1, num_tokens, nullptr};
  p.sink = sink; p.chunk = chunk; p.v_shift = v_shift; p.dist_bias = dist_bias; p.dist_far = dist_far;
  const int form = cols <= 16 ? 0 : 1;
  int waves = 4;
  if (nsplit > 1 && !part_out) {                 // no workspace: the parts are waves of one workgroup
    if (nsplit > 2 || form == 1 || D > 192) return -6;
    waves = 8;
    p.nsplit = nsplit = 1;
  }
  // the first steps are the sequence's first keys: their pages need not wait for its length
  if (nsplit == 1 && window <= 0 && chunk == 0) p.table_cols = table_cols;
  int rc = dtype == VDA_BF16 ? dispatch_d<bf16_t>(p, D, block_size, form, num_seqs, st, kv_fp8, waves)
                             : dispatch_d<f16_t>(p, D, block_size, form, num_seqs, st, kv_fp8, waves);
  if (rc) return rc;
  if (nsplit > 1) {
    launch_reduce(p, dtype, D, num_tokens, nullptr, st);
    VDA_CHECK_LAUNCH();
  }
  return 0;
}

// 1 (default): the wide form where it applies, else the 4-wave form with K/V staged through LDS;
// 0: direct-to-register form, 2: always the 4-wave LDS form, 3: the wide form whenever the shape allows
// (0 / 2 / 3 are for A/B measurements and tests)
static int g_prefill_variant = 1;
static int prefill_cols(int D) { return D <= 128 ? PREFILL_COLS<128> : PREFILL_COLS<256>; }
// (from 128 on: us, 4-wave form with the keys in parts / wide form, 128 of them 67.8 / 49.4 and 88 / 61, 144 25.4 / 22.8, 184 140 / 119; 100 of long
// prompts 97 / 113, of 1000 tokens 44.6 / 39.8; heads of 64, 128 of them, 32 / 8 heads 37 / 29 and, with 2000 keys before, 125 / 89, 8 / 1 heads 74.3 / 75.4; 96,
// 16 / 16 heads of 64 38.9 / 29.5 and on 2000 keys 52 / 80: fewer than 128 depend on the keys)
static long g_prefill_wide_min_wgs = 128;
VDA_EXPORT int vda_set_prefill_variant(int v) { g_prefill_variant = v; return 0; }
VDA_EXPORT int vda_set_prefill_wide_min_wgs(long n) { g_prefill_wide_min_wgs = n; return 0; }

// Query tokens of a wide workgroup (0: the wide form does not apply to this batch).  A group that does not divide the 256 columns leaves at
// most a sixteenth of them idle, or the 4-wave form takes it; and it has prompts of three of its tiles on average: us, 4-wave / wide, attention alone,
// 28 / 4 heads, 2 x 2161 tokens 135 / 93, 8 ragged of some 200 25.0 / 20.7, 24 of 150 34.4 / 28.4, 24 / 8 heads, one of 1000 45 / 37, 2 of 2161 189 / 145; but ragged
// ones of less, 40 / 8, 24 of 40 13.8 / 15.1, 48 / 8 14.5 / 16.6, 28 / 4 25 of 81 on 740 77 / 86.  Heads of 96 gain enough to do without: 24 / 8 heads, with rotary
// embedding and cache write, 37 x 64 34 / 28, 16 x 90 + 300 48 / 34, 22 x 200 57 / 46.
static int wide_tokens(int G, int D, int num_tokens, int num_seqs) {
  const int tokens = 256 / G;
  if (D != 64 && D != 96 && D != 128) return 0;
  if (256 % G && (tokens * G < 240 || (D != 96 && (long)num_tokens < 3L * tokens * num_seqs))) return 0;
  return tokens;
}
// Whether it is taken: workgroups for half of the CUs, and prompts that fill its tiles.  Where they don't, the 4-wave form's smaller tiles do
// less for nobody, the more so where a row of keys is short and the products little: us, 4-wave / wide, with rotary embedding and cache
// write, n x tokens + tokens in the cache: 32 / 8 heads of 128, 160 x 20 + 300 87 / 100, 80 x 40 + 300 82 / 85, 46 x 70 + 300 80 / 72; 8 / 4, 104 x 40 + 300 48 / 52, 60 x 70
// + 300 46 / 42; 64 / 8, 200 x 8 + 300 87 / 106, 80 x 20 76 / 79; 8 / 1, 352 x 20 + 300 59 / 50.
// Of 96, 16 / 8 heads, 104 x 20 27 / 31, 52 x 40 25.2 / 24.6, 51 x 70 38 / 32; 16 / 16, 52 x 40 32 / 34, 51 x 70 + 300 85 / 70, 12 x 300 67 / 48.
// Of 64, in one wave of workgroups, 32 / 8, 26 x 40 17.7 / 18.8, 15 x 70 18.1 / 16.0, 11 x 100 + 300 39 / 28, 8 / 4, 60 x 70 21 / 18; in more, 32 / 32, 32 x 100 51 / 54, 16 / 4,
// 43 x 150 + 300 53 / 59, 12 / 12, 57 x 150 51 / 56, and 32 / 32, 16 x 200 57 / 53, 32 / 8 35 / 30, 8 / 1, 64 x 200 + 300 55 / 50.
// The mean says nothing of a batch of a long prompt among short ones.  Heads of 128, one wide tile of which costs a short prompt some 0.07 us more and a long one
// saves some 6 us in 1000 tokens, 24 in 2000: us, 4-wave / wide, 32 / 8 heads, a prompt of 2000 with 100 of 10 98 / 85, with 250 of 15 125 / 115, with 500 of 10 217 / 217, with
// 1000 253 / 293, 1000 with 100 of 8 54.0 / 51.2, with 200 65 / 68, 500 with 100 of 8 54 / 61, 3000 with 400 of 2 184 / 165; 64 / 8, 2000 with 500 of 10 266 / 276, 1000 with 100 of 8
// 61 / 56; 32 / 32, 1000 with 100 of 8 on 500 279 / 253, with 200 131 / 151, 2000 with 500 of 10 536 / 601, 1500 with 130 136 / 124; 16 / 8, the last 76 / 69.
// (max_q_len: the longest run where the caller knows it, else 0)
static bool wide_pays(int wide, int Hkv, int D, int num_tokens, int num_seqs, long max_q_len) {
  if (g_prefill_variant == 3) return true;
  if (g_prefill_variant != 1 || (long)(num_tokens / wide) * Hkv < g_prefill_wide_min_wgs) return false;
  const int mean = num_tokens / max(num_seqs, 1);
  const long longest = max_q_len < num_tokens ? max_q_len : num_tokens;
  if (D == 128) return mean >= min(40, wide / 2) || longest * longest >= 9000L * num_seqs;
  if (D == 96) return mean >= min(64, wide / 2);
  return mean >= 64 && (mean >= 192 || (long)((mean + wide - 1) / wide) * num_seqs * Hkv <= 256);
}

// Into how many parts the keys of each query tile are cut (1: not at all; what lse_out and the wide form take).  max_keys: an
// upper bound of the sequences' lengths.  Without parts a few tiles walk a long prefix alone, 32 keys in some 1.2 us:
// 100 new tokens on 2000 of each of two, 32 / 8 heads of 64 137 us in one part, 37 in seven; 16 / 8 heads of 256 386 -> 83, 24 / 8 of 96 255 -> 57;
// of 128, on 3500, 300 -> 70; one prompt of 1000, 8 / 1 heads, 47 -> 30.
// Two workgroups a CU are filled, with eight steps a part at least; a part's rows are written and read back once, so that
// many query rows want few parts: their cost grows with the parts as the walk's falls.  The merge is a workgroup a (token, head), of which some
// 3500 a us start: 32 / 8 heads of 64, prompts of 520, 700 and 1000 tokens, one part / two 20.7 / 22.9, 26.0 / 28.2, 34.4 / 39.8; 14 / 2 heads, three of 500
// 22.0 / 25.3; 32 / 8 of 128, 300 on 300 30.1 / 27.5, 100 on 450 of each of four 28.6 / 29.5; 16 / 8 of 256, these 35.8 / 31.9.
// max_q_len: the longest query run where it is known (0: not).  0 parts: the wide form takes the batch.
VDA_EXPORT int vda_prefill_form(int num_seqs, int num_tokens, int Hq, int Hkv, int D, long max_keys, long max_q_len) {
  if (Hkv < 1 || Hq % Hkv || Hq / Hkv > 128) return 1;
  const int G = Hq / Hkv, q_tile = (G <= prefill_cols(D) ? prefill_cols(D) : 128) / G;
  const int wide = wide_tokens(G, D, num_tokens, num_seqs);
  if (wide && wide_pays(wide, Hkv, D, num_tokens, num_seqs, max_q_len)) return 0;
  const long wgs = (long)(num_tokens / q_tile + min(num_seqs, num_tokens)) * Hkv, steps = (max_keys + 31) / 32;
  if (wgs < 1 || wgs > 256 || steps < 16) return 1;
  const double rows = (double)num_tokens * Hq, row_part = rows * D * 8 / 4e6;                 // us
  const long parts = max(1L, min(min(min(512 / wgs, steps / 8), (long)sqrt(1.2 * steps / row_part) + 1), 64L));
  const double walk = (0.7 + 0.0055 * D) * steps, merge = 4 + rows / 3500 + row_part * parts;
  return walk * (1 - 1.0 / parts) > merge ? (int)parts : 1;
}
VDA_EXPORT int vda_prefill_parts(int num_seqs, int num_tokens, int Hq, int Hkv, int D, long max_keys) {
  return max(vda_prefill_form(num_seqs, num_tokens, Hq, Hkv, D, max_keys, 0), 1);
}

// Varlen attention of new tokens against the paged cache (the new tokens' own K/V must already be in
// the cache): causal, or bidirectional within each sequence (encoder models; the shared-prefix pass of
// cascade attention, where one pseudo-sequence holds every query token of the batch).  lse_out, when
// given, receives the log-sum-exp of every (head, token) for merging with another pass.  A workgroup has 128 / (Hq/Hkv) query tokens
// (64 / where heads hold more than 128 values, 256 / in the wide form); the grid over-allocates one tile per sequence.
// max_keys: an upper bound of what a tile sees of a sequence.
VDA_EXPORT int vda_paged_attention_prefill(
    void* out, const void* q, const void* k_cache, const void* v_cache, const int* block_table,
    const int* seq_lens, const int* q_start_loc, const float* alibi, int num_seqs, int num_tokens,
    int Hq, int Hkv, int D, int block_size, int max_blocks, long q_stride, long out_stride, float scale,
    float softcap, int window, int dtype, int kv_fp8, float k_scale, float v_scale, int causal, float* lse_out,
    int max_q_len, const float* sink, int chunk, int v_shift, const float* dist_bias, int dist_far, float* part_out,
    float* part_lse, int nsplit, long max_keys, hipStream_t st) {
  if (Hq % Hkv) return -1;
  const int G = Hq / Hkv;
  if (G > 128) return -4;
  if (!causal && (window > 0 || chunk > 0)) return -5;
  if (chunk < 0 || v_shift < 0 || (Hkv >> v_shift) << v_shift != Hkv) return -7;
  if (dist_bias && dist_far < 0) return -7;
  if (nsplit < 1 || nsplit > 64 || (nsplit > 1 && (!part_out || !part_lse || lse_out))) return -6;
  // not in the direct-to-register form
  const bool extras = sink != nullptr || chunk > 0 || v_shift > 0 || dist_bias != nullptr;
  // The form with K and V in LDS takes a head group's queries as columns of one workgroup.  Heads of 96 values, whose rows are no
  // whole number of pieces a thread, do not pay for it over three steps of keys: us, direct / LDS, 24 / 8 heads, 17 tokens 5.3 / 6.3, 64 7.6 / 8.7,
  // 16 x 60 9.4 / 10.4, 100 10.2 / 10.3, 128 11.4 / 11.2, 300 21.8 / 19.3; of 192 17 tokens 7.5 / 6.3.
  const bool lds = (g_prefill_variant != 0 || extras) && G <= prefill_cols(D) && (D != 96 || extras || max_keys > 96);
  const int q_tile = (lds ? prefill_cols(D) : 128) / G;
  AttnParams p{q, k_cache, v_cache, out, nullptr, nullptr, block_table, seq_lens, q_start_loc, alibi,
               num_seqs, Hq, Hkv, max_blocks, 1, q_stride, out_stride, scale * (kv_fp8 ? k_scale : 1.f), softcap,
               kv_fp8 ? v_scale : 1.f, window, q_tile, causal, num_tokens, lse_out, max_q_len};
  p.sink = sink; p.chunk = chunk; p.v_shift = v_shift; p.dist_bias = dist_bias; p.dist_far = dist_far;
  // Wide form (8 waves, 256 columns, 64-key tiles): heads of 64, 96 and 128 values and enough query tiles to occupy the
  // chip (one workgroup per CU); short chunks keep the 4-wave form, which cuts them into more workgroups.
  // Its copies to LDS ask for caches aligned to 16 bytes.
  const bool aligned = (((uintptr_t)k_cache | (uintptr_t)v_cache) & 15) == 0;
  const int wide = wide_tokens(G, D, num_tokens, num_seqs);
  if (nsplit == 1 && wide && aligned && wide_pays(wide, Hkv, D, num_tokens, num_seqs, max_q_len)) {
    p.q_tile = wide;
    return vda_launch_prefill_wide(p, D, block_size, dtype, kv_fp8, st);
  }
  const int grid_x = num_tokens / q_tile + num_seqs;
  const int form = lds ? 3 : 2;
  p.part_out = part_out; p.part_lse = part_lse; p.nsplit = nsplit;
  const int rc = dtype == VDA_BF16 ? dispatch_d<bf16_t>(p, D, block_size, form, grid_x, st, kv_fp8)
                                   : dispatch_d<f16_t>(p, D, block_size, form, grid_x, st, kv_fp8);
  if (rc || nsplit == 1) return rc;
  launch_reduce(p, dtype, D, num_tokens, q_start_loc, st);
  VDA_CHECK_LAUNCH();
  return 0;
}

// Sparse (vertical-slash) prefill: the 4-wave LDS form, one head per workgroup, visiting only the selected 32-key
// steps (see paged_prefill_lds_kernel).  max_keys: the longest table of the batch (sizes the LDS bitmap check).
template <typename T, int D, bool F8>
static int launch_sparse(const AttnParams& p, const SparseSel& sp, int bs, dim3 grid, hipStream_t st) {
  switch (bs) {
    case 16: hipLaunchKernelGGL((paged_prefill_lds_kernel<T, D, 16, F8, true>), grid, dim3(256), 0, st, p, sp); break;
    case 32: hipLaunchKernelGGL((paged_prefill_lds_kernel<T, D, 32, F8, true>), grid, dim3(256), 0, st, p, sp); break;
    case 64: hipLaunchKernelGGL((paged_prefill_lds_kernel<T, D, 64, F8, true>), grid, dim3(256), 0, st, p, sp); break;
    default: return -2;
  }
  VDA_CHECK_LAUNCH();
  return 0;
}

VDA_EXPORT int vda_paged_attention_prefill_sparse(
    void* out, const void* q, const void* k_cache, const void* v_cache, const int* block_table,
    const int* seq_lens, const int* q_start_loc, const int* vert, const int* vcount, const int* slash,
    const int* scount, const int* key_base, const int* q_base, int NV, int NS, int num_seqs, int num_tokens,
    int Hq, int Hkv, int D, int block_size, int max_blocks, long q_stride, long out_stride, float scale,
    float softcap, int dtype, int kv_fp8, float k_scale, float v_scale, int causal, float* lse_out, long max_keys,
    hipStream_t st) {
  if (Hq % Hkv) return -1;
  if (D != 64 && D != 128) return -3;
  if (max_keys > (long)SPARSE_BM_WORDS * 32 * 32 || (long)max_blocks * block_size > (long)SPARSE_BM_WORDS * 1024)
    return -7;
  AttnParams p{q, k_cache, v_cache, out, nullptr, nullptr, block_table, seq_lens, q_start_loc, nullptr,
               num_seqs, Hq, Hkv, max_blocks, 1, q_stride, out_stride, scale * (kv_fp8 ? k_scale : 1.f), softcap,
               kv_fp8 ? v_scale : 1.f, 0, 128, causal, num_tokens, lse_out, 0};
  SparseSel sp{vert, vcount, slash, scount, key_base, q_base, NV, NS};
  dim3 grid(num_tokens / 128 + num_seqs, Hq, 1);
#define SPARSE_GO(TT) \
  (D == 64 ? (kv_fp8 ? launch_sparse<TT, 64, true>(p, sp, block_size, grid, st)                \
                     : launch_sparse<TT, 64, false>(p, sp, block_size, grid, st))              \
           : (kv_fp8 ? launch_sparse<TT, 128, true>(p, sp, block_size, grid, st)               \
                     : launch_sparse<TT, 128, false>(p, sp, block_size, grid, st)))
  return dtype == VDA_BF16 ? SPARSE_GO(bf16_t) : SPARSE_GO(f16_t);
#undef SPARSE_GO
}

VDA_EXPORT int vda_merge_attn_states(void* out, float* out_lse, const void* pre, const float* pre_lse,
                                     const void* suf, const float* suf_lse, int T, int H, int D, int dtype,
                                     hipStream_t st) {
  if (D % 8) return -1;
  const long n = (long)T * H * (D / 8);
  const int threads = 256;
  const int blocks = (int)((n + threads - 1) / threads);
  if (dtype == VDA_BF16)
    hipLaunchKernelGGL(merge_attn_states_kernel<bf16_t>, dim3(blocks), dim3(threads), 0, st, (bf16_t*)out,
                       out_lse, (const bf16_t*)pre, pre_lse, (const bf16_t*)suf, suf_lse, T, H, D);
  else
    hipLaunchKernelGGL(merge_attn_states_kernel<f16_t>, dim3(blocks), dim3(threads), 0, st, (f16_t*)out,
                       out_lse, (const f16_t*)pre, pre_lse, (const f16_t*)suf, suf_lse, T, H, D);
  VDA_CHECK_LAUNCH();
  return 0;
}
