// Wide prefill attention for gfx950, heads of 64, 96 and 128 values: 8 waves per workgroup, 32 query columns per wave,
// 64-key tiles, 32x32x16 MFMA, products and softmax of neighbouring tiles interleaved.
//
// Same role as the prefill side of the reference's Triton unified attention
// (vllm/attention/ops/triton_unified_attention.py) and its ROCm flash-attention backend
// (vllm/v1/attention/backends/rocm_aiter_fa.py); the structure below is this repo's own.
//
// Why a second form beside paged_prefill_lds_kernel (attention.hip): that kernel gives every wave 32
// columns of 16x16x32 tiles and a 32-key step, which costs ~230 vector-ALU instructions per 32 MFMAs
// (per-lane block-table lookups, address arithmetic for a copy step of only 32 keys, two cross-lane
// maximum exchanges per 16-column tile) -- the VALU, not the matrix pipe, sets its speed.  Here
//   * a column's scores of a 32-key block sit in ONE lane pair (l, l+32) (swapped product
//     S^T = K.Q^T on the 32x32 tile), so the running maximum needs one half-swap per 64 keys;
//   * P never moves between lanes: registers 8t..8t+7 of a score block are, after conversion, the
//     B operand of the P.V product for k-step t.  The K rows are handed to the first product in an order (key_of_row) that makes
//     those eight registers eight consecutive keys, so V needs no regrouping;
//   * so 16-bit K and V go global -> LDS without passing registers, one page number (scalar) for all that a wave copies of a tile,
//     into rings of four tiles;
//   * workgroup id -> (kv head = id mod Hkv, query tile): with 8 kv heads every XCD keeps one head's keys in its L2.
//
// Schedule.  Scores, softmax and P.V of one key depend on each other, so a half step works on three blocks of 32 keys at once:
//   half step h: scores of block h + 1 and P.V of block h - 1 (16 MFMAs), and between them, in slices, the softmax of block h.
// (An MFMA of this size takes the matrix pipe for 32 cycles and the issue for 8; a vector instruction takes 4, an exponential 8.)
// A step is two of them, a tile of 64 keys, with one barrier.  Step t reads blocks of K tiles t and t + 1 and of V tiles t - 1 and
// t, which live in rings of four: it issues batch t + 2 (V of tile t + 2, K of tile t + 3) into the places that step t - 1 read
// last, and waits, before its barrier, for the batch that step t - 1 issued, which is read from step t + 1 on.  LDS reads run
// eight products ahead, across half steps and barriers.
//
// The maximum that weights are relative to is exact after every block: the largest weight, which often carries the row, is one and so exact in
// 16 bits, and the denominator adds the weights in fp32.  One that may lag by 2^8 spares most of the scaling of the 64 sums of a lane (in
// sequences of a few thousand keys some column of 32 moves in most steps) and was 10 % faster, but its largest weight is rounded, so that the
// denominator had to add rounded weights: 0.00272 against 64 bits over ragged prompts of some 1100 tokens where this is at 0.00267 (cache and output in
// bf16), and a log-sum-exp that was off by up to 0.0013.
//
// Measured (MI355X, bf16, 32 / 8 heads, attention alone; before: one barrier a tile, products and softmax of a tile one after the other, K
// and V through registers): 2048 tokens on 8192 keys 348 -> 317 us, 2 x 4096 323 -> 304, 2048 74 -> 69, 8 x 1024 115 -> 113, 16 x 256 36.1 -> 35.3;
// with rotary embedding and cache write: seven portions of some 1100 tokens 261 -> 232, 64 / 8 heads, nine of some 138 39.4 -> 36.3; e4m3 cache, 2 of some
// 1512, one on 368, 261 -> 148 (the order of tiles of launch_bs has its part in the ragged ones).
// What bounds long prompts is power and the scaling: without the latter (a lagging maximum) a step took 3650 cycles (2112 of them MFMA) at 1.9 GHz,
// before 5000 at 2.4.  The two waves of a SIMD taking turns at products and softmax of whole tiles (two barriers a tile) were no faster on long prompts
// and slower on short ones.
//
// Heads of 64 and 96 values keep the images of 128 (their rows' last pieces are zeros that nobody reads: a copy goes to LDS by lane, in whole
// kilobytes, and the ring has room) and have 8 and 12 products a half step for the same softmax, which is then what bounds them.  With rotary
// embedding and cache write, against the 4-wave form, us: 32 / 8 heads of 64, six of some 493 tokens on 2928 212 -> 130, 2 x 3000 265 -> 225, e4m3 cache,
// 15 of some 405 79 -> 63; 24 / 8 of 96, 277 -> 157, 376 -> 239 and, in bf16, 92 -> 62.
//
// Lane maps (l = lane, c = l & 31, h = l >> 5), 32x32x16:
//   A: row c, k = 8h + j        B: k = 8h + j, column c        C: row (r&3) + 8(r>>2) + 4h, column c
// Scores:  row i of a block is key_of_row(i) (bits 2 and 3 of i change places), so register r of block kb is
//          key 32kb + 16(r>>3) + 8h + (r&7) of query column c.
// P.V:     k-step t of a tile (16 keys) takes registers 8(t&1)..+7 of block t>>1: keys 16t + 8h + j.
// LDS:     K image  [key][16 pieces of 16 B], piece p of key k stored at p ^ (k & 15);
//          V image  [16-key part][d][2 pieces of 16 B], piece p of row d stored at p ^ ((d >> 4) & 1).
//          Any 16 lanes that a 16-byte read serves together (rows 0-3, 12-15, 20-27 or the others) touch all 64 banks.
#include "attention.h"
#include <climits>
#include <type_traits>

namespace {

template <typename V8> struct Mfma32;
template <> struct Mfma32<bf16x8> {
  static __device__ __forceinline__ f32x16 run(bf16x8 a, bf16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
};
template <> struct Mfma32<f16x8> {
  static __device__ __forceinline__ f32x16 run(f16x8 a, f16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
};

// max over the lane pair (l, l ^ 32)
__device__ __forceinline__ float pair_max(float x) {
  const unsigned u = __float_as_uint(x);
  auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float pair_sum(float x) {
  const unsigned u = __float_as_uint(x);
  auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

constexpr int KT = 64;               // keys per tile
constexpr int K_BYTES = KT * 256;    // one K image, rows of 128 values
constexpr int V_BYTES = 128 * 128;   // one V image
constexpr int RING = 4;              // tiles of either in LDS
constexpr int SORTED = 16;           // sequences that workgroups sort by length

__device__ __forceinline__ int key_of_row(int i) { return (i & 19) | ((i & 4) << 1) | ((i & 8) >> 1); }

// c += a b, in place: with the builtin, whose result may lie elsewhere, the compiler keeps two copies of the 64 sums across the branches
// of a step and spills the queries (300 bytes).  It does not look into the statement, so the wait between an operand's last vector
// instruction and the MFMA stands here, and settle() stands between these and what reads or scales the sums.
__device__ __forceinline__ void mfma_to(f32x16& c, bf16x8 a, bf16x8 b) {
  asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
}
__device__ __forceinline__ void mfma_to(f32x16& c, f16x8 a, f16x8 b) {
  asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_f16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
}
template <int N> __device__ __forceinline__ void settle(f32x16 (&c)[N]) {
  asm volatile("s_nop 15\n\ts_nop 15" : "+v"(c[0]));
#pragma unroll
  for (int i = 1; i < N; ++i) asm volatile("" : "+v"(c[i]));
}

// Twice 16 bytes a lane from a buffer to LDS, at dst + 16 * lane.  A statement of its own: told of the copy, the compiler would wait for
// all of them before the next LDS read, although they fill another tile of the ring.  Counted in the kernel's loop.
typedef int buf_t __attribute__((ext_vector_type(4)));
// (m0, then two copies: the second reads `step` bytes and 1024 more of voff1 and lands 1024 bytes further on)
__device__ __forceinline__ void copy16x2(buf_t buf, unsigned voff0, unsigned voff1, unsigned step, unsigned dst) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 1\n\tbuffer_load_dwordx4 %1, %3, 0 offen lds\n\tbuffer_load_dwordx4 %2, %3, %4 offen offset:1024 lds"
               ::"s"(dst), "v"(voff0), "v"(voff1), "s"(buf), "s"(step) : "memory", "m0");
}
// The same with both sources named in full
__device__ __forceinline__ void copy16_two(buf_t buf, unsigned voff0, unsigned voff1, unsigned dst) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 1\n\tbuffer_load_dwordx4 %1, %3, 0 offen lds\n\t"
               "s_add_u32 m0, %0, 0x400\n\ts_nop 1\n\tbuffer_load_dwordx4 %2, %3, 0 offen lds"
               ::"s"(dst), "v"(voff0), "v"(voff1), "s"(buf) : "memory", "m0", "scc");
}
constexpr unsigned NOWHERE = 0x40000000;               // past any page
// `bytes` from a page's head on; loads past them bring zeros
__device__ __forceinline__ buf_t page_buffer(uint64_t head, unsigned page, unsigned page_bytes, unsigned bytes) {
  const uint64_t a = head + (uint64_t)page * page_bytes;
  return buf_t{(int)a, (int)(a >> 32) & 0xffff, (int)bytes, 0x00027000};
}

template <typename T, int D, int BS, bool F8, bool GENERAL>
__global__ __launch_bounds__(512, 2) void paged_prefill_wide_kernel(AttnParams p, int ntiles, int levels) {
  using V8 = typename Vec<T>::v8;
  using V4 = typename Vec<T>::v4;
  using CT = typename KVElem<T, F8>::type;
  static_assert(D == 64 || D == 96 || D == 128, "rows of up to 128 values, in blocks of 32");
  constexpr int PART = D / 16, FULL = 2 * PART, DB = D / 32;       // products of the scores, as many of P.V, both; blocks of value rows
  __shared__ __attribute__((aligned(16))) unsigned char smem[RING * (K_BYTES + V_BYTES)];

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c32 = lane & 31, hi = lane >> 5;
  const int G = p.Hq / p.Hkv;
  const int kvh = blockIdx.x % p.Hkv, rank = blockIdx.x / p.Hkv;
  int seq, q0, qs, q_len, seq_len;
  if (levels > 0) {                                  // tile j from the end of every sequence, with another sequence first for each j
    const int j = rank / p.num_seqs;
    seq = (rank - j * p.num_seqs + j) % p.num_seqs;
    qs = p.q_start_loc[seq];
    q_len = p.q_start_loc[seq + 1] - qs;
    seq_len = p.seq_lens[seq];
    const int tiles = (q_len + p.q_tile - 1) / p.q_tile;
    if (j >= tiles) return;                          // uniform over the workgroup
    q0 = (tiles - 1 - j) * p.q_tile;
  } else if (p.num_seqs <= SORTED) {                 // sequence after sequence, the one with the most keys first, each from its end
    const int s = min(lane, p.num_seqs - 1), start = p.q_start_loc[s], end = p.q_start_loc[s + 1], len = p.seq_lens[s];
    const int tiles = lane < p.num_seqs ? (end - start + p.q_tile - 1) / p.q_tile : 0;
    const int place = (min(len, (1 << 26) - 1) << 4) + SORTED - 1 - s;                  // unique
    int first = 0;                                   // rank of this lane's sequence's first tile
#pragma unroll
    for (int i = 0; i < SORTED; ++i)
      first += __builtin_amdgcn_readlane(place, i) > place ? __builtin_amdgcn_readlane(tiles, i) : 0;
    const unsigned long long hit = __ballot(lane < SORTED && rank >= first && rank < first + tiles);
    if (hit == 0) return;                            // uniform over the workgroup
    seq = __builtin_ctzll(hit);
    q0 = (__builtin_amdgcn_readlane(tiles - 1 + first, seq) - rank) * p.q_tile;
    qs = __builtin_amdgcn_readlane(start, seq);
    q_len = __builtin_amdgcn_readlane(end, seq) - qs;
    seq_len = __builtin_amdgcn_readlane(len, seq);
  } else {
    const int tile = ntiles - 1 - rank;
    // tile -> sequence: the largest s whose first tile, q_start_loc[s] / q_tile + s (increasing in s), is not
    // behind this one; 64 candidates per load instead of one dependent load per bisection step
    seq = 0;
    for (int base = 0; base < p.num_seqs; base += 64) {
      const int s = base + lane;
      const bool ok = s < p.num_seqs && p.q_start_loc[s] / p.q_tile + s <= tile;
      const unsigned long long mask = __ballot(ok);
      if (mask == 0) break;
      seq = base + 63 - __builtin_clzll(mask);
      if (mask != ~0ull) break;
    }
    seq = __builtin_amdgcn_readfirstlane(seq);
    qs = p.q_start_loc[seq];
    q0 = (tile - (qs / p.q_tile + seq)) * p.q_tile;
    q_len = p.q_start_loc[seq + 1] - qs;
    seq_len = p.seq_lens[seq];
    if (q0 >= q_len) return;                         // uniform over the workgroup
  }
  const int ctx = seq_len - q_len;
  const int* bt = p.block_table + (long)seq * p.max_blocks;
  const int nblk_valid = (seq_len + BS - 1) / BS;
  const int qt_end = min(q_len, q0 + p.q_tile);

  // this lane's query column
  const int col = wave * 32 + c32;
  const int ti = col / G, hq = col % G;
  const int qt = q0 + ti;
  const bool valid = qt < qt_end;
  const int head = kvh * G + hq;
  const int limit = valid ? (p.causal ? ctx + qt + 1 : seq_len) : 0;
  int lower = (valid && p.window > 0) ? max(0, limit - p.window) : 0;
  if (valid && p.chunk > 0) lower = max(lower, (limit - 1) / p.chunk * p.chunk);     // keys of the query's chunk only
  const float slope = (p.alibi && valid) ? p.alibi[head] : 0.f;
  const float* bias_col = p.dist_bias ? dist_row(p, head) : nullptr;       // this column's distance biases
  const float bfar2 = (p.dist_bias && valid) ? bias_col[p.dist_far] * 1.4426950408889634f : 0.f;
  const long col_off = valid ? (long)(qs + qt) : -1;
  V8 qf[PART];
  {
    const T* qp = (const T*)p.q + (long)(qs + (valid ? qt : q0)) * p.q_stride + (long)head * D + 8 * hi;
#pragma unroll
    for (int s = 0; s < PART; ++s) qf[s] = valid ? ld16<V8>(qp + 16 * s) : V8{};
  }
  int wave_hi = valid ? limit : 0, wave_lo = valid ? lower : 0x7fffffff;
  int full_hi = valid ? limit : 0x7fffffff, full_lo = valid ? lower : 0;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    wave_hi = max(wave_hi, __shfl_xor(wave_hi, o, 64));
    wave_lo = min(wave_lo, __shfl_xor(wave_lo, o, 64));
    full_hi = min(full_hi, __shfl_xor(full_hi, o, 64));
    full_lo = max(full_lo, __shfl_xor(full_lo, o, 64));
  }
  wave_hi = __builtin_amdgcn_readfirstlane(wave_hi);
  wave_lo = __builtin_amdgcn_readfirstlane(wave_lo);
  full_hi = __builtin_amdgcn_readfirstlane(full_hi);
  full_lo = __builtin_amdgcn_readfirstlane(full_lo);
  // workgroup-uniform key range (all waves take part in every tile copy)
  const int wg_hi = p.causal ? ctx + qt_end : seq_len;
  int wg_lo = p.window > 0 ? max(0, ctx + q0 + 1 - p.window) : 0;
  if (p.chunk > 0 && p.causal) wg_lo = max(wg_lo, (ctx + q0) / p.chunk * p.chunk);
  const int kt_lo = wg_lo / KT, kt_hi = (wg_hi + KT - 1) / KT;

  const CT* kc = (const CT*)p.k_cache;
  const CT* vc = (const CT*)p.v_cache;
  const unsigned blk_stride = (unsigned)p.Hkv * BS * D;          // elements per K cache block
  const unsigned v_blk_stride = (unsigned)(p.Hkv >> p.v_shift) * D * BS;     // per V cache block (fewer heads when shared)
  const unsigned k_head = (unsigned)kvh * BS * D, v_head = (unsigned)(kvh >> p.v_shift) * D * BS;

  // ---- copies: wave w takes keys 8 w .. 8 w + 7 of a tile's K and half of the value rows of its 16-key part w / 2, so one page ----
  const int part = wave >> 1, in_page = 16 * part % BS;
  // (in two pieces of 1 KB; the second's rows lie 4 and 32 further on, and a K row's pieces change with bit 2 of the key)
  const int key0 = 8 * (wave & 1) + (lane >> 4), d0 = 64 * (wave & 1) + (lane >> 1);
  // elements, from the page's head; heads of fewer than 128 values leave pieces of the images that nobody reads
  const int piece = (lane & 15) ^ key0;
  const unsigned k_off = (unsigned)(in_page + key0) * D + (piece << 3);
  const unsigned k_off1 = D == 128 ? k_off ^ 32 : (unsigned)(in_page + key0) * D + ((piece ^ 4) << 3);
  const unsigned v_off = (unsigned)d0 * BS + in_page + (((lane & 1) ^ ((d0 >> 4) & 1)) << 3);
  constexpr int K_STEP = 4 * D, V_STEP = 32 * BS;
  const bool k_there = piece < D / 8, k_there1 = (piece ^ 4) < D / 8, v_there = d0 < D, v_there1 = d0 + 32 < D;
  const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;
  // page numbers of this wave's part, of 64 tiles at a time
  const int n = max(kt_hi - kt_lo, 0);               // tiles of this workgroup
  int pages = 0;
  auto fetch_pages = [&](int t) {
    pages = bt[max(min(((kt_lo + t + lane) * KT + 16 * part) / BS, nblk_valid - 1), 0)];
    __builtin_amdgcn_s_waitcnt(0x0f70);              // vmcnt(0), here and not behind the branch, where it would be waited for in every step
  };
  auto page_of = [&](int t) { return __builtin_amdgcn_readlane(pages, t & 63); };
  auto pages_for = [&](int t) {                      // before page_of(t), for every t in turn
    if ((t & 63) == 0) fetch_pages(t);
  };
  int page = 0;                                      // of the K tile that was copied last: V's turn is a batch later
  const uint64_t k_base = (uint64_t)(kc + k_head), v_base = (uint64_t)(vc + v_head);      // of this kv head in page 0
  const unsigned k_page = blk_stride * sizeof(CT), v_page = v_blk_stride * sizeof(CT);
  // an e4m3 cache is widened on its way: a batch waits in registers for a step and is written by commit()
  u32x2 rk[F8 ? 2 : 1], rv[F8 ? 2 : 1];
  auto copy_k = [&](int page, int slot, bool exists) {
    if constexpr (F8) {
      if (exists)
#pragma unroll
        for (int i = 0; i < 2; ++i)
          rk[i] = *reinterpret_cast<const u32x2*>(k_base + (uint64_t)(unsigned)page * k_page +
                                                  (i == 0 ? k_there ? k_off : 0 : k_there1 ? K_STEP + k_off1 : 0));
    } else if constexpr (D == 128) {
      copy16x2(page_buffer(k_base, page, k_page, exists ? BS * D * 2 : 0), k_off * 2, k_off1 * 2, K_STEP * 2 - 1024,
               lds0 + slot * K_BYTES + wave * 2048);
    } else {
      copy16_two(page_buffer(k_base, page, k_page, exists ? BS * D * 2 : 0), k_there ? k_off * 2 : NOWHERE,
                 k_there1 ? (K_STEP + k_off1) * 2 : NOWHERE, lds0 + slot * K_BYTES + wave * 2048);
    }
  };
  auto copy_v = [&](int page, int slot, bool exists) {
    if constexpr (F8) {
      if (exists)
#pragma unroll
        for (int i = 0; i < 2; ++i)
          rv[i] = *reinterpret_cast<const u32x2*>(v_base + (uint64_t)(unsigned)page * v_page + ((i == 0 ? v_there : v_there1) ? i * V_STEP + v_off : 0));
    } else if constexpr (D == 128) {
      copy16x2(page_buffer(v_base, page, v_page, exists ? BS * D * 2 : 0), v_off * 2, v_off * 2, V_STEP * 2 - 1024,
               lds0 + RING * K_BYTES + slot * V_BYTES + wave * 2048);
    } else {
      copy16_two(page_buffer(v_base, page, v_page, exists ? BS * D * 2 : 0), v_there ? v_off * 2 : NOWHERE,
                 v_there1 ? (V_STEP + v_off) * 2 : NOWHERE, lds0 + RING * K_BYTES + slot * V_BYTES + wave * 2048);
    }
  };
  auto commit_k = [&](int slot) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
      *reinterpret_cast<V8*>(smem + slot * K_BYTES + wave * 2048 + i * 1024 + lane * 16) = KVLoad<T, true>::widen(rk[F8 ? i : 0]);
  };
  auto commit_v = [&](int slot) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
      *reinterpret_cast<V8*>(smem + RING * K_BYTES + slot * V_BYTES + wave * 2048 + i * 1024 + lane * 16) = KVLoad<T, true>::widen(rv[F8 ? i : 0]);
  };
  // batch u: V of tile u and K of tile u + 1.  A tile that does not exist is copied from an empty buffer, so that all batches count alike.
  auto batch_v = [&](int u) { copy_v(page, u & (RING - 1), u < n); };
  auto batch_k = [&](int u) {
    page = page_of(u + 1);
    copy_k(page, (u + 1) & (RING - 1), u + 1 < n);
  };
  auto commit = [&](int u) {
    if (u < n) commit_v(u & (RING - 1));
    if (u + 1 < n) commit_k((u + 1) & (RING - 1));
  };

  // ---- operand read addresses (bytes, slot 0) ----
  // K operand of k-step s: row c32 (+32 for the second block), piece 2s + hi, which is k_rd ^ 32 s
  const int k_rd = key_of_row(c32) * 256 + 16 * (hi ^ (key_of_row(c32) & 15));
  const int v_rd = RING * K_BYTES + c32 * 32 + 16 * (hi ^ (c32 >> 4));    // V operand: + 4096 a k-step, + 1024 a block of 32 rows

  float m = -INFINITY, l = 0.f;       // l: this lane's half of the column's sum
  if (p.sink && valid) {               // a sink: the maximum starts there, the sum with its weight of one (in one half)
    m = p.sink[head] * 1.4426950408889634f;
    l = hi == 0 ? 1.f : 0.f;
  }
  f32x16 acc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[db][r] = 0.f;

  const float sl2 = p.scale * 1.4426950408889634f;
  const bool far_plain = p.dist_bias != nullptr && !(p.softcap > 0.f) && p.alibi == nullptr;

  f32x16 S[2];                                       // scores and weights of a tile's two blocks
  V8 pb[2][2];
  // ---- products of a half step, with the operands read AHEAD of them: scores of block kb of the tile in K slot ks (bit 0 of `what`), P.V
  // of block vb of the tile in V slot vs (bit 1).  Where both are there they alternate, so that no MFMA waits for the one before it. ----
  constexpr int AHEAD = D == 96 ? 6 : 8;             // (a divisor of FULL)
  V8 fr[AHEAD];
  auto read = [&](int i, int what, int ks, int kb, int vs, int vb) {
    const int j = what == 3 ? i >> 1 : i;
    if (what == 1 || (what == 3 && (i & 1) == 0))
      fr[i % AHEAD] = *reinterpret_cast<const V8*>(smem + ((ks * K_BYTES + k_rd) ^ (32 * j)) + kb * 8192);
    else
      fr[i % AHEAD] = *reinterpret_cast<const V8*>(smem + vs * V_BYTES + v_rd + (2 * vb + j / DB) * 4096 + j % DB * 1024);
  };
  auto product = [&](int i, int what, int kb, int vb) {
    const int j = what == 3 ? i >> 1 : i;
    if (what == 1 || (what == 3 && (i & 1) == 0)) {
      if (j == 0)
#pragma unroll
        for (int r = 0; r < 16; ++r) S[kb][r] = 0.f;
      S[kb] = Mfma32<V8>::run(fr[i % AHEAD], qf[j], S[kb]);
    } else {
      mfma_to(acc[j % DB], fr[i % AHEAD], pb[vb][j / DB]);
    }
  };
  // blocks of this wave's range, and those of them that need no mask (wave-uniform)
  const int key_lo = kt_lo * KT, blocks = 2 * n;
  const int a_lo = wave_hi > wave_lo ? max((wave_lo - key_lo) >> 5, 0) : blocks, a_hi = min((wave_hi + 31 - key_lo) >> 5, blocks);
  const int w_lo = (full_lo + 31 - key_lo) >> 5, w_hi = (full_hi - key_lo) >> 5;
  const int f_hi = GENERAL ? (far_plain ? (full_hi - p.dist_far - key_lo) >> 5 : INT_MIN) : 0;
  auto active = [&](int h) { return h >= a_lo && h < a_hi; };
  // ---- softmax of a block in slices.  Before it, sm_mask: what a block needs beside the scale, which is otherwise folded into the
  // exponent's fma: causal and window masks; in the GENERAL instance (of its own, so that the common one does not pay for its
  // registers) soft cap, ALiBi and a distance-bias table as well, of which only the last value remains, as a constant of that
  // fma, for blocks at least dist_far behind every column. ----
  float mx, alpha, off, ps[2], mul = sl2, add = 0.f;
  auto sm_mask = [&](int h, int kb) {
    const bool whole = h >= w_lo && h < w_hi;
    if (GENERAL) {
      const bool far = whole && h < f_hi;
      mul = far ? sl2 : 1.f;
      add = far ? bfar2 : 0.f;
      if (far) return;
    } else if (whole) return;
    const int tb = key_lo + 32 * h, left = limit - (tb + 8 * hi), skip = lower - (tb + 8 * hi);      // key k of this lane's: skip <= k < left
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int key0 = 16 * (q >> 1) + 4 * (q & 1);
      f32x4 bq = {0, 0, 0, 0};                       // the biases of this run of four keys
      // keys k .. k + 3 sit limit - 1 - key behind the query: ascending distances from the last
      if (GENERAL && bias_col) bq = dist_bias4(bias_col, left - 1 - (key0 + 3), p.dist_far);
#pragma unroll
      for (int r = 4 * q; r < 4 * q + 4; ++r) {
        const int key = key0 + (r & 3);
        float x = S[kb][r];
        if constexpr (GENERAL) {
          x *= p.scale;
          if (p.softcap > 0.f) x = p.softcap * fast_tanh(x / p.softcap);
          x += slope * (float)(key - (left - 1));
          x += bq[3 - (r & 3)];
          x *= 1.4426950408889634f;
        }
        S[kb][r] = (key < left && key >= skip) ? x : -INFINITY;
      }
    }
  };
  auto sm_max = [&](int kb, int q) {                  // quarter q of the maximum: four keys
    if (q == 0) mx = -INFINITY;
#pragma unroll
    for (int r = 4 * q; r < 4 * q + 4; ++r) mx = fmaxf(mx, S[kb][r]);
  };
  auto sm_move = [&] {
    mx = pair_max(GENERAL ? fmaf(mx, mul, add) : mx * mul);       // the scale is positive
    const float m_new = fmaxf(m, mx), m_use = m_new == -INFINITY ? 0.f : m_new;
    alpha = fexp2(m - m_use);
    m = m_new;
    off = (GENERAL ? add : 0.f) - m_use;
    ps[0] = ps[1] = 0.f;
  };
  auto sm_exp = [&](int kb, int k) {                  // weights 2 k and 2 k + 1 of the lane's 16
    const int t = k >> 2, j = 2 * (k & 3);
    const float a = fexp2(fmaf(S[kb][2 * k], mul, off)), b = fexp2(fmaf(S[kb][2 * k + 1], mul, off));
    pb[kb][t][j] = (T)a;
    pb[kb][t][j + 1] = (T)b;
    ps[0] += a;
    ps[1] += b;
  };
  // What a block's new maximum scales the sums by is due before that block's P.V, in the next half step: there a quarter of the sums is
  // scaled in front of its first product, beside the scores' MFMAs.
  float due = 1.f;
  bool any_due = false;
  auto sm_end = [&](bool first_block) {                // (whose sums are still zero)
    l = l * alpha + (ps[0] + ps[1]);
    due = alpha;
    any_due = !first_block && __any(alpha != 1.f);
  };
  auto scale_due = [&](int j) {
    if (any_due) {
      asm volatile("s_nop 11" : "+v"(acc[j]));         // (the quarter's last product)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[j][r] *= due;
      asm volatile("" : "+v"(acc[j]));
    }
  };

  auto step_end = [&] {
    if (F8) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(4)" ::: "memory");       // all but the last batch have landed
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  // half step h, whose block is number b of tile t: block h + 1 lies in K slot ks, block h - 1 in V slot vs
  auto half_full = [&](int h, auto b_, int ks, int vs, int ks_next, int vs_next, auto extra) {       // all three parts, interleaved
    constexpr int b = decltype(b_)::value;
    sm_mask(h, b);
    // (empty statements keep a slice's results in its place: otherwise the exponentials sink behind the branch of sm_end)
#pragma unroll
    for (int i = 0; i < FULL; ++i) {
      if (i < 2 * DB && (i & 1)) scale_due(i >> 1);
      product(i, 3, 1 - b, 1 - b);
      // the first operands of the next half step as well
      if (i + AHEAD < FULL) read(i + AHEAD, 3, ks, 1 - b, vs, 1 - b);
      else read(i + AHEAD - FULL, 3, ks_next, b, vs_next, b);
      if (i == 1 || i == 2) {                          // (the last scores left the matrix pipe a while ago)
        sm_max(b, 2 * (i - 1));
        sm_max(b, 2 * (i - 1) + 1);
        asm volatile("" : "+v"(mx));
      } else if (i == 3) {
        sm_move();
        asm volatile("" : "+v"(off), "+v"(alpha));
      } else if (i > 3) {
#pragma unroll
        for (int k = (i - 4) * 8 / (FULL - 4); k < (i - 3) * 8 / (FULL - 4); ++k) {
          sm_exp(b, k);
          asm volatile("" : "+v"(ps[0]), "+v"(ps[1]));
        }
      }
      extra(i);
      __builtin_amdgcn_sched_barrier(0);
    }
    sm_end(false);
  };
  auto half_parts = [&](int h, auto b_, int ks, int vs) {       // the parts that exist, one after another
    constexpr int b = decltype(b_)::value;
    auto products = [&](auto what_) {
      constexpr int what = decltype(what_)::value;
#pragma unroll
      for (int i = 0; i < min(AHEAD, PART); ++i) read(i, what, ks, 1 - b, vs, 1 - b);
#pragma unroll
      for (int i = 0; i < PART; ++i) {
        if (what == 2 && i < DB) scale_due(i);
        product(i, what, 1 - b, 1 - b);
        if (i + AHEAD < PART) read(i + AHEAD, what, ks, 1 - b, vs, 1 - b);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    if (active(h + 1)) products(std::integral_constant<int, 1>{});
    if (active(h - 1)) products(std::integral_constant<int, 2>{});
    if (active(h)) {
      sm_mask(h, b);
#pragma unroll
      for (int q = 0; q < 4; ++q) sm_max(b, q);
      sm_move();
#pragma unroll
      for (int k = 0; k < 8; ++k) sm_exp(b, k);
      sm_end(h == a_lo);
    }
  };
  constexpr std::integral_constant<int, 0> first{};
  constexpr std::integral_constant<int, 1> second{};
  auto step_copies = [&](int t) {                    // batch t + 2 (into registers, and t + 1 from there)
    if (F8) commit(t + 1);
    pages_for(t + 3);
    batch_v(t + 2);
    batch_k(t + 2);
  };
  const int full_first = (a_lo + 2) >> 1, full_end = (a_hi - 1) >> 1;       // tiles whose three parts exist in both half steps

  if (n > 0) {
    pages_for(0);
    if constexpr (F8) {                              // K tile 0 and batch 0 in one trip; batch 1, which step 0 commits
      u32x2 k0[2];
      page = page_of(0);
      copy_k(page, 0, true);
      k0[0] = rk[0];
      k0[1] = rk[1];
      batch_v(0);
      batch_k(0);
#pragma unroll
      for (int i = 0; i < 2; ++i)
        *reinterpret_cast<V8*>(smem + wave * 2048 + i * 1024 + lane * 16) = KVLoad<T, true>::widen(k0[i]);
      commit(0);
      batch_v(1);
      batch_k(1);
    } else {                                         // K tile 0, batches 0 and 1
      page = page_of(0);
      copy_k(page, 0, true);
      for (int u = 0; u < 2; ++u) {
        batch_v(u);
        batch_k(u);
      }
    }
    step_end();                                      // all but batch 1 have landed
    if (active(0)) half_parts(-1, second, 0, 0);
    for (int t = 0; t < n; ++t) {
      if (t >= full_first && t < full_end) {
        // K tiles t and t + 1 and V tiles t - 1 and t are there throughout step t, and the next step's first operands with them
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) {
          read(i, 3, t & (RING - 1), 1, (t - 1) & (RING - 1), 1);
          __builtin_amdgcn_sched_barrier(0);         // in the loop's own order: the loop's first wait is for the oldest alone
        }
        for (; t < full_end; ++t) {
          const int s0 = t & (RING - 1), s1 = (t + 1) & (RING - 1);
          if (F8) step_copies(t);
          else pages_for(t + 3);
          half_full(2 * t, first, s0, (t - 1) & (RING - 1), s1, s0, [&](int i) {
            if (!F8 && i == FULL * 6 / 16) batch_v(t + 2);
            if (!F8 && i == FULL * 11 / 16) batch_k(t + 2);
          });
          half_full(2 * t + 1, second, s1, s0, s1, s0, [](int) {});
          step_end();
        }
      }
      step_copies(t);
      half_parts(2 * t, first, t & (RING - 1), (t - 1) & (RING - 1));
      half_parts(2 * t + 1, second, (t + 1) & (RING - 1), t & (RING - 1));
      step_end();
    }
    if (active(2 * n - 1)) half_parts(2 * n, first, 0, (n - 1) & (RING - 1));
  }

  settle(acc);
  l = pair_sum(l);
  if (col_off < 0) return;
  const float inv = l > 0.f ? p.v_scale / l : 0.f;
  // Lane l holds d = 8k + 4hi .. +3 of its row for the sixteen groups k = 4db + rr; a half-swap per pair of
  // groups gives every lane 16 contiguous bytes, so the row leaves in 8 stores of 16 bytes, not 16 of 8.
  T* op = (T*)p.out + col_off * p.out_stride + (long)head * D + 8 * hi;
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int rr = 0; rr < 4; rr += 2) {
      V4 oa, ob;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        oa[i] = (T)(acc[db][4 * rr + i] * inv);
        ob[i] = (T)(acc[db][4 * rr + 4 + i] * inv);
      }
      u32x2 a = __builtin_bit_cast(u32x2, oa), b = __builtin_bit_cast(u32x2, ob);
      auto r0 = __builtin_amdgcn_permlane32_swap(a[0], b[0], false, false);
      auto r1 = __builtin_amdgcn_permlane32_swap(a[1], b[1], false, false);
      u32x4 w;
      w[0] = r0[0]; w[1] = r1[0]; w[2] = r0[1]; w[3] = r1[1];
      *reinterpret_cast<u32x4*>(op + 32 * db + 8 * rr) = w;
    }
  if (p.lse_out && hi == 0)
    p.lse_out[(long)head * p.num_tokens + col_off] =
        l > 0.f ? (m + log2f(l)) * 0.6931471805599453f : -INFINITY;
}

template <typename T, int D, bool F8, bool GENERAL>
int launch_bs(const AttnParams& p, int bs, int ntiles, hipStream_t st) {
  // The order of the tiles.  The longest query run, when the host passed it, bounds the tiles of a sequence, so that a tile of every
  // sequence in turn, the longest (causal) ones first, is a count without a search: for sequences of about one length, and for many.  Where
  // up to 16 are of unlike lengths, that gives neighbours in time no keys to share and ties sequences to shader engines (a
  // workgroup's number decides on its engine): these go one after another, the one with the most keys first.
  // us, tile of every sequence / in the batch's order / sorted, 32 / 8 heads, ragged: 8 of some 1000 tokens on 500 250 / 233 / 227, 15 of 240 on 3700
  // 386 / 378 / 319, 7 of 1100, half of them on 900, 232 / 202 / 203, 4 of 2000 226 / 229 / 227; equal ones: 8 of 1024 113 / 120 / 126, 32 of 64 14.0 / 19.1 / -.
  const int bound = p.max_q_len > 0 ? (p.max_q_len + p.q_tile - 1) / p.q_tile : 0;
  const long by_level = (long)bound * p.num_seqs;
  const bool alike = (long)p.max_q_len * p.num_seqs * 15 <= (long)p.num_tokens * 16;
  // (nor does the order matter where all tiles run at once)
  const int levels = bound > 0 && by_level <= 2L * ntiles && (p.num_seqs > SORTED || alike || by_level * p.Hkv <= 256) ? bound : 0;
  const long ranks = levels > 0 || (bound > 0 && by_level < ntiles) ? by_level : ntiles;
  const dim3 grid((unsigned)(ranks * p.Hkv)), block(512);
  switch (bs) {
    case 16: hipLaunchKernelGGL((paged_prefill_wide_kernel<T, D, 16, F8, GENERAL>), grid, block, 0, st, p, ntiles, levels); break;
    case 32: hipLaunchKernelGGL((paged_prefill_wide_kernel<T, D, 32, F8, GENERAL>), grid, block, 0, st, p, ntiles, levels); break;
    case 64: hipLaunchKernelGGL((paged_prefill_wide_kernel<T, D, 64, F8, GENERAL>), grid, block, 0, st, p, ntiles, levels); break;
    default: return -2;
  }
  VDA_CHECK_LAUNCH();
  return 0;
}

template <typename T, int D, bool F8>
int launch_mode(const AttnParams& p, int bs, int ntiles, hipStream_t st) {
  const bool general = p.softcap > 0.f || p.alibi != nullptr || p.dist_bias != nullptr;
  return general ? launch_bs<T, D, F8, true>(p, bs, ntiles, st) : launch_bs<T, D, F8, false>(p, bs, ntiles, st);
}
template <typename T>
int launch_dim(const AttnParams& p, int D, int bs, bool f8, int ntiles, hipStream_t st) {
  switch (D) {
    case 64: return f8 ? launch_mode<T, 64, true>(p, bs, ntiles, st) : launch_mode<T, 64, false>(p, bs, ntiles, st);
    case 96: return f8 ? -3 : launch_mode<T, 96, false>(p, bs, ntiles, st);
    case 128: return f8 ? launch_mode<T, 128, true>(p, bs, ntiles, st) : launch_mode<T, 128, false>(p, bs, ntiles, st);
  }
  return -3;
}

}  // namespace

// p.q_tile must be 256 / (Hq / Hkv) (columns left over belong to no token)
int vda_launch_prefill_wide(const AttnParams& p, int D, int block_size, int dtype, int kv_fp8, hipStream_t st) {
  const int ntiles = p.num_tokens / p.q_tile + p.num_seqs;
  return dtype == VDA_BF16 ? launch_dim<bf16_t>(p, D, block_size, kv_fp8, ntiles, st) : launch_dim<f16_t>(p, D, block_size, kv_fp8, ntiles, st);
}
