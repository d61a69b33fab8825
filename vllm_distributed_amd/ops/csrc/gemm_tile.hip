// LDS-tiled MFMA GEMM family for gfx950: the compute-bound regime (many rows per weight matrix).
//
//   vda_tile_gemm         out = epilogue(X . W^T) for one dense weight matrix or for the experts of a
//                         routed MoE layer over expert-sorted (token, slot) pairs
//
// One kernel template serves 16-bit operands (v_mfma_f32_16x16x32_bf16/f16) and e4m3 operands: the
// fp8 form issues v_mfma_scale_f32_16x16x128_f8f6f4 with unit block scales, the instruction that runs at
// twice the 16-bit MFMA rate on CDNA4 (the plain 16x16x32 fp8 form runs at the 16-bit rate).
//
// Tile: 256 weight rows x (32 * TN) activation rows x 128 bytes of K per step (128 e4m3 or 64 16-bit
// elements), 8 waves as 4 (weight rows) x 2 (activation rows), each wave 4 x TN accumulator tiles of
// 16 x 16.  The weights are the MFMA A operand and the activations the B operand, so a lane ends up with
// four consecutive output columns of one activation row (an 8-byte store) and the SiLU(gate) * up pair of
// a gated MLP sits in the same lane: a gate/up tile is 128 gate rows plus the 128 up rows of the same
// columns.  Both operands go global -> LDS with 16-byte global_load_lds (no staging registers) into a ring
// of three LDS stages: the fill of step kt + 2 is issued at the start of step kt and is still in flight
// when the step ends (counted s_waitcnt vmcnt + raw s_barrier), so a K step never waits for a load it
// has just issued; one workgroup (two waves per SIMD) per CU.
//
// LDS image: [row][8 chunks of 16 bytes], chunk c of row r stored at c ^ f(r),
//   f(r) = ((r >> 1) & 7) ^ ((((r >> 2) ^ (r >> 3)) & 1) << 1).
// Lane (r = lane & 15, g = lane >> 4) owns bytes [32 g, 32 g + 32) of its row in every K step, for both
// operands alike (any K order works as long as both operands use the same one): two ds_read_b128 of
// chunks 2g and 2g + 1.  ds_read_b128 is served in the lane groups {0-3, 12-15, 20-27}, ..., i.e. rows
// {0-3, 12-15} at chunk q together with rows {4-11} at chunk q ^ 2; a 128-byte row is half a 256-byte bank
// row (row parity picks the half), and f makes the sixteen 16-byte slots of every group distinct.  The LDS
// side of global_load_lds is lane-linear, so the XOR is applied to the global source chunk instead.
//
// Grouped (MoE) work distribution is read from device memory (tile table), so nothing syncs with the
// host and the layer is hipGraph-capturable; the grid covers the worst-case tile count and surplus
// workgroups exit.  Blocks are numbered so that the blocks resident on one XCD at a time share weight and activation
// panels in that XCD's L2 (tile_of_block).
//
// Scales (fp8): SC_TOKEN  out = acc * x_scale[row] * w_scale[expert]            (per-token x per-tensor)
//               SC_BLOCK  acc += partial(K step) * x_scale[row][kb] * w_scale[expert][nb][kb]
//                         (1 x 128 activation groups, 128 x 128 weight blocks: DeepSeek-V3 checkpoints)
// Counterpart of the reference's Triton fused_moe_kernel (vllm/model_executor/layers/fused_moe/
// fused_moe.py:267-476), w8a8_block_fp8_matmul (quantization/utils/fp8_utils.py:570) and
// moe_align_block_size (csrc/moe/moe_align_sum_kernels.cu:17-230).
#include "mfma_tile.h"
#include <type_traits>

// EPI_UP_ACT: the first GEMM of experts without a gate half (rows gathered per pair like EPI_GATE_UP, plain weight
// rows, act(v) out)
enum { EPI_PLAIN = 0, EPI_GATE_UP = 1, EPI_DOWN = 2, EPI_UP_ACT = 3 };
enum { SC_NONE = 0, SC_TOKEN = 1, SC_BLOCK = 2 };

struct TileGemmArgs {
  void* out;                 // [rows_out, N] 16-bit
  const void* x;             // activations, K contiguous
  const void* w;             // weights [E, W_rows, K], K contiguous
  const float* x_scale;      // SC_TOKEN: [x rows]; SC_BLOCK: [x rows, K / 128]
  const float* w_scale;      // SC_TOKEN: [E]; SC_BLOCK: [E, ceil(W_rows / 128), K / 128]
  const float* topk_w;       // EPI_DOWN: routing weight per pair
  const void* bias;          // EPI_PLAIN: optional [N], output dtype
  const int* sorted;         // grouped: pair ids sorted by expert
  const int* tile_expert;    // grouped: expert of m-tile i
  const int* tile_beg;       // grouped: first sorted position of m-tile i
  const int* tile_end;       // grouped: end of that expert's sorted range; wide tiles: of the m-tile
  const int* num_tiles;      // grouped: number of valid m-tiles (device)
  int M;                     // dense: activation rows
  int N;                     // output columns (EPI_GATE_UP: I, the weight has 2 I rows)
  int K;                     // elements
  int top_k;
  int act;                   // EPI_GATE_UP: activation of the gated pair (codes of gated_pair)
  float act_limit;           //              its clamp, for the codes that have one
  int m_tiles;               // grid bound on m-tiles
  int n_tiles;
  long x_stride;             // elements
  long out_stride;           // elements
  long w_expert_stride;      // elements
};

// Which tile a block computes.  Block ids are dealt round-robin to the 8 XCDs.  Tiles are walked in bands of eight m-tiles,
// m first, and an XCD takes 64 of that walk at a time (8 x 8 tiles: what it has in flight shares eight activation and four
// weight panels in its L2); what is left after whole rounds of 512 is cut into eight equal parts.  Dealing 8 x 8 patches to
// the end left XCDs idle: 37 x 16 tiles are 10 patches, two for some XCDs and one for the others.  Layers on 128-row tiles,
// before -> after: 60 experts 2048 x 1408, 3000 tokens 481 -> 423 us, 7680 tokens 973 -> 789; 8 experts 4096 x 14336, 2400
// tokens 2196 -> 2020; where patches came out even (64 experts 2048 x 1024, 2400 tokens) 432 -> 440.  e4m3 experts: 8 of 4096 x 14336, 600 tokens
// 576 -> 470; 60 of 2048 x 1408, 2100 tokens 331 -> 273; 64 of 2048 x 1024, 2500 tokens 328 -> 329.
__device__ __forceinline__ bool tile_of_block(int m_tiles, int n_tiles, int& mi, int& ni) {
  const int total = m_tiles * n_tiles, xcd = blockIdx.x & 7, seq = blockIdx.x >> 3;
  const int whole = total / 512 * 64, last = total - 8 * whole, per = (last + 7) >> 3;
  const int idx = seq < whole ? ((seq >> 6) * 8 + xcd) * 64 + (seq & 63) : 8 * whole + xcd * per + seq - whole;
  if (seq >= whole + per || idx >= total) return false;
  const int band = idx / (8 * n_tiles), rows = min(8, m_tiles - 8 * band), rem = idx - band * 8 * n_tiles;
  ni = rem / rows;
  mi = 8 * band + rem - ni * rows;
  return true;
}
static unsigned tile_blocks(int m_tiles, int n_tiles) { return (unsigned)(((long)m_tiles * n_tiles + 7) / 8 * 8); }

// TI: operand element type (bf16_t / f16_t / uint8_t = e4m3); TO: output type.
// 8 waves as 4 (weight rows) x 2 (activation rows); three LDS stages, the fill of step kt + 2 in flight
// across the barrier that ends step kt (counted s_waitcnt, raw s_barrier: a __syncthreads() would drain it).
template <typename TI, typename TO, int EPI, bool GROUPED, int SC, int TN>
__global__ __launch_bounds__(512, 1) void tile_gemm_kernel(const TileGemmArgs a) {
  using V4 = typename Vec<TO>::v4;
  constexpr int EB = sizeof(TI);             // bytes per operand element
  constexpr int XR = 32 * TN;                // activation rows per tile
  constexpr int WBYTES = 256 * 128, XBYTES = XR * 128, STAGE = WBYTES + XBYTES;
  constexpr int XROUNDS = XR / 64;           // 64 rows per fill round (512 threads x 16 bytes)
  constexpr int NG = 4 + XROUNDS;            // global -> LDS pieces per thread and K step
  static_assert(TN == 2 || TN == 4, "activation rows per tile: 64 or 128");
  __shared__ __attribute__((aligned(16))) uint8_t lds[3 * STAGE];

  // ---- which tile ----------------------------------------------------------------------------
  const int m_tiles = GROUPED ? min(*a.num_tiles, a.m_tiles) : a.m_tiles;
  int mi, ni;
  if (!tile_of_block(m_tiles, a.n_tiles, mi, ni)) return;
  int e = 0, beg = 0, cnt;
  if (GROUPED) {
    e = a.tile_expert[mi];
    beg = a.tile_beg[mi];
    cnt = min(a.tile_end[mi] - beg, XR);
  } else {
    beg = mi * XR;
    cnt = min(a.M - beg, XR);
  }
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int wr = wave >> 1, wc = wave & 1;
  const int n0 = ni * (EPI == EPI_GATE_UP ? 128 : 256);
  const int w_rows = EPI == EPI_GATE_UP ? 2 * a.N : a.N;
  const long kbytes = (long)a.K * EB;
  const uint8_t* wbase = reinterpret_cast<const uint8_t*>(a.w) + (long)e * a.w_expert_stride * EB;
  const uint8_t* xbase = reinterpret_cast<const uint8_t*>(a.x);

  // ---- staging roles: thread t of round j fills LDS row 64 j + (t >> 3), slot t & 7 -----------------
  const int srow = tid >> 3, slot = tid & 7;
  const uint8_t* wsrc[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int rho = 64 * j + srow;
    int row = EPI == EPI_GATE_UP ? (rho < 128 ? n0 + rho : a.N + n0 + rho - 128) : n0 + rho;
    row = min(row, w_rows - 1);
    wsrc[j] = wbase + (long)row * kbytes + ((slot ^ swz(rho)) << 4);
  }
  const uint8_t* xsrc[XROUNDS];
#pragma unroll
  for (int j = 0; j < XROUNDS; ++j) {
    const int tau = 64 * j + srow;
    const int pos = beg + min(tau, cnt - 1);
    long row = pos;
    if (GROUPED) {
      const int p = a.sorted[pos];
      row = (EPI == EPI_GATE_UP || EPI == EPI_UP_ACT) ? p / a.top_k : p;
    }
    xsrc[j] = xbase + row * a.x_stride * EB + ((slot ^ swz(tau)) << 4);
  }
  // Experts: each weight panel starts at a K step of its own (the m-tiles that share it, at the same one), since rows are a power of two
  // apart in most models, and panels all read at the same column fall on few memory channels.  Layers, us, all from the first -> so: bf16, 64
  // experts of 1024 x 2048, 333 tokens 211 -> 184, 700 247 -> 226; 60 of 1408 x 2048, 700 tokens 265 -> 236; e4m3, 16 of 6400 x 4096, 128
  // tokens 296 -> 277, 700 350 -> 332.  On the 256-row tiles below, bound by the matrix cores, it gave nothing (3088 / 3096).
  const int nk = (int)(kbytes >> 7), turn = GROUPED ? (ni * 5 + e * 3) % nk : 0;
  auto step_at = [&](int kt) { return kt + turn < nk ? kt + turn : kt + turn - nk; };
  auto stage = [&](int kt) {                  // ring slot kt % 3 <- K step min(kt, nk - 1) (a re-fill of the
    uint8_t* lw = lds + (kt % 3) * STAGE + wave * 1024;      // last step keeps the operation count uniform)
    uint8_t* lx = lw + WBYTES;
    const long ko = (long)step_at(min(kt, nk - 1)) * 128;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      glds16(wsrc[j] + ko, lw + j * 8192);
#pragma unroll
    for (int j = 0; j < XROUNDS; ++j)
      glds16(xsrc[j] + ko, lx + j * 8192);
  };

  // ---- compute roles -----------------------------------------------------------------------------------
  // weight m-tile mt (0..3) of this wave starts at LDS row: gate/up tiles hold 128 gate rows, then the 128 up
  // rows of the same columns, and a wave takes two gate tiles and the up tiles of the same 32 columns
  auto wrow = [&](int mt) { return EPI == EPI_GATE_UP ? (mt < 2 ? 32 * wr + 16 * mt : 128 + 32 * wr + 16 * (mt - 2))
                                                      : 64 * wr + 16 * mt; };
  const int f = swz(r);                        // tile rows start at multiples of 16: f depends on r only
  const int c0 = ((2 * g) ^ f) << 4, c1 = ((2 * g + 1) ^ f) << 4;
  int woff[4], xoff[TN];
#pragma unroll
  for (int mt = 0; mt < 4; ++mt) woff[mt] = (wrow(mt) + r) * 128;
#pragma unroll
  for (int nt = 0; nt < TN; ++nt) xoff[nt] = WBYTES + (16 * TN * wc + 16 * nt + r) * 128;

  f32x4 acc[4][TN];
#pragma unroll
  for (int mt = 0; mt < 4; ++mt)
#pragma unroll
    for (int nt = 0; nt < TN; ++nt) acc[mt][nt] = f32x4{0, 0, 0, 0};

  // SC_BLOCK: activation-group scale rows of this lane's tokens, weight-block scale rows of its m-tiles
  const float* xs_row[TN];
  const float* ws_row[4];
  const int kblocks = a.K >> 7;
  if (SC == SC_BLOCK) {
#pragma unroll
    for (int nt = 0; nt < TN; ++nt) {
      const int tau = 16 * TN * wc + 16 * nt + r;
      const int pos = beg + min(tau, cnt - 1);
      long row = pos;
      if (GROUPED) {
        const int p = a.sorted[pos];
        row = (EPI == EPI_GATE_UP || EPI == EPI_UP_ACT) ? p / a.top_k : p;
      }
      xs_row[nt] = a.x_scale + row * kblocks;
    }
    const int nblocks = (w_rows + 127) >> 7;
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
      const int rho = wrow(mt);
      int row = EPI == EPI_GATE_UP ? (rho < 128 ? n0 + rho : a.N + n0 + rho - 128) : n0 + rho;
      row = min(row, w_rows - 1);
      ws_row[mt] = a.w_scale + ((long)e * nblocks + (row >> 7)) * kblocks;
    }
  }

  stage(0);
  stage(1);
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NG) : "memory");          // step 0 has landed, step 1 is in flight
  __builtin_amdgcn_s_barrier();
  for (int kt = 0; kt < nk; ++kt) {
    stage(kt + 2);                             // into the slot read during step kt - 1 (all waves are past it)
    float sx[TN], sw[4];
    if (SC == SC_BLOCK) {
#pragma unroll
      for (int nt = 0; nt < TN; ++nt) sx[nt] = xs_row[nt][step_at(kt)];
#pragma unroll
      for (int mt = 0; mt < 4; ++mt) sw[mt] = ws_row[mt][step_at(kt)];
    }
    const uint8_t* base = lds + (kt % 3) * STAGE;
    i32x4 wa[4][2], xb[TN][2];
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
      wa[mt][0] = *reinterpret_cast<const i32x4*>(base + woff[mt] + c0);
      wa[mt][1] = *reinterpret_cast<const i32x4*>(base + woff[mt] + c1);
    }
#pragma unroll
    for (int nt = 0; nt < TN; ++nt) {
      xb[nt][0] = *reinterpret_cast<const i32x4*>(base + xoff[nt] + c0);
      xb[nt][1] = *reinterpret_cast<const i32x4*>(base + xoff[nt] + c1);
    }
#pragma unroll
    for (int nt = 0; nt < TN; ++nt)
#pragma unroll
      for (int mt = 0; mt < 4; ++mt) {
        if (SC == SC_BLOCK) {
          const f32x4 p = mma(wa[mt][0], wa[mt][1], xb[nt][0], xb[nt][1], f32x4{0, 0, 0, 0}, TI{});
          const float s = sw[mt] * sx[nt];
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[mt][nt][i] += p[i] * s;
        } else {
          acc[mt][nt] = mma(wa[mt][0], wa[mt][1], xb[nt][0], xb[nt][1], acc[mt][nt], TI{});
        }
      }
    // step kt + 1 must have landed before anyone reads it; the fill of step kt + 2 stays in flight.
    // (SC_BLOCK reads its scales with ordinary loads: they are older than that fill and done by now.)
    // This step's LDS reads are retired too (lgkmcnt): the next step's fill overwrites the slot they read.
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(NG) : "memory");
    __builtin_amdgcn_s_barrier();
  }

  // ---- epilogue: lane holds out[token tau(nt)][n(mt) + 4 g + i] -----------------------------------------
  const float wsc = SC == SC_TOKEN ? a.w_scale[e] : 1.f;
#pragma unroll
  for (int nt = 0; nt < TN; ++nt) {
    const int tau = 16 * TN * wc + 16 * nt + r;
    if (tau >= cnt) continue;
    long orow = beg + tau;
    float s = wsc;
    float tw = 1.f;
    if (GROUPED) {
      const int p = a.sorted[beg + tau];
      orow = p;
      if (SC == SC_TOKEN) s *= a.x_scale[(EPI == EPI_GATE_UP || EPI == EPI_UP_ACT) ? p / a.top_k : p];
      if (EPI == EPI_DOWN) tw = a.topk_w[p];
    } else if (SC == SC_TOKEN) {
      s *= a.x_scale[orow];
    }
    TO* op = reinterpret_cast<TO*>(a.out) + orow * a.out_stride;
    if (EPI == EPI_GATE_UP) {
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) {
        const int n = n0 + 32 * wr + 16 * mt + 4 * g;
        V4 o;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float gte = acc[mt][nt][i] * s, up = acc[mt + 2][nt][i] * s;
          o[i] = (TO)gated_pair(gte, up, a.act, a.act_limit);
        }
        if (n + 3 < a.N) *reinterpret_cast<V4*>(op + n) = o;
        else
          for (int i = 0; i < 4; ++i) if (n + i < a.N) op[n + i] = o[i];
      }
    } else {
#pragma unroll
      for (int mt = 0; mt < 4; ++mt) {
        const int n = n0 + 64 * wr + 16 * mt + 4 * g;
        V4 o;
        V4 bv = V4{};
        if (EPI == EPI_PLAIN && a.bias && n + 3 < a.N) bv = *reinterpret_cast<const V4*>(reinterpret_cast<const TO*>(a.bias) + n);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float v = acc[mt][nt][i] * s * tw;
          if (EPI == EPI_PLAIN && a.bias) v += n + 3 < a.N ? (float)bv[i] : (n + i < a.N ? (float)reinterpret_cast<const TO*>(a.bias)[n + i] : 0.f);
          if (EPI == EPI_UP_ACT) v = gate_act(v, a.act);
          o[i] = (TO)v;
        }
        if (n + 3 < a.N) *reinterpret_cast<V4*>(op + n) = o;
        else
          for (int i = 0; i < 4; ++i) if (n + i < a.N) op[n + i] = o[i];
      }
    }
  }
}

// ---------------------------------------------------------------------------------------------
// Grouped 16-bit GEMM on tiles of 256 weight rows x up to 288 activation rows, for experts that see more than 128 rows each.
// Four waves, one a SIMD, as 2 (weight rows) x 2 (activation rows): a wave holds 8 x NF accumulator tiles of 16 x 16 and reads
// 17 KB of LDS operands per 72 MFMAs (eight waves of 4 x 8 tiles read 12 per 32, which with the fill is all that an LDS
// delivers in that time).  K is walked in units of 64 elements, whole 128-byte lines of a row (half lines, in steps of 32, kept the L2
// busy with twice the requests), through two LDS slots, a unit in two halves.  Dealt out between the MFMAs of unit u:
//
//   half 0: to three quarters, the reads of half 1 (second register set); barrier: the slot of unit u is free
//   from there to three quarters of half 1: the copies of unit u + 2 into it
//   half 1: at a quarter, wait for the own copies of unit u + 1; barrier; then the reads of its half 0
//
// so a copy has one and a half to two and a half halves of MFMAs to arrive.  Write-after-read: copies of unit u + 2 follow a barrier that every
// wave reaches with its reads of unit u done.  Read-after-write: the reads of unit u + 1 follow one that every wave reaches
// with its copies of it landed (the AHEAD younger ones may be in flight).
//
// An expert's rows are cut into the fewest tiles of at most 288 rows, of like sizes (align_tiles in moe.hip): batches of 2048 or
// 4096 tokens over eight experts are 256-row tiles but for a few rows, which opened tiles of their own in half of the experts.
// NF, the 16-row fragments of a wave, is a template argument: tiles of few rows do few MFMAs.
//
// LDS image of a slot: [row][8 chunks of 16 bytes], chunk c of row r at c ^ ((r >> 1) & 7), on the source side of the copy.  Of a fragment read
// the lanes of rows {0-3, 12-15} at chunk q are served with those of {4-11} at q ^ 1: they touch the sixteen 16-byte columns of
// a 256-byte bank row once each.
// What bounds it: the MFMAs run 70 % of the cycles, at a clock that the chip's power takes down to 1.7 GHz of 2.4; without copies the
// second product of 8 experts 4096 x 14336 over 8198 rows takes 617 us (1.56 PFLOP/s, a large library product reaches 1.60), with them 760;
// the results of the first, which leave in bursts with the MFMAs idle, are a tenth of it.  Asking the L2 ahead for a share of each line made it 3 % slower.
// us, eight waves of 64 x 128 sums -> this, whole layer: 4099 tokens of 8 experts 4096 x 14336, top 2, 2940 -> 2260 (1.28 PFLOP/s with rows that
// exist); 4096 of 64 experts 2048 x 1024, top 8, 576 -> 469; 4096 of 16 experts 4096 x 6400 1453 -> 1151.
constexpr int WIDE_UNIT = (256 + WIDE_ROWS) * 128;

// 16 bytes a lane from a buffer to LDS, at dst + 16 * lane.  As a statement of its own: told of the copy, the compiler waits for
// all of them before the next LDS read, although they fill another slot of the ring.  Waited for by the counts in the loop.
__device__ __forceinline__ void wide_copy(i32x4 buf, unsigned voff, int soff, unsigned dst) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               ::"s"(dst), "v"(voff), "s"(buf), "s"(soff) : "memory", "m0");
}
__device__ __forceinline__ i32x4 wide_buffer(const void* p) {
  const uint64_t at = reinterpret_cast<uint64_t>(p);
  return i32x4{__builtin_amdgcn_readfirstlane((int)(uint32_t)at), __builtin_amdgcn_readfirstlane((int)((at >> 32) & 0xffff)), -1, 0x00020000};
}

// c += a b as a statement, with the sums in accumulator registers (ACC) or, the 32 that are more than 256, in ordinary ones: left to
// itself the compiler moves hundreds of them to and fro in each step.  It does not look into these: operands come from LDS
// reads that the loop waits for, sums are touched again sixteen MFMAs later at the earliest, and the loop is followed by enough
// wait states for a reader.
template <bool ACC> __device__ __forceinline__ void wide_mfma(f32x4& c, bf16x8 a, bf16x8 b) {
  if (ACC) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
  else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
}
template <bool ACC> __device__ __forceinline__ void wide_mfma(f32x4& c, f16x8 a, f16x8 b) {
  if (ACC) asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
  else asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
}

// gate_act and gated_pair with the choice made once for four values
__device__ __forceinline__ f32x4 gate_four(f32x4 g, int kind) {
  auto all = [&](int k) { return f32x4{gate_act(g[0], k), gate_act(g[1], k), gate_act(g[2], k), gate_act(g[3], k)}; };
  switch (kind) {
    case 1: return all(1);
    case 2: return all(2);
    case 3: return all(3);
    case 8: return all(8);
    default: return all(0);
  }
}
__device__ __forceinline__ f32x4 gated_four(f32x4 g, f32x4 u, int kind, float limit) {
  if (kind == 9) {
#pragma unroll
    for (int i = 0; i < 4; ++i) g[i] = gated_pair(g[i], u[i], 9, limit);
    return g;
  }
  return gate_four(g, kind) * u;
}

// one tile: acc[mt][nt] = the sum over K of W fragment mt . X fragment nt, then the epilogue.  pair, tw: the pair of each row
// of the tile and its routing weight, in LDS
template <typename T, int EPI, int NF>
__device__ __forceinline__ void wide_walk(const TileGemmArgs& a, uint8_t* lds, const int* pair, const float* tw, int e, int beg, int cnt,
                                          int n0) {
  using V8 = typename Vec<T>::v8;
  using V4 = typename Vec<T>::v4;
  constexpr int WT = 8, CP = 8 + NF, READS = WT + NF;  // copies of 1 KB of a wave in a unit, and its fragment reads in half of one
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int wi = wave & 1, xi = wave >> 1;
  const int w_rows = EPI == EPI_GATE_UP ? 2 * a.N : a.N;
  const unsigned kbytes = (unsigned)a.K * 2u;
  const i32x4 wbuf = wide_buffer(reinterpret_cast<const uint8_t*>(a.w) + (long)e * a.w_expert_stride * 2), xbuf = wide_buffer(a.x);
  const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds;

  // copies: lane L of a 1 KB piece fills row L >> 3 of its eight, position L & 7.  Wave w takes pieces w, w + 4, ...
  unsigned voff[CP];                         // (host: both operands of an expert below 4 GiB)
  {
    const int lrow = lane >> 3, chunk = ((lane & 7) ^ ((4 * wave + (lrow >> 1)) & 7)) << 4;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int rho = 8 * (wave + 4 * j) + lrow;
      const int row = EPI == EPI_GATE_UP ? (rho < 128 ? n0 + rho : a.N + n0 + rho - 128) : n0 + rho;
      voff[j] = (unsigned)min(row, w_rows - 1) * kbytes + chunk;
    }
#pragma unroll
    for (int j = 0; j < NF; ++j) {
      const int p = pair[min(8 * (wave + 4 * j) + lrow, cnt - 1)];
      const int xrow = EPI == EPI_DOWN ? p : p / a.top_k;
      voff[8 + j] = (unsigned)xrow * (unsigned)(a.x_stride * 2) + chunk;
    }
  }
  const int units = a.K >> 6;
  auto copy = [&](int u, int j) {            // piece j of unit u (the last unit's again beyond the end: into a slot that is free)
    wide_copy(j < 8 ? wbuf : xbuf, voff[j], min(u, units - 1) * 128,
              lds0 + (u & 1) * WIDE_UNIT + (j < 8 ? 0 : 256 * 128) + (wave + 4 * (j < 8 ? j : j - 8)) * 1024);
  };
  // weight fragment mt of wave column wi starts at tile row wrow(mt); with a gate half four are gate rows and four the up rows of
  // the same columns
  auto wrow = [&](int mt) { return EPI == EPI_GATE_UP ? (mt < 4 ? 64 * wi + 16 * mt : 128 + 64 * wi + 16 * (mt - 4))
                                                      : 128 * wi + 16 * mt; };
  const int cpos = r * 128 + ((g ^ (r >> 1)) << 4);    // half 0 of a unit; half 1 is at cpos ^ 64
  f32x4 acc[WT][NF];
#pragma unroll
  for (int mt = 0; mt < WT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NF; ++nt) acc[mt][nt] = f32x4{0, 0, 0, 0};
  V8 wf[2][WT], xf[2][NF];
  auto read = [&](int u, int h, int i) {     // fragment i of half h, in the order in which they are needed
    const uint8_t* slot = lds + (u & 1) * WIDE_UNIT + (h ? cpos ^ 64 : cpos);
    if (i < WT) wf[h][i] = *reinterpret_cast<const V8*>(slot + wrow(0) * 128 + (wrow(i) - wrow(0)) * 128);
    else xf[h][i - WT] = *reinterpret_cast<const V8*>(slot + (256 + 16 * NF * xi) * 128 + (i - WT) * 2048);
  };

#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int j = 0; j < CP; ++j) copy(u, j);
  asm volatile("s_waitcnt vmcnt(%0)" ::"i"(CP) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
#pragma unroll
  for (int i = 0; i < READS; ++i) read(0, 0, i);
  constexpr int ALL = WT * NF, FREE = ALL * 3 / 4, LAND = ALL / 4;
  // n operations over w places: how many stand before place i
  auto upto = [](int i, int n, int w) constexpr { return (i * n + w - 1) / w; };
  constexpr int AHEAD = ((ALL + LAND - FREE) * CP + ALL - 1) / ALL;      // copies of unit u + 2 before unit u + 1 is waited for
  static_assert(READS <= FREE && CP <= ALL, "one read and one copy behind an MFMA at most");
  for (int u = 0; u < units; ++u) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int m = 0; m < ALL; ++m) {
        if (h == 0 && m == FREE) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (h == 1 && m == LAND) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"i"(AHEAD) : "memory");
        const int nt = m / WT, mt = m % WT;
        if (nt < 8) wide_mfma<true>(acc[mt][nt], wf[h][mt], xf[h][nt]);
        else wide_mfma<false>(acc[mt][nt], wf[h][mt], xf[h][nt]);
        const int i = h ? m - LAND : m, before = upto(i, READS, FREE);
        if (i >= 0 && i < FREE && upto(i + 1, READS, FREE) > before) read(u + h, 1 - h, before);
        const int c = h * ALL + m - FREE, done = upto(c, CP, ALL);
        if (c >= 0 && c < ALL && upto(c + 1, CP, ALL) > done) copy(u + 2, done);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_nop 15\n\ts_nop 7" ::: "memory");

  // ---- a lane holds rows 16 (NF xi + nt) + r, columns 4 g + i of fragment mt.  Four nt at a time through this wave's quarter of the
  // ring, so that a row is stored in 128 bytes or more at once ----
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  constexpr int CG = EPI == EPI_GATE_UP ? 16 : 32;     // lanes of a row, four columns each
  constexpr int ROW = 4 * 16 * WT + 16;                // bytes between rows: 16-byte columns of a bank row in turn
  uint8_t* mine = lds + wave * (WIDE_UNIT / 2);
  static_assert(64 * ROW <= WIDE_UNIT / 2, "four fragments of rows fit a quarter");
#pragma unroll
  for (int q = 0; q < NF; q += 4) {
    constexpr int Q = 4;
    const int rows = 16 * (NF - q < Q ? NF - q : Q);
#pragma unroll
    for (int nt = q; nt < NF && nt < q + Q; ++nt)
#pragma unroll
      for (int mt = 0; mt < WT; ++mt)
        *reinterpret_cast<f32x4*>(mine + (16 * (nt - q) + r) * ROW + 64 * mt + 16 * g) = acc[mt][nt];
    asm volatile("" ::: "memory");
    auto store = [&](auto finish) {
#pragma unroll 4                                       // several rows in flight: a wave is alone on its SIMD
      for (int i0 = 0; i0 < rows; i0 += 64 / CG) {
        const int row = i0 + lane / CG, token = 16 * (NF * xi + q) + row, cl = 4 * (lane % CG);
        const int n = n0 + (EPI == EPI_GATE_UP ? 64 : 128) * wi + cl;
        f32x4 v = *reinterpret_cast<const f32x4*>(mine + row * ROW + 4 * cl), u = v;
        if (EPI == EPI_GATE_UP) u = *reinterpret_cast<const f32x4*>(mine + row * ROW + 256 + 4 * cl);
        v = finish(v, u, token);
        T* op = reinterpret_cast<T*>(a.out) + (long)pair[token] * a.out_stride + n;
        V4 o;
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = (T)v[i];
        if (token < cnt) {
          if (n + 3 < a.N) *reinterpret_cast<V4*>(op) = o;
          else
            for (int i = 0; i < 4; ++i) if (n + i < a.N) op[i] = o[i];
        }
      }
    };
    if (EPI == EPI_DOWN) store([&](f32x4 v, f32x4, int token) { return v * tw[token]; });
    else if (a.act == 0) store([&](f32x4 v, f32x4 u, int) { v = gate_four(v, 0); return EPI == EPI_GATE_UP ? v * u : v; });
    else store([&](f32x4 v, f32x4 u, int) { return EPI == EPI_GATE_UP ? gated_four(v, u, a.act, a.act_limit) : gate_four(v, a.act); });
    asm volatile("" ::: "memory");
  }
}

template <typename T, int EPI>
__global__ __launch_bounds__(256, 1) void moe_wide_gemm_kernel(const TileGemmArgs a) {
  __shared__ __attribute__((aligned(16))) uint8_t lds[2 * WIDE_UNIT];
  __shared__ int pair[WIDE_ROWS];
  __shared__ float tw[EPI == EPI_DOWN ? WIDE_ROWS : 1];
  int mi, ni;
  if (!tile_of_block(min(*a.num_tiles, a.m_tiles), a.n_tiles, mi, ni)) return;
  const int e = a.tile_expert[mi], beg = a.tile_beg[mi], cnt = min(a.tile_end[mi] - beg, WIDE_ROWS);
  const int n0 = ni * (EPI == EPI_GATE_UP ? 128 : 256);
  for (int i = threadIdx.x; i < cnt; i += 256) {
    const int p = a.sorted[beg + i];
    pair[i] = p;
    if (EPI == EPI_DOWN) tw[i] = a.topk_w[p];
  }
  __syncthreads();
  const auto walk = [&](auto nf) { wide_walk<T, EPI, decltype(nf)::value>(a, lds, pair, tw, e, beg, cnt, n0); };
  switch ((cnt + 31) >> 5) {
    case 9: return walk(std::integral_constant<int, 9>());
    case 8: return walk(std::integral_constant<int, 8>());
    case 7: return walk(std::integral_constant<int, 7>());
    case 6: return walk(std::integral_constant<int, 6>());
    case 5: return walk(std::integral_constant<int, 5>());
    case 4: case 3: return walk(std::integral_constant<int, 4>());
    default: return walk(std::integral_constant<int, 2>());
  }
}

// ---------------------------------------------------------------------------------------------
template <typename T>
static int launch_wide_gemm(const TileGemmArgs& a, int epi, hipStream_t st) {
  const dim3 grid(tile_blocks(a.m_tiles, a.n_tiles)), block(256);
  if (epi == EPI_GATE_UP) hipLaunchKernelGGL((moe_wide_gemm_kernel<T, EPI_GATE_UP>), grid, block, 0, st, a);
  else if (epi == EPI_DOWN) hipLaunchKernelGGL((moe_wide_gemm_kernel<T, EPI_DOWN>), grid, block, 0, st, a);
  else if (epi == EPI_UP_ACT) hipLaunchKernelGGL((moe_wide_gemm_kernel<T, EPI_UP_ACT>), grid, block, 0, st, a);
  else return -4;
  return 0;
}

// in_dtype: operand type (VDA_BF16 / VDA_F16 / VDA_FP8); out_dtype VDA_BF16 / VDA_F16.
// rows_per_tile: 128 or 64 activation rows per tile, or 256 (grouped 16-bit operands; M: rows of x, for its 32-bit
// offsets).  Grouped when sorted != nullptr.
template <typename TI, typename TO, int SC>
static int launch_tile_gemm(const TileGemmArgs& a, int epi, bool grouped, int rows_per_tile, hipStream_t st) {
  const dim3 grid(tile_blocks(a.m_tiles, a.n_tiles)), block(512);
#define LAUNCH(EPI, GR, TN) hipLaunchKernelGGL((tile_gemm_kernel<TI, TO, EPI, GR, SC, TN>), grid, block, 0, st, a)
#define BY_TN(EPI, GR) do { if (rows_per_tile == 128) LAUNCH(EPI, GR, 4); else LAUNCH(EPI, GR, 2); } while (0)
  if (grouped) {
    if (epi == EPI_GATE_UP) BY_TN(EPI_GATE_UP, true);
    else if (epi == EPI_DOWN) BY_TN(EPI_DOWN, true);
    else if (epi == EPI_UP_ACT) BY_TN(EPI_UP_ACT, true);
    else return -4;
  } else {
    if (epi != EPI_PLAIN) return -4;
    BY_TN(EPI_PLAIN, false);
  }
#undef BY_TN
#undef LAUNCH
  return 0;
}

VDA_EXPORT int vda_tile_gemm(void* out, const void* x, const void* w, const float* x_scale, const float* w_scale,
                             const float* topk_w, const void* bias, const int* sorted, const int* tile_expert,
                             const int* tile_beg, const int* tile_end, const int* num_tiles, int M, int N, int K,
                             int top_k, int max_m_tiles, long x_stride, long out_stride, long w_expert_stride,
                             int epi, int scale_mode, int rows_per_tile, int in_dtype, int out_dtype, int act,
                             float act_limit, hipStream_t st) {
  const bool grouped = sorted != nullptr;
  const int eb = in_dtype == VDA_FP8 ? 1 : 2;
  const bool wide = rows_per_tile == 256;
  if (rows_per_tile != 128 && rows_per_tile != 64 && !wide) return -1;
  if (wide && (!grouped || scale_mode != SC_NONE || in_dtype == VDA_FP8 || in_dtype != out_dtype || x_stride * 2 * (long)M >= (1L << 32)
               || w_expert_stride * 2 >= (1L << 32) || M < 1)) return -1;
  if (N < 1 || K < 1 || ((long)K * eb) % 128) return -1;
  if ((x_stride * eb) % 16 || (w_expert_stride * eb) % 16) return -1;       // 16-byte global_load_lds
  if (epi == EPI_GATE_UP && N % 64) return -1;
  if (N % 4 && out_stride % 4) return -1;
  if (scale_mode != SC_NONE && in_dtype != VDA_FP8) return -1;
  if (scale_mode != SC_NONE && (!x_scale || !w_scale)) return -1;
  if (scale_mode == SC_BLOCK && K % 128) return -1;
  if (grouped && (!tile_expert || !tile_beg || !tile_end || !num_tiles || max_m_tiles < 1)) return -1;
  if (!grouped && M < 1) return M == 0 ? 0 : -1;
  TileGemmArgs a;
  a.out = out; a.x = x; a.w = w; a.x_scale = x_scale; a.w_scale = w_scale; a.topk_w = topk_w; a.bias = bias;
  a.sorted = sorted; a.tile_expert = tile_expert; a.tile_beg = tile_beg; a.tile_end = tile_end; a.num_tiles = num_tiles;
  a.M = M; a.N = N; a.K = K; a.top_k = top_k > 0 ? top_k : 1; a.act = act; a.act_limit = act_limit;
  a.m_tiles = grouped ? max_m_tiles : (M + rows_per_tile - 1) / rows_per_tile;
  a.n_tiles = epi == EPI_GATE_UP ? (N + 127) / 128 : (N + 255) / 256;
  a.x_stride = x_stride; a.out_stride = out_stride; a.w_expert_stride = w_expert_stride;
  int rc;
#define BY_SC(TI, TO) (scale_mode == SC_NONE ? launch_tile_gemm<TI, TO, SC_NONE>(a, epi, grouped, rows_per_tile, st) \
    : scale_mode == SC_TOKEN ? launch_tile_gemm<TI, TO, SC_TOKEN>(a, epi, grouped, rows_per_tile, st) \
    : launch_tile_gemm<TI, TO, SC_BLOCK>(a, epi, grouped, rows_per_tile, st))
  if (wide) {
    rc = in_dtype == VDA_BF16 ? launch_wide_gemm<bf16_t>(a, epi, st) : launch_wide_gemm<f16_t>(a, epi, st);
  } else if (in_dtype == VDA_FP8) {
    if (scale_mode == SC_NONE) return -1;
    if (out_dtype == VDA_BF16) rc = BY_SC(uint8_t, bf16_t);
    else if (out_dtype == VDA_F16) rc = BY_SC(uint8_t, f16_t);
    else return -3;
  } else if (in_dtype == VDA_BF16 && out_dtype == VDA_BF16) {
    rc = launch_tile_gemm<bf16_t, bf16_t, SC_NONE>(a, epi, grouped, rows_per_tile, st);
  } else if (in_dtype == VDA_F16 && out_dtype == VDA_F16) {
    rc = launch_tile_gemm<f16_t, f16_t, SC_NONE>(a, epi, grouped, rows_per_tile, st);
  } else return -3;
#undef BY_SC
  if (rc) return rc;
  VDA_CHECK_LAUNCH();
  return 0;
}
