// Weight-only quantised GEMM for every M: out[M, N] = X[M, K] . dequant(Wq)[N, K]^T (+ bias), 4- or 8-bit weights
// with one (scale, zero) pair per output row and group of G input elements (value = (q - zero) * scale), 16-bit
// activations: GPTQ / AWQ W4A16, 8-bit GPTQ, GGUF Q4_0 / Q8_0 after repacking.  The weights stay packed in HBM and
// in LDS; they are widened to the activation type only on their way into the MFMA operand registers.
//
// Two kernels.  Few activation rows (decode): the weight stream is the whole cost, so wq_stream_kernel keeps
// it out of LDS altogether: packed words go global -> registers four K steps ahead, are
// widened in registers and fed to the MFMAs as the A operand, while the activations of a K step are shared by the
// waves through an LDS ring (the scheme of gemm_decode.hip with a quarter / half of its HBM bytes).  More rows:
// wq_tile_kernel, tiles of 256 weight rows by up to 256 activation rows, one wave a SIMD, whose vector instructions widen the next
// product's weights behind the MFMAs of this one.
//
// Layouts (made by ops.wq_pack_* at load time):
//   qweight 4 bit  uint32 [N, K / 8]: word j of row n holds K elements 8 j .. 8 j + 7, element e in nibble
//                  e / 2 + 4 * (e % 2): (w >> 4 i) & 0x000F000F is the pair (2 i, 2 i + 1) as two 16-bit fields
//   qweight 8 bit  uint8 [N, K]: unsigned bytes (signed formats are stored + 128 with zero = 128)
//   sz             T [K / G, N, 2]: (scale, zero) of row n in group k / G; G a multiple of 32
// Takes the place of the reference's csrc/quantization/gptq/q_gemm.cu:1815 (exllama GEMM), awq/gemm_kernels.cu,
// gptq_marlin/ (W4A16 / W8A16 for any batch) and gguf/gguf_kernel.cu:91,207 for the formats above.
#include <type_traits>

#include "gemm_dense.h"

struct WqGemmArgs {
  DenseGemmArgs d;        // out, x, bias, residual, ws, M, N, K, tiles, splits, strides (d.w: packed weights)
  const void* sz;         // [K / G, N, 2]
  int group;              // G
  int gshift;             // log2(G / 32) when G is a power of two (30 when one group spans K), else -1
  unsigned group_magic;   // see wq_group_of
  int per_element;        // streaming kernel: scale every weight element even where the unscaled form applies
};

template <typename T, int BITS>
__device__ __forceinline__ typename Vec<T>::v8 wq_expand(const uint32_t* q, float s, float nzs) {
  typename Vec<T>::v8 o;
  if (BITS == 4) {
    const uint32_t lo = q[0] & 0x0F0F0F0Fu, hi = (q[0] >> 4) & 0x0F0F0F0Fu;
    o[0] = (T)fmaf((float)(lo & 0xff), s, nzs);
    o[4] = (T)fmaf((float)((lo >> 8) & 0xff), s, nzs);
    o[1] = (T)fmaf((float)((lo >> 16) & 0xff), s, nzs);
    o[5] = (T)fmaf((float)(lo >> 24), s, nzs);
    o[2] = (T)fmaf((float)(hi & 0xff), s, nzs);
    o[6] = (T)fmaf((float)((hi >> 8) & 0xff), s, nzs);
    o[3] = (T)fmaf((float)((hi >> 16) & 0xff), s, nzs);
    o[7] = (T)fmaf((float)(hi >> 24), s, nzs);
  } else {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      o[4 * h + 0] = (T)fmaf((float)(q[h] & 0xff), s, nzs);
      o[4 * h + 1] = (T)fmaf((float)((q[h] >> 8) & 0xff), s, nzs);
      o[4 * h + 2] = (T)fmaf((float)((q[h] >> 16) & 0xff), s, nzs);
      o[4 * h + 3] = (T)fmaf((float)(q[h] >> 24), s, nzs);
    }
  }
  return o;
}

// ---- decode: weights global -> registers, activations through an LDS ring -----------------------------------
// A K step is 128 elements.  Lane (r, g) of a wave holds, for each of the wave's two 16-row weight fragments, the
// 32 consecutive elements [128 kt + 32 g, + 32) of row r (16 bytes of nibbles / 32 bytes) and that row's
// (scale, zero) pair; MFMA j of the step multiplies elements 32 g + 8 j .. + 7, so the activation operand of lane
// (c, g) is the 16-byte chunk 4 g + j of activation row c's 256 bytes.  The ring stores chunk i of row c at
// position i ^ (c & 15): the sixteen lanes of one g read sixteen different positions (all 64 banks, once each).
// Vector-memory operations complete in order: every iteration issues one ring fill and then one weight step and
// waits with a counted s_waitcnt for the fill the next iteration reads; the weight steps are issued from inline
// assembly so the compiler cannot drain the queue at the loop head.
//
// POST (4-bit weights whose groups are whole K steps): the weights enter the MFMAs unscaled.  Or-ing a float's
// exponent over a nibble field makes the 16-bit float BIAS + q (BIAS = 128 for bf16, 1024 for fp16, both exact), so
// a packed word becomes an operand register pair by pair with one shift and one and-or; a third MFMA per step
// multiplies the activations by ones, and at the end of a group
//     total += scale * (sum_k (BIAS + q_k) x_k  -  (BIAS + zero) * sum_k x_k)
// in fp32 on the accumulators: 2 x 4 fused multiply-adds per fragment instead of a convert, a multiply-add and a
// pack per weight element, which is what bounds the per-element form below the HBM rate.
template <typename T> struct WqMagic;
template <> struct WqMagic<bf16_t> { static constexpr uint32_t OR = 0x43004300u; static constexpr float BIAS = 128.f; };
template <> struct WqMagic<f16_t> { static constexpr uint32_t OR = 0x64006400u; static constexpr float BIAS = 1024.f; };

template <typename T, int BITS, int MT16, int WM, bool POST>
__global__ __launch_bounds__(256 * WM, WM == 1 ? 2 : 1) void wq_stream_kernel(const WqGemmArgs wa) {
  using V8 = typename Vec<T>::v8;
  using V4 = typename Vec<T>::v4;
  const DenseGemmArgs& a = wa.d;
  constexpr int WAVES = 4 * WM;
  constexpr int SX = 4;                                // activation ring depth (filled three steps ahead)
  constexpr int DW = 4;                                // weight steps in registers (eight: 57344 x 8192 in 4 bits 66 us, four 62)
  static_assert(!POST || BITS == 4, "unscaled operands exist for 4-bit weights only");
  constexpr int NQ = BITS / 4;                         // 16-byte loads per fragment and step
  constexpr int LW = 2 * NQ + 2;                       // vector-memory operations of one weight step
  constexpr int STEPB = 16 * BITS;                     // packed bytes of one row in a step
  constexpr int XB = MT16 * WM * 16 * 256;             // bytes of one ring slot
  constexpr int P = MT16;                              // 1 KiB pieces per wave per ring slot
  static_assert(P * WAVES * 1024 == XB, "rows must divide over the waves");
  // issued after the ring fill that the next iteration reads: three weight steps and two fills
  constexpr int YOUNGER = 3 * LW + 2 * P;
  static_assert(YOUNGER < 64, "vmcnt is a 6-bit counter");
  __shared__ __attribute__((aligned(16))) uint8_t lds[SX * XB];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int wr = wave & 3, wm = wave >> 2;
  const int n0 = (blockIdx.x * 4 + wr) * 32;
  const int nk_all = a.K >> 7;
  const int kt0 = blockIdx.y * a.units_per_split;
  const int nk = min(a.units_per_split, nk_all - kt0);           // >= 1 by the host's choice of splits
  // Where this workgroup starts: at a group's first step, another one for each workgroup.  Rows are a power of two apart in most
  // models: with all workgroups at the same column of their rows, what they read falls on few memory channels (13 activation
  // rows, 57344 x 8192: 4 bits 71.6 -> 66.1 us, 8 bits 112 -> 104).
  int turn = 0;
  {
    const int per = wa.gshift <= 2 ? 1 : 1 << (wa.gshift - 2);   // steps of a group
    if (a.splits == 1 && wa.gshift < 30 && nk % per == 0) turn = (int)(blockIdx.x * 5u % (unsigned)(nk / per)) * per;
  }
  auto at_step = [&](int kt) {                                   // past the end: any step
    const int t = min(kt, nk - 1) + turn;
    return t < nk ? t : t - nk;
  };

  const uint8_t* wp[2];
  const uint8_t* sp[2];
#pragma unroll
  for (int mt = 0; mt < 2; ++mt) {
    const int row = min(n0 + 16 * mt + r, a.N - 1);
    wp[mt] = reinterpret_cast<const uint8_t*>(a.w) + (long)row * ((long)a.K * BITS / 8) + (long)kt0 * STEPB + g * (STEPB / 4);
    // per-element form: the pair of the lane's own row; POST: the pairs of the four output rows 4 g .. 4 g + 3
    sp[mt] = reinterpret_cast<const uint8_t*>(wa.sz) + (POST ? (long)min(n0 + 16 * mt + 4 * g, a.N - 4) * 4 : (long)row * 4);
  }
  const uint8_t* xp[P];
#pragma unroll
  for (int j = 0; j < P; ++j) {
    const int tau = 4 * WAVES * j + (tid >> 4);
    const long row = min(tau, a.M - 1);
    xp[j] = reinterpret_cast<const uint8_t*>(a.x) + row * a.x_stride * 2 + (long)kt0 * 256 + (((tid & 15) ^ (tau & 15)) << 4);
  }
  auto fill = [&](int kt) {          // ring slot kt % 4 <- K step min(kt, nk - 1)
    const long ko = (long)at_step(kt) * 256;
    uint8_t* dst = lds + (kt & 3) * XB + wave * 1024;
#pragma unroll
    for (int j = 0; j < P; ++j) glds16(xp[j] + ko, dst + j * WAVES * 1024);
  };
  i32x4 wreg[DW][2][NQ];
  typename std::conditional<POST, i32x4, uint32_t>::type sreg[DW][2];
  const long plane = (long)a.N * 4;
  auto wload = [&](int u, int kt) {
    const int kk = at_step(kt);
    const long so = (long)((((kt0 + kk) << 2) + g) >> wa.gshift) * plane;
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
      const uint8_t* p = wp[mt] + (long)kk * STEPB;
      if constexpr (NQ == 1)
        asm volatile("global_load_dwordx4 %0, %1, off" : "=&v"(wreg[u][mt][0]) : "v"(p) : "memory");
      else
        asm volatile("global_load_dwordx4 %0, %2, off nt\n\tglobal_load_dwordx4 %1, %2, off offset:16 nt"
                     : "=&v"(wreg[u][mt][0]), "=&v"(wreg[u][mt][NQ - 1]) : "v"(p) : "memory");
    }
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
      const uint8_t* p = sp[mt] + so;
      if constexpr (POST) asm volatile("global_load_dwordx4 %0, %1, off" : "=&v"(sreg[u][mt]) : "v"(p) : "memory");
      else asm volatile("global_load_dword %0, %1, off" : "=&v"(sreg[u][mt]) : "v"(p) : "memory");
    }
  };

  f32x4 acc[2][MT16];
  f32x4 part[POST ? 2 : 1][POST ? MT16 : 1], xsum[POST ? MT16 : 1];      // POST: this group's unscaled sums
#pragma unroll
  for (int mt = 0; mt < 2; ++mt)
#pragma unroll
    for (int nt = 0; nt < MT16; ++nt) acc[mt][nt] = f32x4{0, 0, 0, 0};
  if constexpr (POST) {
#pragma unroll
    for (int nt = 0; nt < MT16; ++nt) { part[0][nt] = part[1][nt] = xsum[nt] = f32x4{0, 0, 0, 0}; }
  }
  V8 ones;
#pragma unroll
  for (int i = 0; i < 8; ++i) ones[i] = (T)1.f;

  // prologue in the loop's own order (W .. W | X0 W X1 W X2 W), so the same counted wait holds from the start
#pragma unroll
  for (int u = 0; u < DW - 3; ++u) wload(u, u);
#pragma unroll
  for (int u = 0; u < 3; ++u) { fill(u); wload(DW - 3 + u, DW - 3 + u); }
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(YOUNGER) : "memory");      // X0 and every weight step before it
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);

  for (int kb = 0; kb < nk; kb += DW) {
#pragma unroll
    for (int u = 0; u < DW; ++u) {
      const int kt = kb + u;
      fill(kt + 3);                                                  // slot (kt - 1) % 4: read last iteration
      if (kt < nk) {
        const uint8_t* base = lds + (u & 3) * XB + (wm * MT16 * 16 + r) * 256;
        if constexpr (POST) {
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            V8 wf[2];
#pragma unroll
            for (int mt = 0; mt < 2; ++mt) {
              const uint32_t w = (uint32_t)wreg[u][mt][0][j];
              const u32x4 d = {(w & 0x000F000Fu) | WqMagic<T>::OR, ((w >> 4) & 0x000F000Fu) | WqMagic<T>::OR,
                               ((w >> 8) & 0x000F000Fu) | WqMagic<T>::OR, ((w >> 12) & 0x000F000Fu) | WqMagic<T>::OR};
              wf[mt] = __builtin_bit_cast(V8, d);
            }
            const int ch = ((4 * g + j) ^ r) << 4;
#pragma unroll
            for (int nt = 0; nt < MT16; ++nt) {
              const V8 xf = *reinterpret_cast<const V8*>(base + nt * 4096 + ch);
              part[0][nt] = mfma16(wf[0], xf, part[0][nt]);
              part[1][nt] = mfma16(wf[1], xf, part[1][nt]);
              xsum[nt] = mfma16(ones, xf, xsum[nt]);
            }
          }
          const int here = (kt0 + at_step(kt)) << 2;
          if ((here >> wa.gshift) != ((here + 4) >> wa.gshift) || kt + 1 == nk) {   // the group ends with this step
#pragma unroll
            for (int mt = 0; mt < 2; ++mt) {
              const V8 pv = __builtin_bit_cast(V8, sreg[u][mt]);               // (scale, zero) of rows 4 g .. 4 g + 3
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                const float s = (float)pv[2 * i], zb = (float)pv[2 * i + 1] + WqMagic<T>::BIAS;
#pragma unroll
                for (int nt = 0; nt < MT16; ++nt) {
                  acc[mt][nt][i] = fmaf(s, fmaf(-zb, xsum[nt][i], part[mt][nt][i]), acc[mt][nt][i]);
                  part[mt][nt][i] = 0.f;
                }
              }
            }
#pragma unroll
            for (int nt = 0; nt < MT16; ++nt) xsum[nt] = f32x4{0, 0, 0, 0};
          }
        } else {
        float sc[2], nz[2];
#pragma unroll
        for (int mt = 0; mt < 2; ++mt) {
          const V4 pv = __builtin_bit_cast(V4, u32x2{sreg[u][mt], 0u});
          sc[mt] = (float)pv[0];
          nz[mt] = -(float)pv[1] * sc[mt];
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          V8 wf[2];
#pragma unroll
          for (int mt = 0; mt < 2; ++mt) {
            uint32_t q[2];
            if (BITS == 4) { q[0] = (uint32_t)wreg[u][mt][0][j]; q[1] = 0u; }
            else { q[0] = (uint32_t)wreg[u][mt][(2 * j) >> 2][(2 * j) & 3]; q[1] = (uint32_t)wreg[u][mt][(2 * j + 1) >> 2][(2 * j + 1) & 3]; }
            wf[mt] = wq_expand<T, BITS>(q, sc[mt], nz[mt]);
          }
          const int ch = ((4 * g + j) ^ r) << 4;
#pragma unroll
          for (int nt = 0; nt < MT16; ++nt) {
            const V8 xf = *reinterpret_cast<const V8*>(base + nt * 4096 + ch);
#pragma unroll
            for (int mt = 0; mt < 2; ++mt) acc[mt][nt] = mfma16(wf[mt], xf, acc[mt][nt]);
          }
        }
        }
      }
      wload(u, kt + DW);
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(YOUNGER) : "memory");
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                  // nothing in flight into registers or LDS

  // ---- epilogue: lane holds out[token 16 (wm MT16 + nt) + r][n0 + 16 mt + 4 g + i] ------------------------
  float* wsp = a.splits > 1 ? a.ws + (long)blockIdx.y * a.M * a.N : nullptr;
#pragma unroll
  for (int nt = 0; nt < MT16; ++nt) {
    const int tok = 16 * (wm * MT16 + nt) + r;
    if (tok >= a.M) continue;
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
      const int n = n0 + 16 * mt + 4 * g;
      if (n >= a.N) continue;
      if (wsp) {
        float* op = wsp + (long)tok * a.N + n;
        if (n + 3 < a.N) *reinterpret_cast<f32x4*>(op) = acc[mt][nt];
        else
          for (int i = 0; i < 4; ++i) if (n + i < a.N) op[i] = acc[mt][nt][i];
      } else {
        T* op = reinterpret_cast<T*>(a.out) + (long)tok * a.out_stride;
        V4 o;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float v = acc[mt][nt][i];
          if (a.bias && n + i < a.N) v += (float)reinterpret_cast<const T*>(a.bias)[n + i];
          o[i] = (T)v;
        }
        if (n + 3 < a.N && a.out_stride % 4 == 0) *reinterpret_cast<V4*>(op + n) = o;
        else
          for (int i = 0; i < 4; ++i) if (n + i < a.N) op[n + i] = o[i];
      }
    }
  }
}

// ---- many rows: one wave a SIMD, all operands through LDS ---------------------------------------------------
// A workgroup of four waves has 256 weight rows and 32 NT activation rows; wave w widens the weights of its 64 rows, once for all
// activation rows, and holds 64 x 32 NT sums (up to 256 accumulation registers, so one wave a SIMD).  A K unit is 64 elements: four
// products of 16, of which lane (r, h) has elements 32 h + 8 j .. + 7 of row r, as the packed words and a row's pieces of 16 bytes have them.
//   Copies to LDS run DX - 1 units ahead for activations, DW - 1 for weights, one behind each fragment's products; a unit's last third begins with
//   the wait for the next one and the only barrier, from which on fragments of the next unit are read, four ahead.
//   The widening of product j + 1 (some 3 instructions an element) is cut into 16 slices, spread evenly over the MFMAs of product j: a wave issues an
//   instruction in 4 cycles, an MFMA of 32x32x16 takes 32, and what lies between two of them beyond 7 instructions leaves the matrix pipe idle.
// LDS images: activations [row][8 pieces of 16 B], piece p of row t at p ^ ((t >> 1) & 7); weights [row][2 or 4 pieces], piece p of row t at p ^ ((t >> 3) & 1)
// (4 bits) or p ^ ((t >> 2) & 3): the 16 lanes that a read serves together (rows 0-3, 12-15, 20-27 or the others) touch all banks.
//
// us, before (tiles of 256 x 32 XT, two groups of waves that took turns at widening and products, of 64 x 16 XT sums a wave and two barriers per 32
// elements; weights were widened twice) / now, groups of 128: 4 bits, 160, 256 and 512 rows, 57344 x 8192 305 / 155, 312 / 218, 610 / 430;
// 8192 x 28672 151 / 87, 159 / 117, 290 / 207; 10240 x 8192 71 / 45, 78 / 61, 129 / 93; 6144 x 4096 39 / 31, 44 / 37, 59 / 46; 8 bits, 57344 x 8192 286 / 173, 292 / 237, 558 / 449;
// 8192 x 28672 147 / 88, 160 / 127, 272 / 216.  512 x 57344 x 8192 is 1.12 PFLOP/s, of 256 rows the matrix pipe works 69 % of the cycles, at 1.93 GHz: what bounds the large ones is
// power; of 64 rows 28 %: widening.
typedef int wq_buf_t __attribute__((ext_vector_type(4)));
constexpr unsigned WQ_RECORDS = 0xffffffc0u, WQ_NOWHERE = 0xfffffff0u;      // a copy from past the records brings zeros
// 16 or 4 bytes a lane to LDS, at dst + AT + 16 (4) * lane.  Statements of their own: told of the copies, the compiler would wait for them before
// every LDS read.
template <int AT> __device__ __forceinline__ void wq_copy16(wq_buf_t buf, unsigned voff, unsigned soff, unsigned dst) {
  asm volatile("s_add_u32 m0, %0, %4\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               ::"s"(dst), "v"(voff), "s"(buf), "s"(soff), "n"(AT) : "memory", "m0", "scc");
}
template <int AT> __device__ __forceinline__ void wq_copy4(wq_buf_t buf, unsigned voff, unsigned soff, unsigned dst) {
  asm volatile("s_add_u32 m0, %0, %4\n\ts_nop 0\n\tbuffer_load_dword %1, %2, %3 offen lds"
               ::"s"(dst), "v"(voff), "s"(buf), "s"(soff), "n"(AT) : "memory", "m0", "scc");
}
// the group of 32 elements number k32 (magic: 2^32 over a group's number of those, rounded up; 0: one)
__device__ __forceinline__ unsigned wq_group_of(unsigned k32, unsigned magic) { return magic ? __umulhi(k32, magic) : k32; }
__device__ __forceinline__ wq_buf_t wq_buffer(const void* p) {
  const uint64_t at = reinterpret_cast<uint64_t>(p);
  return wq_buf_t{__builtin_amdgcn_readfirstlane((int)at), __builtin_amdgcn_readfirstlane((int)(at >> 32) & 0xffff), (int)WQ_RECORDS, 0x00027000};
}
template <typename V8> __device__ __forceinline__ f32x16 wq_mfma32(V8 a, V8 b, f32x16 c) {
  if constexpr (std::is_same<V8, bf16x8>::value) return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  else return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

template <int LO, int HI, typename F> __device__ __forceinline__ void wq_each(F&& fn) {
  if constexpr (LO < HI) {
    fn(std::integral_constant<int, LO>{});
    wq_each<LO + 1, HI>(fn);
  }
}
template <int BITS, int NT> struct WqTile {
  static constexpr int XB = 32 * NT * 128;             // a unit's activations
  static constexpr int ROWB = 8 * BITS, WB = 256 * ROWB, SB = 2 * 1024, PB = WB + SB;   // weights, (scale, zero) pairs of both halves
  static constexpr int DX = NT > 5 ? 3 : 4;            // ring slots
  static constexpr int ROOM = (160 * 1024 - DX * XB) / PB;
  static constexpr int DW = ROOM < 8 ? ROOM : 8;
  static constexpr int LX = NT, LW = 2 * (BITS / 4) + 2;                                // copies of a wave and unit
  static constexpr int YOUNGER = (DX - 3) * (LX + LW) + (DW > DX ? LW : 0);
  static_assert(DW >= DX && YOUNGER < 64, "");
};

template <typename T, int BITS, int NT>
__global__ __launch_bounds__(256, 1) void wq_tile_kernel(const WqGemmArgs wa) {
  using V8 = typename Vec<T>::v8;
  using V4 = typename Vec<T>::v4;
  using C = WqTile<BITS, NT>;
  const DenseGemmArgs& a = wa.d;
  constexpr int XR = 32 * NT, NQ = BITS / 4, DX = C::DX, DW = C::DW, AHEAD = 4, FLAT = 4 * NT;
  constexpr int COPIES = C::LX + C::LW, EACH = NT < 4 ? 2 : 1;      // copies behind a fragment's products
  constexpr int LATEST = FLAT - (COPIES + EACH - 1) / EACH, MEET = 3 * NT - 2 < LATEST ? 3 * NT - 2 : LATEST;
  static_assert(MEET >= 4, "");
  __shared__ __attribute__((aligned(16))) uint8_t lds[DX * C::XB + DW * C::PB];

  // workgroup -> tile: each XCD (blockIdx.x % 8) takes a contiguous run of tiles, the row tiles of one weight tile next to each other
  const int tiles = a.m_tiles * a.n_tiles, per = (tiles * a.splits + 7) >> 3;
  const int t = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || t >= tiles * a.splits) return;
  const int sp = t / tiles, mi = t % tiles % a.m_tiles, ni = t % tiles / a.m_tiles;
  const int nu_all = (a.K + 63) >> 6;
  const int u0 = sp * a.units_per_split;
  const int nun = min(a.units_per_split, nu_all - u0);
  if (nun <= 0) return;
  const int beg = mi * XR, cnt = min(a.M - beg, XR), n0 = ni * 256;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 31, h = lane >> 5;
  const int turn = a.splits == 1 ? (int)((unsigned)ni * 5u % (unsigned)nun) : 0;
  auto unit_at = [&](int u) {
    const int v = min(u, nun - 1) + turn;
    return u0 + (v < nun ? v : v - nun);
  };

  // ---- copies: the wave's own 64 weight rows and their pairs, eight activation rows of every 32 ----
  const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lds;
  const wq_buf_t xbuf = wq_buffer(reinterpret_cast<const uint8_t*>(a.x) + (long)beg * a.x_stride * 2);
  const wq_buf_t wbuf = wq_buffer(reinterpret_cast<const uint8_t*>(a.w) + (long)n0 * ((long)a.K * BITS / 8));
  const wq_buf_t sbuf = wq_buffer(wa.sz);
  unsigned voff_x[NT], voff_w[C::LW - 2], voff_s;
  bool late_w[C::LW - 2];                              // a piece of a unit's second half
  const int xchunk = (lane & 7) ^ ((lane >> 4) | (wave & 1) << 2);           // rows 32 i + 8 wave + lane / 8: (row >> 1) & 7
#pragma unroll
  for (int i = 0; i < NT; ++i) {
    const int row = min(32 * i + 8 * wave + (lane >> 3), cnt - 1);
    voff_x[i] = (unsigned)row * (unsigned)(a.x_stride * 2) + (xchunk << 4);
  }
#pragma unroll
  for (int i = 0; i < C::LW - 2; ++i) {
    // 4 bits: 32 rows a copy, two pieces of 16 bytes; 8 bits: 16 rows, four
    const int row = BITS == 4 ? 32 * i + (lane >> 1) : 16 * i + (lane >> 2);
    const int piece = BITS == 4 ? (lane & 1) ^ ((row >> 3) & 1) : (lane & 3) ^ ((row >> 2) & 3);
    voff_w[i] = (unsigned)min(64 * wave + row, a.N - 1 - n0) * (unsigned)(a.K * BITS / 8) + (piece << 4);
    late_w[i] = piece >= BITS / 4;
  }
  voff_s = (unsigned)min(n0 + 64 * wave + lane, a.N - 1) * 4u;
  // a batch: the activations of unit ux, the weights of unit uw, behind each other in the rings
  unsigned xdst = lds0 + wave * 1024, wdst = lds0 + DX * C::XB + wave * (64 * C::ROWB), sdst = lds0 + DX * C::XB + C::WB + wave * 256;
  const unsigned plane = (unsigned)a.N * 4u;
  unsigned xoff = 0, woff = 0, soff[2] = {0, 0};
  bool xhalf = false, whalf = false;                   // a unit of 32 elements, at the end of K
  // (in four stages, for the loop; the values of the last batch are in use until stage 3)
  int kx = 0, kw = 0;
  unsigned group0 = 0, group1 = 0;
  auto batch = [&](int ux, int uw, int stage) {
    if (stage == 0) {
      kx = unit_at(ux) << 6;
    } else if (stage == 1) {
      kw = unit_at(uw) << 6;
    } else if (stage == 2) {
      group0 = wq_group_of((unsigned)(kw >> 5), wa.group_magic) * plane;
      group1 = kw + 32 >= a.K ? group0 : wq_group_of((unsigned)(kw >> 5) + 1, wa.group_magic) * plane;
    } else {
      xoff = (unsigned)kx * 2;
      xhalf = kx + 32 >= a.K;
      woff = (unsigned)kw * BITS / 8;
      whalf = kw + 32 >= a.K;
      soff[0] = group0;
      soff[1] = group1;
    }
  };
  // copy i of a batch (i a constant): activations, weights, pairs
  auto copy = [&](auto i_) {
    constexpr int i = decltype(i_)::value;
    if constexpr (i < NT) {
      wq_copy16<i * 4096>(xbuf, xhalf && xchunk >= 4 ? WQ_NOWHERE : voff_x[i], xoff, xdst);
      if constexpr (i == NT - 1) xdst = xdst + C::XB == lds0 + wave * 1024 + DX * C::XB ? lds0 + wave * 1024 : xdst + C::XB;
    } else if constexpr (i < NT + C::LW - 2) {
      wq_copy16<(i - NT) * 1024>(wbuf, whalf && late_w[i - NT] ? WQ_NOWHERE : voff_w[i - NT], woff, wdst);
    } else if constexpr (i < COPIES) {
      constexpr int p = i - (COPIES - 2);
      wq_copy4<p * 1024>(sbuf, voff_s, soff[p], sdst);
      if constexpr (p == 1) {
        const bool last = sdst + C::PB == lds0 + DX * C::XB + C::WB + wave * 256 + DW * C::PB;
        wdst = last ? wdst - (DW - 1) * C::PB : wdst + C::PB;
        sdst = last ? sdst - (DW - 1) * C::PB : sdst + C::PB;
      }
    }
  };

  // ---- operands: lane (r, h) has elements 32 h .. 32 h + 31 of a unit, eight to each of its four products of 16 ----
  const int x_rd = r * 128, x_sw = (r >> 1) & 7;
  int xr = 0, wr = 0;                                  // slots that are read
  i32x4 wq[2][NQ], wn[2][NQ];
  uint32_t pr[2];
  auto read_w = [&] {
    const uint8_t* base = lds + DX * C::XB + wr * C::PB;
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
      const uint8_t* p = base + wave * (64 * C::ROWB) + (32 * mt + r) * C::ROWB;
#pragma unroll
      for (int q = 0; q < NQ; ++q)
        wn[mt][q] = *reinterpret_cast<const i32x4*>(p + ((BITS == 4 ? h ^ ((r >> 3) & 1) : (2 * h + q) ^ ((r >> 2) & 3)) << 4));
      pr[mt] = *reinterpret_cast<const uint32_t*>(base + C::WB + h * 1024 + wave * 256 + (32 * mt + r) * 4);
    }
    wr = wr + 1 == DW ? 0 : wr + 1;
  };
  V8 xf[AHEAD];
  u32x4 wf[2][2];                                      // [which of two products][row tile]
  float sc[2], nz[2];
  auto take_w = [&] {
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
#pragma unroll
      for (int q = 0; q < NQ; ++q) wq[mt][q] = wn[mt][q];
      const V4 pv = __builtin_bit_cast(V4, u32x2{pr[mt], 0u});
      sc[mt] = (float)pv[0];
      nz[mt] = -(float)pv[1] * sc[mt];
    }
  };
  // Widening in 16 slices: slice 2 k spreads the words that elements 2 i and 2 i + 1 (i = k & 3) of product j's operand of row tile k >> 2 are
  // in, slice 2 k + 1 scales and packs them.
  uint32_t nib[2];
  float raw[2];
  auto widen = [&](int j, int slice) {
    typedef T T2 __attribute__((ext_vector_type(2)));
    const int mt = slice >> 3, i = (slice >> 1) & 3;
    if ((slice & 1) == 0) {
      if constexpr (BITS == 4) {
        if (i == 0) {                                  // (kept apart: bytes convert in one instruction, nibbles in two)
          nib[0] = (uint32_t)wq[mt][0][j] & 0x0F0F0F0Fu;
          nib[1] = ((uint32_t)wq[mt][0][j] >> 4) & 0x0F0F0F0Fu;
          asm volatile("" : "+v"(nib[0]), "+v"(nib[1]));
        }
        const uint32_t m = nib[i & 1];
        raw[0] = (float)(i < 2 ? m & 0xff : (m >> 8) & 0xff);
        raw[1] = (float)(i < 2 ? (m >> 16) & 0xff : m >> 24);
      } else {
        const uint32_t q = (uint32_t)wq[mt][j >> 1][2 * (j & 1) + (i >> 1)];
        raw[0] = (float)(i & 1 ? (q >> 16) & 0xff : q & 0xff);
        raw[1] = (float)(i & 1 ? q >> 24 : (q >> 8) & 0xff);
      }
      asm volatile("" : "+v"(raw[0]), "+v"(raw[1]));
    } else {
      const T2 o = {(T)fmaf(raw[0], sc[mt], nz[mt]), (T)fmaf(raw[1], sc[mt], nz[mt])};
      wf[j & 1][mt][i] = __builtin_bit_cast(uint32_t, o);
    }
  };
  // fragment f of the unit in slot `slot`: product f / NT, rows 32 (f % NT) ..
  auto read_x = [&](int f, int slot) {
    xf[f % AHEAD] = *reinterpret_cast<const V8*>(lds + slot * C::XB + x_rd + f % NT * 4096 + (((4 * h + f / NT) ^ x_sw) << 4));
  };

  f32x16 acc[2][NT];
#pragma unroll
  for (int mt = 0; mt < 2; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[mt][nt][i] = 0.f;

  for (int v = 1 - DW; v < 0; ++v) {
    if (v == -1) {
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(C::YOUNGER) : "memory");
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
    }
    for (int stage = 0; stage < 4; ++stage) batch(max(v + DX - 1, 0), v + DW - 1, stage);
    if (v + DX - 1 >= 0) wq_each<0, NT>(copy);
    wq_each<NT, COPIES>(copy);
  }
  read_w();
#pragma unroll
  for (int f = 0; f < AHEAD; ++f) read_x(f, 0);
  take_w();
#pragma unroll
  for (int k = 0; k < 16; ++k) widen(0, k);

  for (int u = 0; u < nun; ++u) {
    const int next = xr + 1 == DX ? 0 : xr + 1;
    wq_each<0, FLAT>([&](auto f_) {
      constexpr int f = decltype(f_)::value, j = f / NT, nt = f % NT;
      if (f == MEET) {                                 // the next unit is there, for all waves
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(C::YOUNGER) : "memory");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        batch(u + DX - 1, u + DW - 1, 3);
        read_w();
      }
      wq_each<0, 2>([&](auto mt_) {
        constexpr int mt = decltype(mt_)::value, s = 2 * nt + mt;
        acc[mt][nt] = wq_mfma32(__builtin_bit_cast(V8, wf[j & 1][mt]), xf[f % AHEAD], acc[mt][nt]);
        if (mt == 1) {
          if (f + AHEAD < FLAT) read_x(f + AHEAD, xr);
          else read_x(f + AHEAD - FLAT, next);
        }
        // a share of the next product's widening behind each product, and a copy
#pragma unroll
        for (int k = s * 8 / NT; k < (s + 1) * 8 / NT; ++k) {
          if (j == 3 && k == 0) take_w();              // (this unit's words are widened)
          widen((j + 1) & 3, k);
        }
        if constexpr (f >= MEET && (EACH == 2 || mt == 0)) copy(std::integral_constant<int, EACH * (f - MEET) + (EACH == 2 ? mt : 0)>{});
        if constexpr (mt == 1 && f >= MEET - 4 && f < MEET - 1) batch(u + DX - 1, u + DW - 1, f - (MEET - 4));
        __builtin_amdgcn_sched_barrier(0);
      });
    });
    xr = next;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");     // nothing in flight into LDS

  // ---- out[token beg + 32 nt + r][n0 + 64 wave + 32 mt + 8 q + 4 h + i] = acc[mt][nt][4 q + i] ----
  const int nb = n0 + 64 * wave + 4 * h;
  V4 bias[2][4];
#pragma unroll
  for (int mt = 0; mt < 2; ++mt)
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int n = nb + 32 * mt + 8 * q + i;
        bias[mt][q][i] = a.splits == 1 && a.bias && n < a.N ? reinterpret_cast<const T*>(a.bias)[n] : (T)0.f;
      }
  const bool wide = a.out_stride % 4 == 0;
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int tok = 32 * nt + r;
    if (tok >= cnt) continue;
    // (in their places until here: read out of them all at once, the sums would not fit)
    asm volatile("" : "+a"(acc[0][nt]), "+a"(acc[1][nt]));
    float* wsp = a.ws + ((long)sp * a.M + beg + tok) * a.N;
    T* op = reinterpret_cast<T*>(a.out) + (long)(beg + tok) * a.out_stride;
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int n = nb + 32 * mt + 8 * q;
        if (n >= a.N) continue;
        f32x4 v;
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = acc[mt][nt][4 * q + i];
        if (a.splits > 1) {                            // (N is a multiple of 4)
          *reinterpret_cast<f32x4*>(wsp + n) = v;
        } else {
          V4 o;
#pragma unroll
          for (int i = 0; i < 4; ++i) o[i] = (T)(v[i] + (float)bias[mt][q][i]);
          if (wide && n + 3 < a.N) *reinterpret_cast<V4*>(op + n) = o;
          else
            for (int i = 0; i < 4; ++i) if (n + i < a.N) op[n + i] = o[i];
        }
      }
  }
}

// ---- decode, fewer weight rows than fill the chip: K over the waves of a workgroup --------------------------
// Up to 16 activation rows.  The kernel above splits K over workgroups there, and the sum of the parts is a launch of its own
// (5 us and a gap of 2, of 20 in all).  Here a workgroup owns 32 weight rows and its KS waves a slice of K each: nothing is shared until
// the waves' sums meet in LDS, so there is no barrier in the loop, and the activations, a few rows that the L2 holds, go
// straight to registers.  Operands, steps of 128 elements and the unscaled form (POST) are the ones above.  Behind a step's
// arithmetic its registers take the activations two steps ahead and the weights four ahead (plain loads, which the
// compiler counts: were they inline assembly, a build that has to spill would spill what has not arrived).
// Bound by the memory system's latency and by activations from the L2, of which a wave of 32 weight rows reads M / 8 (4 bits) bytes
// a byte of weights.  Twice the steps in flight, or eight waves, are slower.
constexpr int WQ_KS = 4;
// Up to how many activation rows (of 16) this kernel leads, by what the kernel above would launch.  A step of 128 elements takes a
// wave here 0.4 (one row) to 0.7 us (16), in 8 bits 0.55 to 0.9, and it walks a quarter of them; the kernel above cuts K into
// up to 32 parts for 5 us of a launch that sums them.  us, kernel above / this, weights cold, 1, 8 and 16 rows:
//   one workgroup a CU there: 4 bits 2048 x 4096 10.1 / 7.0, 10.2 / 8.4, 10.5 / 9.9; x 6144 10.6 / 8.8, 11.1 / 10.7, 11.4 / 12.8; x 8192 11.2 / 10.5,
//     11.7 / 12.8, 11.7 / 15.7; 8 bits x 4096 12.4 / 8.8, 12.7 / 10.3, 13.0 / 11.8; x 8192 13.8 / 13.8, 14.7 / 16.3, 15.2 / 19.1
//   more: 4 bits 8192 x 8192 18.9 / 15.5, 19.5 / 15.2, 19.8 / 17.9; x 14336 25.9 / 23.2, 26.7 / 24.8, (10 rows) 26.9 / 25.5; x 28672 38.9 / 40.5,
//     40.0 / 44.0; 4096 x 14336 19.9 / 18.8, 20.3 / 21.1; 8 bits 8192 x 28672 67 / 52, 70 / 57, (12 rows) 67 / 59; 4096 x 28672 45.7 / 43.9,
//     46.0 / 47.4; 3072 x 14336 25.7 / 22.1, 26.4 / 25.6, x 28672 38.1 / 40.5, 38.6 / 46.8
//   wide layers in 4 bits, by how many workgroups a CU has to take here: 10240 x 8192 22.1 / 21.5, 23.5 / 25.9, 24.3 / 31.2; 14336 x 8192 29.5 / 23.3,
//     30.3 / 27.0, 31.6 / 31.8; 28672 x 4096 25.5 / 23.9, 26.2 / 28.5, 27.6 / 34.5
//   scaled in registers (groups of 64), which costs both more arithmetic: 2048 x 8192 13.0 / 13.0, 13.3 / 13.2, 13.6 / 14.9; 8192 x 14336 30.7 / 24.7,
//     30.8 / 25.8; 8192 x 28672 48.5 / 44.3, 49.0 / 46.0; 4096 x 28672 33.3 / 38.7; 10240 x 8192 25.2 / 24.3, 25.9 / 25.2, 26.4 / 29.8; 14336 x 8192
//     36.1 / 26.0, 35.9 / 27.6, 36.8 / 31.0; 28672 x 8192 52.8 / 46.4, 52.1 / 50.0, 52.7 / 58.9
//   workgroups of 128 weight rows that fill the chip, nothing to sum: 57344 x 8192 4 bits 61.8 / 65.6, 8 bits 111 / 96 (one row), 107 / 107 (10)
static int wq_slices_rows(int N, int K, int bits, bool scaled) {
  const int nk = K >> 7, groups = (N + 127) / 128, wgs = groups * max(1, min(min((512 + groups - 1) / groups, nk / 8), 32));
  if (groups * 4 >= 512 * 3) return bits == 8 ? 4 : 0;
  if (wgs <= 256) {
    if (nk <= 32) return 16;
    if (bits == 4) return scaled ? (nk <= 48 ? 16 : nk <= 64 ? 10 : 0) : nk <= 48 ? 8 : nk <= 64 ? 2 : 0;
    return nk <= 40 ? 12 : nk <= 48 ? 10 : nk <= 64 && groups >= 24 ? 4 : 0;
  }
  if (bits == 8) {
    if (nk <= 64) return groups <= 128 || nk <= 32 ? 16 : 12;
    return groups >= 40 ? 12 : groups >= 32 ? (nk <= 160 ? 12 : 4) : nk <= 128 ? 10 : 0;
  }
  if (scaled) {
    if (groups > 128) return nk <= 32 ? 12 : 8;
    if (groups > 96) return nk <= 64 ? 16 : 10;
    if (groups > 64) return nk <= 32 ? 16 : nk <= 128 ? 8 : 1;
    return nk <= 64 ? 16 : nk <= 128 ? 10 : groups >= (nk <= 160 ? 32 : 48) ? 8 : 0;
  }
  if (groups > 128) return nk <= 32 ? 2 : nk <= 64 ? 1 : 0;
  if (groups > 96) return nk <= 32 ? 10 : nk <= 64 ? 16 : nk <= 128 ? 8 : 0;
  if (groups > 64) return nk <= 32 ? 8 : nk <= 64 ? 1 : 0;
  return nk <= 64 ? 16 : nk <= 128 ? (groups >= 40 ? 10 : 4) : nk <= 176 ? (groups >= 40 ? 4 : 0) : groups >= 48 ? 1 : 0;
}
static bool wq_unscaled(int N, int bits, int group) { return bits == 4 && group % 128 == 0 && N % 4 == 0; }
static bool wq_unscaled_or_8(int N, int bits, int group) { return bits == 8 || wq_unscaled(N, bits, group); }
static bool wq_slices_pay(int M, int N, int K, int bits, int group, bool no_split) {
  if (no_split && (N + 127) / 128 * 4 < 512 * 3) return M <= 16 && (K <= 8192 || M <= (bits == 4 ? 10 : 12));   // K in one part there
  return M <= wq_slices_rows(N, K, bits, !wq_unscaled(N, bits, group));
}
// (for the test of the rule, which runs on the host)
VDA_EXPORT int vda_wq_slices_pay(int M, int N, int K, int bits, int group, int no_split) { return wq_slices_pay(M, N, K, bits, group, no_split); }
template <typename T, int BITS, bool POST>
__global__ __launch_bounds__(64 * WQ_KS, 2) void wq_slices_kernel(const WqGemmArgs wa) {
  using V8 = typename Vec<T>::v8;
  using V4 = typename Vec<T>::v4;
  const DenseGemmArgs& a = wa.d;
  constexpr int KS = WQ_KS, DW = 4, XD = 2;
  constexpr int NQ = BITS / 4, STEPB = 16 * BITS;
  __shared__ f32x4 sums[KS][2][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int r = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * 32;
  const int nk_all = a.K >> 7;
  const int kt0 = (int)((long)nk_all * wave / KS), nk = (int)((long)nk_all * (wave + 1) / KS) - kt0;

  const uint8_t* wp[2];
  const uint8_t* sp[2];
#pragma unroll
  for (int mt = 0; mt < 2; ++mt) {
    const int row = min(n0 + 16 * mt + r, a.N - 1);
    wp[mt] = reinterpret_cast<const uint8_t*>(a.w) + (long)row * ((long)a.K * BITS / 8) + (long)kt0 * STEPB + g * (STEPB / 4);
    sp[mt] = reinterpret_cast<const uint8_t*>(wa.sz) + (POST ? (long)min(n0 + 16 * mt + 4 * g, a.N - 4) * 4 : (long)row * 4);
  }
  const uint8_t* xp = reinterpret_cast<const uint8_t*>(a.x) + (long)min(r, a.M - 1) * a.x_stride * 2 + (long)kt0 * 256 + g * 64;
  i32x4 wreg[DW][2][NQ], xreg[XD][4];
  using Pairs = typename std::conditional<POST, i32x4, uint32_t>::type;
  Pairs sreg[DW][2];
  const long plane = (long)a.N * 4;
  auto xload = [&](int u, int kt) {
    const i32x4* p = reinterpret_cast<const i32x4*>(xp + (long)min(kt, nk - 1) * 256);
#pragma unroll
    for (int j = 0; j < 4; ++j) xreg[u][j] = p[j];
  };
  auto wload = [&](int u, int kt) {
    const int kk = min(kt, nk - 1);
    const long so = (long)((((kt0 + kk) << 2) + g) >> wa.gshift) * plane;
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int q = 0; q < NQ; ++q) wreg[u][mt][q] = reinterpret_cast<const i32x4*>(wp[mt] + (long)kk * STEPB)[q];
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) sreg[u][mt] = *reinterpret_cast<const Pairs*>(sp[mt] + so);
  };

  f32x4 acc[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}}, part[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}}, xsum = {0, 0, 0, 0};
  V8 ones;
#pragma unroll
  for (int i = 0; i < 8; ++i) ones[i] = (T)1.f;
  if (nk > 0) {
    // in the loop's own order
#pragma unroll
    for (int u = 0; u < DW - XD; ++u) wload(u, u);
#pragma unroll
    for (int u = 0; u < XD; ++u) { xload(u, u); wload(DW - XD + u, DW - XD + u); }
    for (int kb = 0; kb < nk; kb += DW) {
#pragma unroll
      for (int u = 0; u < DW; ++u) {
        const int kt = kb + u;
        if (kt < nk) {
          float sc[2], nz[2];
          if constexpr (!POST) {
#pragma unroll
            for (int mt = 0; mt < 2; ++mt) {
              const V4 pv = __builtin_bit_cast(V4, u32x2{sreg[u][mt], 0u});
              sc[mt] = (float)pv[0];
              nz[mt] = -(float)pv[1] * sc[mt];
            }
          }
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const V8 xf = __builtin_bit_cast(V8, xreg[u % XD][j]);
            V8 wf[2];
#pragma unroll
            for (int mt = 0; mt < 2; ++mt) {
              if constexpr (POST) {
                const uint32_t w = (uint32_t)wreg[u][mt][0][j];
                const u32x4 d = {(w & 0x000F000Fu) | WqMagic<T>::OR, ((w >> 4) & 0x000F000Fu) | WqMagic<T>::OR,
                                 ((w >> 8) & 0x000F000Fu) | WqMagic<T>::OR, ((w >> 12) & 0x000F000Fu) | WqMagic<T>::OR};
                wf[mt] = __builtin_bit_cast(V8, d);
              } else {
                uint32_t q[2];
                if (BITS == 4) { q[0] = (uint32_t)wreg[u][mt][0][j]; q[1] = 0u; }
                else { q[0] = (uint32_t)wreg[u][mt][(2 * j) >> 2][(2 * j) & 3]; q[1] = (uint32_t)wreg[u][mt][(2 * j + 1) >> 2][(2 * j + 1) & 3]; }
                wf[mt] = wq_expand<T, BITS>(q, sc[mt], nz[mt]);
              }
            }
            if constexpr (POST) {
              part[0] = mfma16(wf[0], xf, part[0]);
              part[1] = mfma16(wf[1], xf, part[1]);
              xsum = mfma16(ones, xf, xsum);
            } else {
              acc[0] = mfma16(wf[0], xf, acc[0]);
              acc[1] = mfma16(wf[1], xf, acc[1]);
            }
          }
          if constexpr (POST) {
            const int here = (kt0 + kt) << 2;
            if ((here >> wa.gshift) != ((here + 4) >> wa.gshift) || kt + 1 == nk) {   // the group, or what this wave has of it, ends
#pragma unroll
              for (int mt = 0; mt < 2; ++mt) {
                const V8 pv = __builtin_bit_cast(V8, sreg[u][mt]);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                  const float s = (float)pv[2 * i], zb = (float)pv[2 * i + 1] + WqMagic<T>::BIAS;
                  acc[mt][i] = fmaf(s, fmaf(-zb, xsum[i], part[mt][i]), acc[mt][i]);
                  part[mt][i] = 0.f;
                }
              }
              xsum = f32x4{0, 0, 0, 0};
            }
          }
        }
        __builtin_amdgcn_sched_barrier(0);
        xload(u % XD, kt + XD);
        wload(u, kt + DW);
      }
    }
  }
  sums[wave][0][lane] = acc[0];
  sums[wave][1][lane] = acc[1];
  __syncthreads();
  if (threadIdx.x >= 128) return;
  // out[token r][n0 + 16 mt + 4 g + i]
  const int mt = threadIdx.x >> 6, n = n0 + 16 * mt + 4 * g;
  if (r >= a.M || n >= a.N) return;
  f32x4 v = sums[0][mt][lane];
#pragma unroll
  for (int w = 1; w < KS; ++w) v += sums[w][mt][lane];
  T* op = reinterpret_cast<T*>(a.out) + (long)r * a.out_stride;
  V4 o;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (a.bias && n + i < a.N) v[i] += (float)reinterpret_cast<const T*>(a.bias)[n + i];
    o[i] = (T)v[i];
  }
  if (n + 3 < a.N && a.out_stride % 4 == 0) *reinterpret_cast<V4*>(op + n) = o;
  else
    for (int i = 0; i < 4; ++i) if (n + i < a.N) op[n + i] = o[i];
}

template <typename T, int BITS>
static int launch_wq_slices(const WqGemmArgs& wa, hipStream_t st) {
  const DenseGemmArgs& a = wa.d;
  const dim3 grid((unsigned)((a.N + 31) / 32));
  if constexpr (BITS == 4) {
    if (!wa.per_element && wq_unscaled(a.N, 4, wa.group)) {
      hipLaunchKernelGGL((wq_slices_kernel<T, 4, true>), grid, dim3(64 * WQ_KS), 0, st, wa);
      return 0;
    }
  }
  hipLaunchKernelGGL((wq_slices_kernel<T, BITS, false>), grid, dim3(64 * WQ_KS), 0, st, wa);
  return 0;
}

template <typename T, int BITS>
static int launch_wq_stream(const WqGemmArgs& wa, hipStream_t st) {
  const DenseGemmArgs& a = wa.d;
  const dim3 grid((unsigned)((a.N + 127) / 128), (unsigned)a.splits);
  // unscaled operands need 4-bit weights, groups made of whole K steps and four whole output rows per lane
  const bool post = BITS == 4 && !wa.per_element && (wa.group % 128 == 0) && a.N % 4 == 0;
#define LAUNCH(MT16, WM)                                                                                              \
  do {                                                                                                                \
    if constexpr (BITS == 4) {                                                                                        \
      if (post) { hipLaunchKernelGGL((wq_stream_kernel<T, 4, MT16, WM, true>), grid, dim3(256 * WM), 0, st, wa); break; } \
    }                                                                                                                 \
    hipLaunchKernelGGL((wq_stream_kernel<T, BITS, MT16, WM, false>), grid, dim3(256 * WM), 0, st, wa);                \
  } while (0)
  if (a.M <= 16) LAUNCH(1, 1);
  else if (a.M <= 32) LAUNCH(2, 1);
  else if (a.M <= 64) LAUNCH(4, 1);
  else LAUNCH(4, 2);
#undef LAUNCH
  if (a.splits > 1) {
    const long quads = (long)a.M * (a.N >> 2);
    hipLaunchKernelGGL((dense_gemm_reduce_kernel<T, DG_PLAIN>), dim3((unsigned)((quads + 255) / 256)), dim3(256), 0, st, a);
  }
  return 0;
}

template <typename T, int BITS>
static int launch_wq_tile(const WqGemmArgs& wa, int nt, hipStream_t st) {
  const DenseGemmArgs& a = wa.d;
  const dim3 grid((unsigned)(((long)a.m_tiles * a.n_tiles * a.splits + 7) / 8 * 8));
  switch (nt) {
    case 1: case 2: hipLaunchKernelGGL((wq_tile_kernel<T, BITS, 2>), grid, dim3(256), 0, st, wa); break;
    case 3: hipLaunchKernelGGL((wq_tile_kernel<T, BITS, 3>), grid, dim3(256), 0, st, wa); break;
    case 4: hipLaunchKernelGGL((wq_tile_kernel<T, BITS, 4>), grid, dim3(256), 0, st, wa); break;
    case 5: hipLaunchKernelGGL((wq_tile_kernel<T, BITS, 5>), grid, dim3(256), 0, st, wa); break;
    case 6: hipLaunchKernelGGL((wq_tile_kernel<T, BITS, 6>), grid, dim3(256), 0, st, wa); break;
    case 7: hipLaunchKernelGGL((wq_tile_kernel<T, BITS, 7>), grid, dim3(256), 0, st, wa); break;
    default: hipLaunchKernelGGL((wq_tile_kernel<T, BITS, 8>), grid, dim3(256), 0, st, wa); break;
  }
  if (a.splits > 1) {
    const long quads = (long)a.M * (a.N >> 2);
    hipLaunchKernelGGL((dense_gemm_reduce_kernel<T, DG_PLAIN>), dim3((unsigned)((quads + 255) / 256)), dim3(256), 0, st, a);
  }
  return 0;
}

// Into how many parts the kernel of up to 128 rows cuts K, for N / 128 workgroups each, of which the chip holds 512 (256 beyond 64 rows).
// As many as one round holds: a few workgroups more make a second one.  us, weights cold, parts that just exceed a round -> those that fit:
// 13 rows of 10240 x 8192 21.9 -> 19.5, 64 rows 36.1 -> 31.5 (8 bits 50.3 -> 41.8); 64 of 28672 x 8192 72.6 -> 63.9; 65 rows of 10240 x 8192 63.4 ->
// 45.2, of 5120 x 13824 58.4 -> 40.0, of 14336 x 4096 47.8 -> 34.0, of 22016 x 4096 62.2 -> 53.9.  Where two parts fit and one already
// gives two thirds of the CUs a workgroup, one saves the launch that sums: 8 bits 28672 x 4096, 13 rows, two 36.0, one 31.0, x 8192 60.6 -> 53.0; 171 blocks,
// the fewest, 17, 32 and 64 rows, x 4096 36.4 -> 32.8, 38.6 -> 33.9, 47.1 -> 41.1, x 8192 62.7 -> 57.3, 65.9 -> 59.1, 78.0 -> 71.7; 4 bits
// 21.8 -> 20.5, 25600 x 5120 28.1 -> 25.0, but 64 rows 45.4 / 51.0 and 28672 x 8192, four rows, 34.8 / 36.9.  From 257 workgroups on one part leaves more idle
// than a second round costs: 304 of them, 13 rows, 44.5 with one, 39.8 with two.
static int wq_parts(int M, int N, int K, int bits) {
  const int groups = (N + 127) / 128, nk = K >> 7, slots = M <= 64 ? 512 : 256;
  if (groups * 4 >= slots * 3) return 1;
  if (M <= 64 && groups > 170 && groups <= 256 && (bits == 8 || (M <= 32 && nk <= 40))) return 1;
  const int parts = slots == 512 && groups > 256 ? 2 : slots / groups;
  return max(1, min(min(parts, nk / 8), 32));
}
// (for the test of the rule, which runs on the host)
VDA_EXPORT int vda_wq_parts(int M, int N, int K, int bits) { return wq_parts(M, N, K, bits); }

// From how many of up to 128 rows the tiled kernel leads.  us, kernel above / tiled:
//   8 bits, 17, 33, 64, 96 and 128 rows: 57344 x 8192 114 / 112, 131 / 112, 138 / 118, 207 / 133 (here the tiled kernel before, as at 128), 207 / 149;
//     8192 x 28672 69 / 54, 79 / 53, 83 / 58, 98 / 67, 103 / 77; 8192 x 8192 26 / 23, 33 / 25, 36 / 28, 40 / 31, 42 / 35; 5120 x 13824 35 / 26, 41 / 27, 45 / 29;
//     but of short rows 28672 x 4096 34 / 32, 40 / 35, 41 / 38, 6144 x 4096 15.4 / 15.9, 17.7 / 17.8, 21 / 21, 27 / 23
//   4 bits scaled in registers (groups of 64), 48, 64, 96: 57344 x 8192 106 / 100, 107 / 100, 214 / 117; 10240 x 8192 29 / 29, 30 / 31, 47 / 36; 28672 x 4096
//     37 / 36, 38 / 37, 56 / 44; 6144 x 4096 17 / 20, 18 / 22, 26 / 26
//   4 bits unscaled: the kernel above has exact operands, whose sums are nearer to the product than those of weights rounded to 16 bits
static bool wq_tiles_pay(int M, int N, int K, int bits, int group, bool no_split) {
  if (M <= 64) return bits == 8 && !no_split && M > (K >= 8192 ? 16 : 32);
  return !wq_unscaled(N, bits, group);
}

// Which kernel takes a product, and in how many parts of K.  ws_bytes: the most that the parts' fp32 sums may take (0: one part).
struct WqPlan {
  enum { SLICES, STREAM, TILES } kernel;
  int nt, m_tiles, n_tiles, splits, units_per_split;
};
// log2(group / 32) of a power of two, 30 of one group, else -1
static int wq_group_shift(int K, int group) {
  if (group == K) return 30;
  for (int sh = 0; sh < 16; ++sh)
    if (group == (32 << sh)) return sh;
  return -1;
}
// Returns 0, or a negative code for shapes that are not taken.
static int wq_plan(WqPlan& p, int M, int N, int K, int group, int bits, long out_stride, size_t ws_bytes, int splits, int variant) {
  if (M < 1 || N < 1 || K < 32 || K % 32 || group < 32 || group % 32 || K % group || (bits != 4 && bits != 8)) return -1;
  const bool can_stream = M <= 128 && K % 128 == 0 && wq_group_shift(K, group) >= 0;
  const bool streams = variant == 2 || variant == 3;
  if (streams && !can_stream) return -1;
  const bool no_split = N % 4 || out_stride % 4 || ws_bytes == 0;
  int units;
  p.nt = 0;
  if (streams || (variant == 0 && can_stream && !wq_tiles_pay(M, N, K, bits, group, no_split))) {
    const int groups = (N + 127) / 128, parts = wq_parts(M, N, K, bits);
    p.kernel = WqPlan::STREAM;
    p.m_tiles = 1;
    p.n_tiles = groups;
    units = K >> 7;
    // (layers that the kernel below takes in one part with a workgroup on most CUs lead there at any number of rows: 28672 x 4096 in 8 bits, 4, 8
    // and 13 rows, slices 31.9, 35.0 and 38.1 us, this 30.1, 30.6 and 31.2; with 172 of them, 22016 x 4096, slices 24.9, 26.9 and 29.3, this
    // 29.0, 29.4 and 29.9)
    const bool whole = parts == 1 && groups >= 224 && groups <= 256 && wq_unscaled_or_8(N, bits, group);
    if (variant == 0 && splits < 1 && !whole && wq_slices_pay(M, N, K, bits, group, no_split)) {
      p.kernel = WqPlan::SLICES;
      splits = 1;
    }
    if (splits < 1) splits = parts;
  } else {
    p.kernel = WqPlan::TILES;
    p.m_tiles = (M + 255) / 256;
    p.nt = ((M + p.m_tiles - 1) / p.m_tiles + 31) / 32;
    p.n_tiles = (N + 255) / 256;
    units = (K + 63) >> 6;
    if (splits < 1) {
      const long tiles = (long)p.m_tiles * p.n_tiles;
      const double unit = 0.4 + 0.16 * p.nt;
      double best = 1e30;
      for (int s = 1; s <= min(16, max(units / 4, 1)); ++s) {
        const double t = (double)((tiles * s + 255) / 256) * ((units + s - 1) / s * unit + 2) + (s > 1 ? 5 + s * (double)M * N * 8 / 4e6 : 0);
        if (t < best) { best = t; splits = s; }
      }
    }
  }
  splits = min(splits, units);
  if (no_split) splits = 1;
  while (splits > 1 && (size_t)splits * M * N * sizeof(float) > ws_bytes) --splits;
  p.units_per_split = (units + splits - 1) / splits;
  p.splits = (units + p.units_per_split - 1) / p.units_per_split;
  return 0;
}
// fp32 slabs of [M, N] that such a product wants as its workspace (0: none)
VDA_EXPORT int vda_wq_gemm_slabs(int M, int N, int K, int group, int bits, long out_stride, size_t ws_bytes, int splits, int variant) {
  WqPlan p;
  return wq_plan(p, M, N, K, group, bits, out_stride, ws_bytes, splits, variant) == 0 && p.splits > 1 ? p.splits : 0;
}

// x [M, K] 16-bit (row stride x_stride elements), qw packed [N, K] (bits 4 or 8), sz [K / group, N, 2] of x's type,
// out [M, N].  K % 32 == 0, group % 32 == 0 and K % group == 0, N % 4 == 0 for split K.  variant: 0 picks by shape,
// 1 the tiled kernel, 2 the streaming kernel (M <= 128, K % 128 == 0, group a power of two or K), 3 the streaming
// kernel in its per-element form.  ws: the sums of K's parts (vda_wq_gemm_slabs says how many, of the same sizes and ws_bytes).  Returns 0
// or a negative code for shapes it does not take.
VDA_EXPORT int vda_wq_gemm(void* out, const void* x, const void* qw, const void* sz, const void* bias, float* ws,
                           size_t ws_bytes, int M, int N, int K, int group, int bits, long x_stride, long out_stride,
                           int dtype, int splits, int variant, hipStream_t st) {
  if (M < 1) return M == 0 ? 0 : -1;
  if (N < 1 || K < 32 || K % 32 || group < 32 || group % 32 || K % group) return -1;
  if (bits != 4 && bits != 8) return -1;
  if (x_stride % 8 || (N % 4 && out_stride % 4)) return -1;
  if (dtype != VDA_BF16 && dtype != VDA_F16) return -3;
  if ((long)N * K * bits / 8 >= (1LL << 32) || (long)M * x_stride * 2 >= (1LL << 32)) return -2;
  WqGemmArgs wa;
  DenseGemmArgs& a = wa.d;
  a.out = out; a.x = x; a.w = qw; a.bias = bias; a.residual = nullptr; a.ws = ws;
  a.M = M; a.N = N; a.K = K; a.x_stride = x_stride; a.out_stride = out_stride; a.res_stride = 0;
  wa.sz = sz; wa.group = group;
  wa.gshift = wq_group_shift(K, group);
  wa.group_magic = group == 32 ? 0u : (unsigned)(((1ull << 32) + group / 32 - 1) / (group / 32));
  WqPlan plan;
  const int code = wq_plan(plan, M, N, K, group, bits, out_stride, ws_bytes, splits, variant);
  if (code) return code;
  if (plan.splits > 1 && !ws) return -1;
  wa.per_element = variant == 3;
  a.m_tiles = plan.m_tiles; a.n_tiles = plan.n_tiles; a.splits = plan.splits; a.units_per_split = plan.units_per_split;
  int rc;
#define BY_TYPE(LAUNCH, ...)                                                                                            \
  (dtype == VDA_BF16 ? (bits == 4 ? LAUNCH<bf16_t, 4>(__VA_ARGS__) : LAUNCH<bf16_t, 8>(__VA_ARGS__))                       \
                     : (bits == 4 ? LAUNCH<f16_t, 4>(__VA_ARGS__) : LAUNCH<f16_t, 8>(__VA_ARGS__)))
  if (plan.kernel == WqPlan::SLICES) rc = BY_TYPE(launch_wq_slices, wa, st);
  else if (plan.kernel == WqPlan::STREAM) rc = BY_TYPE(launch_wq_stream, wa, st);
  else rc = BY_TYPE(launch_wq_tile, wa, plan.nt, st);
#undef BY_TYPE
  if (rc) return rc;
  VDA_CHECK_LAUNCH();
  return 0;
}
