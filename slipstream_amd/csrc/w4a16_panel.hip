// W4A16 panel kernel (m > 64, g == 128): y = x @ dequant(W)^T at the sizes where the matrix
// cores, not the weight bytes, set the time (a prefill chunk's or a packed step's tokens).
//
// A workgroup of four waves, one per SIMD, multiplies a panel of 16 MT activation rows
// (MT = 8 to 16) with 64 NS weight rows; wave w owns 16 NS of them (NS = 4 16-row MFMA tiles,
// or two where m fits one panel and 256-row tiles would leave half the chip idle: 197 x
// 4096 x 28672 73.6 -> 66.4 us, 130 x 4096 x 28672 73.7 -> 54.0)
// against every activation row of the panel. Per 128-key stage (one quantisation group):
//   - every weight is unpacked and dequantised once per workgroup, straight into the MFMA
//     operand registers (19 VALU instructions per eight weights), and feeds MT MFMAs: at
//     MT = 16 1.2 VALU instructions per MFMA, which issue while the matrix core works;
//   - every activation fragment read from LDS feeds NS MFMAs (the wide kernel's two, with
//     eight waves reading, make its LDS reads as long as its MFMAs).
// Activations come into LDS by DMA in half stages of 64 keys, a ring of four: one being
// read, one landed (so that fragments are read ahead across the barrier), two on their
// way; at a stage's end, though, the compiler's waits for the scale and zero-point
// loads, which it cannot tell from the DMAs behind them, leave none on its way. One
// wave per SIMD has nothing to hide behind, so the order is written out: every MFMA is
// followed by an instruction or two of the next key step's dequantisation, at times a
// fragment read six tiles ahead, a DMA instruction or a weight load (weights two stages
// ahead), and the scheduler is held to that order.
//
// The weights are the MFMA's row operand, so a lane's accumulators are consecutive output
// columns; with tile row i of wave tile ns holding weight row 4 NS (i / 4) + 4 ns + i % 4 they
// are 4 NS consecutive ones, stored as they are (no pass through LDS).
//
// Measured: 2240 x 4096 x 28672 662 -> 444 us (794 -> 1184 TFLOP/s; the dense bf16 product
// through hipBLASLt 365 us on the same card, these MFMAs alone with no loads or
// dequantisation 346 us: the clock falls to 1.9-2.0 GHz under them), 2240 x 14336 x 4096
// 353 -> 290 us. What is left: dequantisation about 75 us of the 444, activation DMA 65,
// weight loads 30 (each taken out alone).
#include <utility>

#include "w4a16_common.h"

namespace ss {
namespace {

constexpr int kPanelTab = 4 * 2 * 64 * 8;  // LDS bytes of the four waves' scale tables (two stages each)

// Eight int4 weights (one word: keys 8j .. 8j + 7 of a row) -> T((q - z) s) in key order.
// A nibble OR-ed into the mantissa of fp16 1024 is 1024 + q, and an FMA reads either fp16
// half in place: (1024 + q) s - (1024 + z) s. For 16-bit scales the constant is exact in
// fp32 (zero points to 7167; finite for scales below 3e35), so the FMA gives (q - z) s,
// rounded once to T. Nineteen instructions a word (the
// byte converts of dequant_word take 23).
template <int HALF>
__device__ __forceinline__ void fma_half(uint32_t t, float s, float c, float& r) {
  if constexpr (HALF)
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(t), "v"(s), "v"(c));
  else
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[0,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(t), "v"(s), "v"(c));
}
template <typename T>
__device__ __forceinline__ u32x4 dequant_pairs(uint32_t w, uint32_t magic, float s, float c) {
  float lo[4], hi[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t t = ((w >> (4 * i)) & 0x000F000Fu) | magic;
    fma_half<0>(t, s, c, lo[i]);
    fma_half<1>(t, s, c, hi[i]);
  }
  return u32x4{Elem<T>::pack2(lo[0], lo[1]), Elem<T>::pack2(lo[2], lo[3]), Elem<T>::pack2(hi[0], hi[1]),
               Elem<T>::pack2(hi[2], hi[3])};
}

// acc += a b on the matrix core, the accumulator in AGPRs. Written as asm because the
// compiler moved half of the accumulators between register files in every stage. What it
// therefore does not look after: the operands come from LDS reads it does wait for and
// from VALU results many instructions old, an accumulator is touched once per key step,
// and between a stage's last product and anything that follows the loop (after it the
// compiler copies accumulators wherever it likes) stand the barrier and the rotation of the
// stages' registers: over twenty instructions, where eleven cycles are needed. (An s_nop of
// that length in every stage took 2 % of the time.) tests/test_panel_code.py counts them in
// the compiled code.
template <typename T>
__device__ __forceinline__ void mfma_acc(f32x4& acc, u32x4 a, u32x4 b) {
  if constexpr (sizeof(T) == 2 && __is_same(T, bf16_t))
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
  else
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}
// Position of 16-byte chunk c of row r within the row's 128 LDS bytes: c ^ panel_swizzle(r).
// A 16-byte LDS read runs in four passes of sixteen lanes, lanes 0-3, 12-15, 20-27 first,
// then 4-11, 16-19, 28-31, and the same of the upper half: a pass takes rows 0-3 and 12-15
// of one key group and rows 4-11 of the next (whose chunk differs by 2). Rows 2p and 2p + 1
// lie in different halves of the 64 banks; this value keeps the row pairs of a pass apart
// (with p itself every pass hits each bank twice).
__device__ __forceinline__ int panel_swizzle(int r) {
  const int p = r >> 1;
  return (((p >> 2) ^ (p >> 1)) & 1) << 2 | ((p >> 2) & 1) << 1 | (p & 1);
}

// f(integral constant 0), ..., f(integral constant N - 1)
template <typename F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

template <typename T, int MT, int NS>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void w4a16_panel_kernel(
    const W4Params p, float* __restrict__ part, int kchunk, int ks, int n_tiles, int m_blocks) {
  constexpr int WR = 16 * NS;  // weight rows of a wave
  constexpr int BM = 16 * MT;
  constexpr int XBYTES = BM * 128;  // one half stage of activations (64 keys)
  constexpr int XI = MT / 2;        // DMA instructions per wave and half stage (eight rows each)
  static_assert(MT % 2 == 0, "whole DMA instructions per wave");
  extern __shared__ __attribute__((aligned(16))) char s_dyn[];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ln = lane & 15, kg = lane >> 4;
  // workgroup -> (K range, weight tile, activation block): each XCD (workgroups go round
  // robin over the eight) takes a contiguous eighth of the list, in which the activation
  // blocks of a (range, weight tile) pair follow each other, so that its L2 serves their
  // weights and no XCD has more than its share (whole pairs per XCD: 2158 x 2560 x 4864,
  // 19 pairs of 12 blocks, put 36 workgroups on three of them and took two rounds, 104 us)
  const int total = ks * n_tiles * m_blocks, per_xcd = (total + 7) >> 3;
  const int item = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if (item >= total) return;
  const int pair = item / m_blocks;
  const int zr = pair % ks;
  const int nb = (pair / ks) * 4 * WR + wave * WR;  // this wave's weight rows
  const int m0 = (item - pair * m_blocks) * BM;
  const int rows = min(BM, p.m - m0);
  const int i0 = zr * kchunk;
  const int i1 = min(p.k >> 7, i0 + kchunk);
  float2* const s_tab = reinterpret_cast<float2*>(s_dyn + 4 * XBYTES) + wave * 2 * WR;  // [stage % 2][WR rows]

  // ---- weights: tile ns is 4 ns rows further on; rows past N read zeros (out of the
  // descriptor's range, no memory access) and are never stored. Half h of a stage: keys
  // 64 h + 16 kg .. + 15 of the lane's row, its key steps' words 0 and 1.
  const __amdgpu_buffer_rsrc_t rw = buffer_rsrc(p.qw, (uint32_t)((int64_t)p.n * p.k / 2));
  const int w_row = p.k / 2;  // bytes
  const int w_off = (nb + (ln >> 2) * 4 * NS + (ln & 3)) * w_row + 8 * kg;
  typedef u32x2 Words[NS][2];
  auto load_w1 = [&](int i, int ns, int h, Words& w) {
    w[ns][h] = __builtin_bit_cast(
        u32x2, __builtin_amdgcn_raw_buffer_load_b64(rw, w_off, i * 64 + h * 32 + ns * 4 * w_row, 0));
  };
  auto load_w = [&](int i, Words& w) {
#pragma unroll
    for (int ns = 0; ns < NS; ++ns)
#pragma unroll
      for (int h = 0; h < 2; ++h) load_w1(i, ns, h, w);
  };

  // ---- scale and zero point of the wave's rows at one stage, one row per lane, turned
  // around through the wave's own table
  const int esize = p.sdt == SS_DTYPE_F32 ? 4 : 2;
  const __amdgpu_buffer_rsrc_t rsc = scale_rsrc(p, esize);
  const __amdgpu_buffer_rsrc_t rzp = buffer_rsrc(p.qz, (uint32_t)((int64_t)p.n * p.groups * 4));
  const int g_row = min(nb + lane % WR, p.n - 1) * p.groups;
  const uint32_t f16_mask = p.sdt == SS_DTYPE_F16 ? ~0u : 0u, bf16_mask = p.sdt == SS_DTYPE_BF16 ? ~0u : 0u;
  auto load_sz = [&](int i, uint32_t& sb, int& zb) {
    sb = scale_bits(rsc, g_row + i, esize);
    zb = __builtin_amdgcn_raw_buffer_load_b32(rzp, (g_row + i) * 4, 0, 0);
  };
  float sc[NS], cz[NS], scn[NS], czn[NS];  // this stage's scales and - s (1024 + z), and the next's
  auto turn_sz = [&](int i, uint32_t sb, int zb) {
    const float s = decode_scale_masked(sb, f16_mask, bf16_mask);
    s_tab[(i & 1) * WR + lane % WR] = float2{s, -s * (1024.f + (float)zb)};
#pragma unroll
    for (int ns = 0; ns < NS; ++ns) {
      const float2 t = s_tab[(i & 1) * WR + (ln >> 2) * 4 * NS + ns * 4 + (ln & 3)];
      scn[ns] = t.x;
      czn[ns] = t.y;
    }
  };

  // ---- activations: DMA instruction u of wave w brings rows 8 (4 u + w) + l / 8 of the
  // half stage; rows past M are out of the descriptor's range: zeros
  const i32x4w rx = wide_rsrc((const T*)p.x + (int64_t)m0 * p.x_stride,
                              (uint32_t)(((int64_t)(rows - 1) * p.x_stride + p.k) * sizeof(T)));
  const int x_tile = 32 * (int)p.x_stride * (int)sizeof(T);
  const int x_row = 8 * wave + (lane >> 3);
  const int x_off = x_row * (int)p.x_stride * (int)sizeof(T) + 16 * ((lane & 7) ^ panel_swizzle(x_row));
  const LdsW lds_x = (LdsW)s_dyn;
  const int hn = 2 * i1 - 1;  // the last half stage of the range
  int x_so = 0;  // scalar offset of the next DMA instruction
  auto dma_begin = [&](int h) {  // half stage h (past the range: the last one again, never read)
    x_so = __builtin_amdgcn_readfirstlane(min(h, hn) * 128);
    asm volatile("s_nop 4" : : "s"(x_so));  // a VALU-written SGPR: five wait states before a VMEM reads it
  };
  auto dma_next = [&](int h, int u) {
    asm_dma_b128(rx, lds_x + (h & 3) * XBYTES + u * 4096 + wave * 1024, x_off, x_so);
    asm volatile("s_add_i32 %0, %0, %1" : "+s"(x_so) : "s"(x_tile) : "scc");  // scalar-written: no wait states
  };
  auto dma_x = [&](int h) {
    dma_begin(h);
#pragma unroll
    for (int u = 0; u < XI; ++u) dma_next(h, u);
  };
  // fragment (tile mt, key step s of a half) of lane (ln, kg): row 16 mt + ln, chunk 2 kg + s
  const int a_off0 = ln * 128 + 16 * ((2 * kg) ^ panel_swizzle(ln)), a_off1 = ln * 128 + 16 * ((2 * kg + 1) ^ panel_swizzle(ln));

  f32x4 acc[MT][NS];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int ns = 0; ns < NS; ++ns) acc[mt][ns] = f32x4{0.f, 0.f, 0.f, 0.f};

  const uint32_t magic = in_vgpr(W4Elem<f16_t>::kMagicPair);
  u32x4 b[2][NS];  // operands of the key step in work and of the next
  Words w0, w1, w2;  // stages i, i + 1 and i + 2
  uint32_t sb1, sb2;
  int zb1, zb2;
  constexpr int LA = 6;  // fragment reads ahead of their MFMAs
  constexpr int AR = LA + 2;
  u32x4 a[AR];
  // prologue: three half stages and the first stage's weights landed, its first step dequantised
  asm volatile("s_nop 4");  // descriptor SGPRs written by VALU before the first asm load
  dma_x(2 * i0);
  dma_x(2 * i0 + 1);
  dma_x(2 * i0 + 2);
  load_sz(i0, sb1, zb1);
  load_w(i0, w0);
  turn_sz(i0, sb1, zb1);
  load_sz(min(i0 + 1, i1 - 1), sb1, zb1);
  load_w(min(i0 + 1, i1 - 1), w1);
#pragma unroll
  for (int ns = 0; ns < NS; ++ns) {
    sc[ns] = scn[ns];
    cz[ns] = czn[ns];
    b[0][ns] = dequant_pairs<T>(w0[ns][0][0], magic, sc[ns], cz[ns]);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  {
    const char* const xs = (const char*)s_dyn + ((2 * i0) & 3) * XBYTES;
#pragma unroll
    for (int t = 0; t < LA; ++t) a[t] = *reinterpret_cast<const u32x4*>(xs + t * 2048 + a_off0);
  }

  for (int i = i0; i < i1; ++i) {
    uint32_t v[4];
    float f[8];
    static_for<2>([&](auto hc) __attribute__((always_inline)) {
      constexpr int h = hc;
      const int in = min(i + 2, i1 - 1);
      const char* const xs = (const char*)s_dyn + ((2 * i + h) & 3) * XBYTES;
      const char* const xn = (const char*)s_dyn + ((2 * i + h + 1) & 3) * XBYTES;
      static_for<2 * MT>([&](auto tc) __attribute__((always_inline)) {
        constexpr int t = tc, s = t / MT, mt = t % MT, step = 2 * h + s;
        constexpr int tr = t + LA;  // the fragment to read now
        if constexpr (tr < 2 * MT)
          a[(tr + h * 2 * MT) % AR] = *reinterpret_cast<const u32x4*>(xs + (tr % MT) * 2048 + (tr < MT ? a_off0 : a_off1));
        else
          a[(tr + h * 2 * MT) % AR] = *reinterpret_cast<const u32x4*>(xn + (tr - 2 * MT) * 2048 + a_off0);
        // the memory instructions one at a time between the products: issued together they
        // wait for room in the address unit's queue, and the matrix core with them
        if constexpr (t == 0) dma_begin(2 * i + h + 3);
        if constexpr (t % 2 == 1 && t / 2 < XI) dma_next(2 * i + h + 3, t / 2);
        if constexpr (h == 0 && t % 2 == 0 && t / 2 < 2 * NS) load_w1(in, t / 4, t / 2 % 2, w2);
        if constexpr (h == 0 && t == 2 * MT - 1) load_sz(in, sb2, zb2);
        if constexpr (step == 2 && mt == MT - 2) turn_sz(i + 1, sb1, zb1);
        static_for<NS>([&](auto nc) __attribute__((always_inline)) {
          constexpr int ns = nc;
          mfma_acc<T>(acc[mt][ns], b[s][ns], a[(t + h * 2 * MT) % AR]);
          // beside the product an instruction or two of the next step's operands: nineteen
          // for each of the four weight tiles, an operand always a few instructions old
          constexpr int kOps = 19 * NS, kSlots = NS * MT, slot = mt * NS + ns;
          constexpr int o0 = slot * kOps / kSlots, o1 = (slot + 1) * kOps / kSlots;
          static_for<o1 - o0>([&](auto oc) __attribute__((always_inline)) {
            constexpr int q = (o0 + oc) / 19, r = (o0 + oc) % 19;
            const uint32_t word = step == 0 ? w0[q][0][1] : step == 1 ? w0[q][1][0] : step == 2 ? w0[q][1][1] : w1[q][0][0];
            if constexpr (r < 3)
              v[r + 1] = word >> (4 * (r + 1));
            else if constexpr (r < 7)
              v[r - 3] = ((r == 3 ? word : v[r - 3]) & 0x000F000Fu) | magic;
            else if constexpr (r < 15)
              fma_half<r & 1 ? 0 : 1>(v[(r - 7) / 2], step < 3 ? sc[q] : scn[q], step < 3 ? cz[q] : czn[q],
                                      f[(r & 1 ? 0 : 4) + (r - 7) / 2]);
            else
              b[s ^ 1][q][r - 15] = Elem<T>::pack2(f[2 * (r - 15)], f[2 * (r - 15) + 1]);
          });
          __builtin_amdgcn_sched_barrier(0);
        });
      });
      // half stage 2 i + h + 2 has landed (requested a half stage ago; newer: what this
      // half stage requested); after the barrier its buffer may be read and the
      // one of 2 i + h overwritten
      asm volatile("s_waitcnt vmcnt(%0)" : : "n"(XI + (h == 0 ? 2 * NS + 2 : 0)) : "memory");
      // the bare barrier: the fragments read ahead stay in flight (__syncthreads would wait
      // for them); every read of the buffer that is overwritten next has fed its MFMA
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
    });
#pragma unroll
    for (int ns = 0; ns < NS; ++ns) {
      sc[ns] = scn[ns];
      cz[ns] = czn[ns];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        w0[ns][h] = w1[ns][h];
        w1[ns][h] = w2[ns][h];
      }
    }
    sb1 = sb2;
    zb1 = zb2;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no DMA into LDS is left when the workgroup ends

  // ---- results: lane holds C[m0 + 16 mt + ln][nb + 4 NS kg + 4 ns + e]
  const int n = nb + 4 * NS * kg;
  if (n >= p.n) return;
  const bool whole = n + 4 * NS <= p.n;
  if (ks > 1) {
    const bool vec = whole && p.n % 4 == 0;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int m = m0 + 16 * mt + ln;
      if (m >= p.m) continue;
      float* const dst = part + ((int64_t)zr * p.m + m) * p.n + n;
#pragma unroll
      for (int ns = 0; ns < NS; ++ns) {
        if (vec) {
          *reinterpret_cast<f32x4*>(dst + 4 * ns) = acc[mt][ns];
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (n + 4 * ns + e < p.n) dst[4 * ns + e] = acc[mt][ns][e];
        }
      }
    }
    return;
  }
  const bool vec = whole && p.o_stride % 8 == 0 && ((uintptr_t)p.out & 15) == 0;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int m = m0 + 16 * mt + ln;
    if (m >= p.m) continue;
    T* const o = (T*)p.out + (int64_t)m * p.o_stride + n;
    if (vec) {
#pragma unroll
      for (int h = 0; h < NS / 2; ++h)
        store16(o + 8 * h, u32x4{Elem<T>::pack2(acc[mt][2 * h][0], acc[mt][2 * h][1]),
                                 Elem<T>::pack2(acc[mt][2 * h][2], acc[mt][2 * h][3]),
                                 Elem<T>::pack2(acc[mt][2 * h + 1][0], acc[mt][2 * h + 1][1]),
                                 Elem<T>::pack2(acc[mt][2 * h + 1][2], acc[mt][2 * h + 1][3])});
    } else {
#pragma unroll
      for (int ns = 0; ns < NS; ++ns)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + 4 * ns + e < p.n) o[4 * ns + e] = (T)acc[mt][ns][e];
    }
  }
}

size_t panel_lds_bytes(int mt) { return (size_t)4 * mt * 16 * 128 + kPanelTab; }

template <typename T, int MT, int NS>
int launch_panel(const W4Params& p, const PanelPlan& pl, float* part, hipStream_t stream) {
  auto kern = w4a16_panel_kernel<T, MT, NS>;
  static bool attr_set = false;
  const size_t lds = panel_lds_bytes(MT);
  if (!attr_set) {
    if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess) {
      ss_host::set_error("w4a16 gemm: cannot reserve %zu bytes of LDS", lds);
      return SS_ERR_UNSUPPORTED;
    }
    attr_set = true;
  }
  const int64_t grid = ((int64_t)pl.ks * pl.n_tiles * pl.m_blocks + 7) / 8 * 8;
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(256), lds, stream, p, part, pl.kchunk, pl.ks, pl.n_tiles,
                     pl.m_blocks);
  return ss_host::launch_status("w4a16 gemm (panel)");
}

template <typename T>
int launch_panel_typed(const W4Params& p, const PanelPlan& pl, float* part, hipStream_t stream) {
  if (pl.ns == 4) {
    switch (pl.mt) {
      case 8: return launch_panel<T, 8, 4>(p, pl, part, stream);
      case 10: return launch_panel<T, 10, 4>(p, pl, part, stream);
      case 12: return launch_panel<T, 12, 4>(p, pl, part, stream);
      case 14: return launch_panel<T, 14, 4>(p, pl, part, stream);
      case 16: return launch_panel<T, 16, 4>(p, pl, part, stream);
    }
  } else {
    switch (pl.mt) {
      case 8: return launch_panel<T, 8, 2>(p, pl, part, stream);
      case 10: return launch_panel<T, 10, 2>(p, pl, part, stream);
      case 12: return launch_panel<T, 12, 2>(p, pl, part, stream);
      case 14: return launch_panel<T, 14, 2>(p, pl, part, stream);
      case 16: return launch_panel<T, 16, 2>(p, pl, part, stream);
    }
  }
  ss_host::set_error("w4a16 gemm: panel of %d tiles", pl.mt);
  return SS_ERR_UNSUPPORTED;
}

}  // namespace

// The panel height and K split of least estimated time, and whether that beats a kernel
// of estimated time `other` (us). A workgroup takes 0.95 + 0.143 MT us a stage (MT = 8: 2.07
// us, 16: 3.25 us measured, one workgroup per CU), with two weight tiles a wave 1.0 + 0.068
// MT (MT = 10: 1.6, 16: 2.15), and about 4 us around its stages; a K split adds the partials'
// round trip (4 TB/s) and the reduce launch. The constant part is the dequantisation's and
// the loads' issue: one wave issues an instruction every five cycles or so.
bool plan_w4a16_panel(PanelPlan& pl, int64_t m, int64_t n, int64_t k, int g, double other) {
  if (m <= 64 || g != 128 || k % 128 || (n + 256) * (k / 2) >= ((int64_t)1 << 31)) return false;
  const int64_t stages = k / 128;
  const int64_t cus = ss_host::device_cu_count();
  double best = 0.93 * other;  // within the estimate's error the other kernel keeps the shape
  bool found = false;
  for (int shape = 0; shape < 10; ++shape) {
    const int ns = shape < 5 ? 4 : 2, mt = 8 + 2 * (shape % 5);
    const int64_t n_tiles = (n + 64 * ns - 1) / (64 * ns);
    const int64_t m_blocks = (m + 16 * mt - 1) / (16 * mt);
    for (int64_t ks = 1; ks <= 16; ++ks) {
      const int64_t per = (stages + ks - 1) / ks;
      if ((stages + per - 1) / per != ks || (ks > 1 && per < 8)) continue;
      const int64_t rounds = (n_tiles * m_blocks * ks + cus - 1) / cus;
      double t = (double)rounds * ((double)per * (ns == 4 ? 0.95 + 0.143 * mt : 1.0 + 0.068 * mt) + 4.0);
      if (ks > 1) t += (double)ks * (double)m * (double)n * 8e-6 / 4.0 + 4.0;
      if (t < best) {
        best = t;
        found = true;
        pl.mt = mt;
        pl.ns = ns;
        pl.ks = (int)ks;
        pl.kchunk = (int)per;
        pl.n_tiles = (int)n_tiles;
        pl.m_blocks = (int)m_blocks;
      }
    }
  }
  return found && (pl.ks == 1 || (int64_t)pl.ks * m * n * 4 < (int64_t)kOutOfRange) &&
         (int64_t)pl.ks * pl.n_tiles * pl.m_blocks <= 0x7ffffff0;
}

int launch_w4a16_panel(const W4Params& p, const PanelPlan& pl, int act_dtype, float* part, hipStream_t stream) {
  if (act_dtype == SS_DTYPE_BF16) return launch_panel_typed<bf16_t>(p, pl, part, stream);
  return launch_panel_typed<f16_t>(p, pl, part, stream);
}

}  // namespace ss
