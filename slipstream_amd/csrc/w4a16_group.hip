// W4A16 group kernel (m <= 64, groups of 32, 64 or 128 keys, any whole number of 128-key
// stages): small products, where the time is a few memory round trips. (Above 64 rows it
// runs only where the untiled kernel's scale table does not fit its LDS.)
//
// A workgroup owns 16 NS weight rows and 16 MT activation rows; its waves (up to sixteen)
// split K into contiguous runs of 128-key stages, and each wave requests the weights,
// scales, zero points and activations of P stages at once, straight into registers, before
// it uses any of them: for most calls of this size all of its run, so that the whole
// workgroup costs one memory round trip, one LDS pass that adds the waves' sums in wave
// order, and the store. There is no staging of activations (every fragment is read in MFMA
// layout; the rows are in the L2) and no scale table.
//
// An MFMA of 16x16x32 must stay inside one quantisation group for the fp32 fold
//     acc += s G - s (MAGIC + z) X,  G = sum x (MAGIC + q),  X = sum x,
// which groups of 64 keys take every 32 as smaller groups do: the MAGIC part that cancels
// carries the rounding of G and X, and grows with their length (fp16, folded per 64: 6.3 %
// of the results of 896 x 9728 not the nearest to the exact sum, per 32 5.5 %).
//
// A lane's 16-byte weight load is 32 consecutive keys of its row. The four lanes of a
// row hold four such runs, and a 4 x 4 exchange of their words (two v_permlane32_swap, two
// v_permlane16_swap) gives each lane the words of keys 32 s + 8 kg in step s.
//
// Scales and zero points: each lane loads every fourth group of its row's round and the
// wave turns them around through its own part of LDS; one load per group in every lane kept
// the address unit busy for as long as everything else (4864 x 896, m = 11, g = 64: 11.8
// us so, 9.8 us with the table). Rounds of fewer live stages than P ask for nothing (offsets
// past the buffers; repeating a live stage instead cost 8.9 -> 9.8 us).
//
// Measured (m = 11, g = 64, weights from HBM) against the untiled kernel's activation
// staging and scale tables: 896 x 9728 16.1 -> 5.8 us, 4864 x 896 25.8 -> 8.3 us. What is left
// are the launch, one round trip to HBM and the LDS pass (0.3-0.9 TB/s of weights).
#include "w4a16_common.h"

namespace ss {
namespace {

// Word j of lane row i (of four 16-lane rows) <-> word i of lane row j.
__device__ __forceinline__ u32x4 exchange_words(u32x4 w) {
  const auto a = __builtin_amdgcn_permlane32_swap(w[0], w[2], false, false);
  const auto b = __builtin_amdgcn_permlane32_swap(w[1], w[3], false, false);
  const auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
  const auto d = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
  return u32x4{c[0], c[1], d[0], d[1]};
}

// GS: 32-key MFMA steps per scale, all in one quantisation group (4: g % 128 == 0, 2: g ==
// 64, 1: any other g % 32 == 0); per: stages of a wave's run.
template <typename T, int MT, int NS, int GS, int P>
__global__ __launch_bounds__(1024) void w4a16_group_kernel(const W4Params p, int per) {
  typedef W4Elem<T> E;
  constexpr int NG = 4 / GS;   // groups of a stage
  constexpr int FS = GS == 4 ? 4 : 1;  // steps of a fold
  constexpr int NGR = P * NG;  // and of a round
  constexpr int EL = (NGR + 3) / 4;  // of those, a lane's
  extern __shared__ __attribute__((aligned(16))) char s_dyn[];
  f32x4* const s_red = (f32x4*)s_dyn;  // [wave][mt][ns][lane]; before that:

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ln = lane & 15, kg = lane >> 4;
  const int n0 = blockIdx.x * 16 * NS, m0 = blockIdx.y * 16 * MT;
  const int rows = min(16 * MT, p.m - m0);
  float2* const s_tab = (float2*)s_dyn + wave * (NGR * 16 * NS);  // the wave's round: [group][row] of (s, s (MAGIC + z))
  const int stages = p.k >> 7;
  const int i0 = wave * per, i1 = min(stages, i0 + per);

  const __amdgpu_buffer_rsrc_t rw = buffer_rsrc(p.qw, (uint32_t)((int64_t)p.n * p.k / 2));
  const int esize = p.sdt == SS_DTYPE_F32 ? 4 : 2;
  const __amdgpu_buffer_rsrc_t rsc = scale_rsrc(p, esize);
  const __amdgpu_buffer_rsrc_t rzp = buffer_rsrc(p.qz, (uint32_t)((int64_t)p.n * p.groups * 4));
  const uint32_t f16_mask = p.sdt == SS_DTYPE_F16 ? ~0u : 0u, bf16_mask = p.sdt == SS_DTYPE_BF16 ? ~0u : 0u;
  const __amdgpu_buffer_rsrc_t rx = buffer_rsrc(
      (const T*)p.x + (int64_t)m0 * p.x_stride, (uint32_t)(((int64_t)(rows - 1) * p.x_stride + p.k) * sizeof(T)));
  // rows past N repeat row N - 1 and rows past M row M - 1: never stored
  int w_off[NS], g_off[NS], x_off[MT];
#pragma unroll
  for (int ns = 0; ns < NS; ++ns) {
    const int r = min(n0 + 16 * ns + ln, p.n - 1);
    w_off[ns] = r * (p.k / 2) + 16 * kg;
    g_off[ns] = r * p.groups;
  }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
    x_off[mt] = (int)((int64_t)min(16 * mt + ln, rows - 1) * p.x_stride * (int64_t)sizeof(T)) + 16 * kg;

  // quantisation group of the e-th 32 GS keys
  auto group_at = [&](int e) { return GS == 2 ? e : (int)((uint32_t)(e * (32 * GS)) / (uint32_t)p.g); };
  const uint32_t magic = in_vgpr(E::kMagicPair);
  const u32x4 ones = {E::kOnePair, E::kOnePair, E::kOnePair, E::kOnePair};
  f32x4 acc[MT][NS];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int ns = 0; ns < NS; ++ns) acc[mt][ns] = f32x4{0.f, 0.f, 0.f, 0.f};

  for (int i = i0; i < i1; i += P) {
    // every load of the round before any use; stages past the run lie out of every
    // descriptor's range (zeros, no memory access) and fold with scale 0
    u32x4 w[P][NS], x[P][4][MT];
    uint32_t sb[NS][EL];
    int zb[NS][EL];
    const int gl = group_at(i1 * NG - 1);  // the run's last group
    // a lane takes every fourth of the round's groups of its row
#pragma unroll
    for (int ns = 0; ns < NS; ++ns)
#pragma unroll
      for (int j = 0; j < EL; ++j) {
        const int e = 4 * j + kg;
        const int gi = g_off[ns] + min(group_at(i * NG + e), gl);
        sb[ns][j] = scale_bits(rsc, gi, esize);
        zb[ns][j] = __builtin_amdgcn_raw_buffer_load_b32(rzp, gi * 4, 0, 0);
      }
#pragma unroll
    for (int u = 0; u < P; ++u) {
      const int st = i + u;
      const int wo = st < i1 ? st * 64 : kOutOfRange, xo = st < i1 ? st * 256 : kOutOfRange;
#pragma unroll
      for (int ns = 0; ns < NS; ++ns)
        w[u][ns] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rw, w_off[ns], wo, kNonTemporal));
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          x[u][s][mt] = __builtin_bit_cast(
              u32x4, __builtin_amdgcn_raw_buffer_load_b128(rx, x_off[mt] + 64 * s, xo, 0));
    }
    __builtin_amdgcn_sched_barrier(0);
    // the wave's own table: its LDS operations run in order, no barrier
#pragma unroll
    for (int ns = 0; ns < NS; ++ns)
#pragma unroll
      for (int j = 0; j < EL; ++j) {
        const float sc = decode_scale_masked(sb[ns][j], f16_mask, bf16_mask);
        if (NGR % 4 == 0 || 4 * j + kg < NGR)
          s_tab[(4 * j + kg) * 16 * NS + 16 * ns + ln] = float2{sc, sc * (E::kMagic + (float)zb[ns][j])};
      }
    asm volatile("" ::: "memory");
#pragma unroll
    for (int u = 0; u < P; ++u) {
      const bool live = i + u < i1;
#pragma unroll
      for (int ns = 0; ns < NS; ++ns) w[u][ns] = exchange_words(w[u][ns]);
      f32x4 G[MT][NS], X[MT];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        if (s % FS == 0) {
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) {
            X[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ns = 0; ns < NS; ++ns) G[mt][ns] = f32x4{0.f, 0.f, 0.f, 0.f};
          }
        }
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          x[u][s][mt] = permute_x(x[u][s][mt]);
          X[mt] = Elem<T>::mfma(x[u][s][mt], ones, X[mt]);
        }
#pragma unroll
        for (int ns = 0; ns < NS; ++ns) {
          const u32x4 b = nibbles_to_operand(w[u][ns][s], magic);
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) G[mt][ns] = Elem<T>::mfma(x[u][s][mt], b, G[mt][ns]);
        }
        if (s % FS == FS - 1) {
#pragma unroll
          for (int ns = 0; ns < NS; ++ns) {
            const float2 t = s_tab[(u * NG + s / GS) * 16 * NS + 16 * ns + ln];
            const float sc = live ? t.x : 0.f, cz = live ? t.y : 0.f;
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
              for (int e = 0; e < 4; ++e) acc[mt][ns][e] = fmaf(sc, G[mt][ns][e], fmaf(-cz, X[mt][e], acc[mt][ns][e]));
          }
        }
      }
    }
  }

  // ---- the waves' sums added in wave order, one output element per thread
  __syncthreads();  // the buffer overlays the tables
  const int waves = blockDim.x >> 6;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int ns = 0; ns < NS; ++ns) s_red[((wave * MT + mt) * NS + ns) * 64 + lane] = acc[mt][ns];
  __syncthreads();
  const float* const red = (const float*)s_dyn;
  constexpr int kOut = MT * NS * 256;
  for (int q = threadIdx.x; q < kOut; q += blockDim.x) {
    // element e of lane (ln, kg) of tile (mt, ns): row 16 mt + 4 kg + e, column 16 ns + ln;
    // consecutive threads take consecutive columns
    const int c = q % (16 * NS), r = q / (16 * NS);
    const int src = (((r >> 4) * NS + (c >> 4)) * 64 + ((r >> 2) & 3) * 16 + (c & 15)) * 4 + (r & 3);
    float y = 0.f;
#pragma unroll 4
    for (int w = 0; w < waves; ++w) y += red[w * kOut + src];
    if (m0 + r < p.m && n0 + c < p.n) ((T*)p.out)[(int64_t)(m0 + r) * p.o_stride + n0 + c] = (T)y;
  }
}

// Stages a wave requests at once: what 128 registers hold.
constexpr int group_round(int mt, int ns) { return mt == 1 ? (ns == 1 ? 4 : 2) : (mt == 2 && ns == 1 ? 2 : 1); }

template <typename T, int MT, int NS, int GS>
int launch_group(const W4Params& p, const GroupPlan& pl, hipStream_t stream) {
  constexpr int P = group_round(MT, NS);
  const size_t red = (size_t)MT * NS * 64 * 16, tab = (size_t)P * (4 / GS) * 16 * NS * 8;
  const size_t lds = pl.waves * (red > tab ? red : tab);
  hipLaunchKernelGGL((w4a16_group_kernel<T, MT, NS, GS, P>), dim3((unsigned)pl.n_tiles, (unsigned)pl.m_blocks),
                     dim3((unsigned)(64 * pl.waves)), lds, stream, p, pl.per);
  return ss_host::launch_status("w4a16 gemm (group)");
}

template <typename T, int MT, int NS>
int launch_group_g(const W4Params& p, const GroupPlan& pl, hipStream_t stream) {
  if (p.g % 128 == 0) return launch_group<T, MT, NS, 4>(p, pl, stream);
  if (p.g == 64) return launch_group<T, MT, NS, 2>(p, pl, stream);
  return launch_group<T, MT, NS, 1>(p, pl, stream);
}

template <typename T>
int launch_group_typed(const W4Params& p, const GroupPlan& pl, hipStream_t stream) {
  if (pl.mt == 1 && pl.ns == 4) return launch_group_g<T, 1, 4>(p, pl, stream);
  if (pl.mt == 1) return pl.ns == 1 ? launch_group_g<T, 1, 1>(p, pl, stream) : launch_group_g<T, 1, 2>(p, pl, stream);
  if (pl.mt == 2) return pl.ns == 1 ? launch_group_g<T, 2, 1>(p, pl, stream) : launch_group_g<T, 2, 2>(p, pl, stream);
  return launch_group_g<T, 4, 1>(p, pl, stream);
}

}  // namespace

// Weight tiles and waves of a workgroup. The widest workgroup (each activation fragment
// then serves 16 NS weight rows) that still leaves one per CU: at m = 16, g = 64 4096 x
// 28672 32.1 us with four tiles against 34.4 with two and 41.5 with one; at m = 11 896 x
// 9728 5.8 with two (304 workgroups) against 6.5 with four (152) and 7.0 with one; 14336 x
// 4096 (256 workgroups of one tile) 27 against 35 with two. As many waves as there are
// rounds of P stages (896 x 9728: four waves 5.8 us, seven of one stage 6.8), at most
// eight, or sixteen where the grid leaves CUs idle (4864 x 896, 56 workgroups: 8.9 with
// sixteen, 10.0 with eight).
bool plan_w4a16_group(GroupPlan& pl, int64_t m, int64_t n, int64_t k, int g) {
  if (k % 128 || g % 32) return false;
  const int64_t stages = k / 128, cus = ss_host::device_cu_count();
  pl.mt = m <= 16 ? 1 : (m <= 32 ? 2 : 4);
  pl.ns = 1;
  for (int c : {4, 2})
    if (c * pl.mt <= 4 && (n + 16 * c - 1) / (16 * c) >= cus) {
      pl.ns = c;
      break;
    }
  const int64_t round = group_round(pl.mt, pl.ns);
  int64_t waves = (stages + round - 1) / round;
  const int64_t most = (n + 16 * pl.ns - 1) / (16 * pl.ns) >= cus || pl.mt == 4 ? 8 : 16;
  if (waves > most) waves = most;
  pl.per = (int)((stages + waves - 1) / waves);
  pl.waves = (int)((stages + pl.per - 1) / pl.per);
  pl.n_tiles = (int)((n + 16 * pl.ns - 1) / (16 * pl.ns));
  pl.m_blocks = (int)((m + 16 * pl.mt - 1) / (16 * pl.mt));
  return true;
}

int launch_w4a16_group(const W4Params& p, const GroupPlan& pl, int act_dtype, hipStream_t stream) {
  if (act_dtype == SS_DTYPE_BF16) return launch_group_typed<bf16_t>(p, pl, stream);
  return launch_group_typed<f16_t>(p, pl, stream);
}

}  // namespace ss
