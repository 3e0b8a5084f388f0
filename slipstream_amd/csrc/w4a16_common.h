// Device helpers shared by the W4A16 kernels: the call's parameters, int4 unpacking and
// dequantisation, scale decoding, buffer descriptors and LDS DMA.
#pragma once

#include "ss_common.h"

namespace ss {

struct W4Params {
  const void* x;
  void* out;
  const uint32_t* qw;
  const void* sc;
  const int32_t* qz;
  int64_t x_stride, o_stride;  // elements
  int m, n, k, g, groups, sdt;
  int kw;  // waves (K slices) per workgroup
};

// The panel kernel (w4a16_panel.hip): its grid and K split.
struct PanelPlan {
  int mt, ns;  // 16-row activation tiles of a workgroup, 16-row weight tiles of a wave
  int ks, kchunk;  // K ranges and 128-key stages per range
  int n_tiles, m_blocks;
};
// The group kernel (w4a16_group.hip): tiles, waves and stages per wave of a workgroup.
struct GroupPlan {
  int mt, ns, waves, per;
  int n_tiles, m_blocks;
};
bool plan_w4a16_group(GroupPlan& pl, int64_t m, int64_t n, int64_t k, int g);
int launch_w4a16_group(const W4Params& p, const GroupPlan& pl, int act_dtype, hipStream_t stream);

bool plan_w4a16_panel(PanelPlan& pl, int64_t m, int64_t n, int64_t k, int g, double other);
int launch_w4a16_panel(const W4Params& p, const PanelPlan& pl, int act_dtype, float* part, hipStream_t stream);

namespace {


constexpr int kMaxKW = 8;
// Cache policy of the weight loads: non-temporal (every weight is read once per call;
// streaming without cache allocation measured ~14 % more bandwidth on gfx950).
constexpr int kNonTemporal = 2;
// Cache policy sc1 (device scope): a store written through this XCD's L2 to the point of
// device coherence, a load not served by possibly stale lines of this CU's or XCD's caches.
constexpr int kDeviceScope = 16;

// s_waitcnt vmcnt(0): every vector memory operation of this wave, stores included, has
// completed. Inline asm with a memory clobber, so the compiler keeps every load and store
// written before it on this side of the wait (the waitcnt builtin is not a memory
// operation, and the stores it must cover could be sunk past it).
__device__ __forceinline__ void wait_vm0() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Arrival count of one output tile's K ranges in a 64-bit word: bits 8.. hold the call's
// tag, bits 0..7 the ranges arrived. A word with another tag (an earlier call, or memory
// never written) counts as zero arrivals, so the workspace needs no initialisation; the
// last range resets the word to zero, which the first compare-and-swap of the next call
// (or of a replayed launch: a captured graph passes the same tag again) expects.
// No cache maintenance: the partials are device-scope stores the caller has waited for
// (vmcnt 0) before it arrives, the count is a device-scope atomic, and the last range
// reads the partials with device-scope loads. (Release/acquire fences at device scope
// write back or invalidate a whole L2 per wave, several times slower.) This relies on
// sc1 stores reaching the point of device coherence before their vmcnt decrements, and
// on sc1 loads not being served by this XCD's possibly stale L2 lines: the gfx950
// memory model's meaning of the agent-scope cache policy bits.
__device__ __forceinline__ bool arrive_last(unsigned long long* word, unsigned long long tag, int ranges) {
  unsigned long long old = 0ull;
  unsigned long long now;
  do {
    const unsigned long long have = (old & ~0xFFull) == tag ? (old & 0xFFull) : 0ull;
    now = tag | (have + 1);
  } while (!__hip_atomic_compare_exchange_weak(word, &old, now, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                              __HIP_MEMORY_SCOPE_AGENT));
  if ((int)(now & 0xFFull) != ranges) return false;
  __hip_atomic_store(word, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return true;
}

template <typename T>
struct W4Elem;
template <>
struct W4Elem<bf16_t> {
  static constexpr uint32_t kMagicPair = 0x43004300u;  // bf16 128.0 in both halves
  static constexpr uint32_t kOnePair = 0x3F803F80u;    // bf16 1.0 in both halves
  static constexpr float kMagic = 128.f;
  static __device__ __forceinline__ float to_f32(uint32_t h) { return __builtin_bit_cast(float, h << 16); }
};
template <>
struct W4Elem<f16_t> {
  static constexpr uint32_t kMagicPair = 0x64006400u;  // fp16 1024.0 in both halves
  static constexpr uint32_t kOnePair = 0x3C003C00u;    // fp16 1.0 in both halves
  static constexpr float kMagic = 1024.f;
  static __device__ __forceinline__ float to_f32(uint32_t h) {
    return (float)__builtin_bit_cast(f16_t, (uint16_t)h);
  }
};

__device__ __forceinline__ float load_scale(const void* s, int64_t i, int sdt) {
  if (sdt == SS_DTYPE_F16) return (float)((const f16_t*)s)[i];
  if (sdt == SS_DTYPE_BF16) return __builtin_bit_cast(float, (uint32_t)((const uint16_t*)s)[i] << 16);
  return ((const float*)s)[i];
}

// Scales read without branching on their dtype around the load (a load inside a
// dtype branch makes the compiler wait for every outstanding load at the join):
// the aligned dword holding scale gi, through a descriptor over the array (scale_rsrc),
// shifted so the scale's bits are the low ones; decoded afterwards.
__device__ __forceinline__ uint32_t scale_bits(__amdgpu_buffer_rsrc_t rs, int64_t gi, int esize) {
  const int off = (int)(gi * esize);
  return (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rs, off & ~3, 0, 0) >> (8 * (off & 2));
}
__device__ __forceinline__ float decode_scale(uint32_t bits, int sdt) {
  const float f16 = (float)__builtin_bit_cast(f16_t, (uint16_t)(bits & 0xFFFFu));
  const float b16 = __builtin_bit_cast(float, bits << 16);
  return sdt == SS_DTYPE_F16 ? f16 : (sdt == SS_DTYPE_BF16 ? b16 : __builtin_bit_cast(float, bits));
}

// decode_scale without a branch on the dtype (the branches split the loop body into
// blocks, and the compiler then sinks whole folds past them, keeping every stage's
// MFMA partial sums live): all three decodings, merged under uniform bit masks
// (f16_mask / bf16_mask all-ones for that dtype, else zero).
__device__ __forceinline__ float decode_scale_masked(uint32_t bits, uint32_t f16_mask, uint32_t bf16_mask) {
  const uint32_t f16 = __builtin_bit_cast(uint32_t, (float)__builtin_bit_cast(f16_t, (uint16_t)(bits & 0xFFFFu)));
  const uint32_t b16 = bits << 16;
  return __builtin_bit_cast(float, (f16 & f16_mask) | (b16 & bf16_mask) | (bits & ~(f16_mask | bf16_mask)));
}

// Sum over the 16 lanes of a DPP row (every lane of the row gets the total).
template <int CTRL>
__device__ __forceinline__ float dpp_f32(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
}
__device__ __forceinline__ float row16_sum(float x) {
  x += dpp_f32<0xB1>(x);   // quad_perm [1,0,3,2]
  x += dpp_f32<0x4E>(x);   // quad_perm [2,3,0,1]
  x += dpp_f32<0x141>(x);  // row_half_mirror
  x += dpp_f32<0x140>(x);  // row_mirror
  return x;
}

// A constant held in a VGPR. gfx9 VOP3 instructions take no literal and read at most
// one SGPR, so (w & mask) | magic becomes one v_and_or_b32 only when the magic word
// already sits in a VGPR (the mask goes to the SGPR slot); otherwise it takes a
// v_and and a v_or with literals.
__device__ __forceinline__ uint32_t in_vgpr(uint32_t c) {
  uint32_t v;
  asm volatile("v_mov_b32 %0, %1" : "=v"(v) : "s"(c));
  return v;
}

// Eight nibbles -> eight 16-bit (MAGIC + q) values in the order k0,k4,k1,k5,k2,k6,k3,k7.
__device__ __forceinline__ u32x4 nibbles_to_operand(uint32_t w, uint32_t magic) {
  return u32x4{(w & 0x000F000Fu) | magic, ((w >> 4) & 0x000F000Fu) | magic, ((w >> 8) & 0x000F000Fu) | magic,
               ((w >> 12) & 0x000F000Fu) | magic};
}

// Eight consecutive 16-bit x values -> the same order as nibbles_to_operand.
__device__ __forceinline__ u32x4 permute_x(u32x4 d) {
  return u32x4{pick_halves<0, 0>(d[0], d[2]), pick_halves<1, 1>(d[0], d[2]), pick_halves<0, 0>(d[1], d[3]),
               pick_halves<1, 1>(d[1], d[3])};
}

// acc + a.lo * b.lo + a.hi * b.hi over packed 16-bit pairs, fp32 accumulation
template <typename T>
__device__ __forceinline__ float dot2_acc(uint32_t a, uint32_t b, float acc);
template <>
__device__ __forceinline__ float dot2_acc<bf16_t>(uint32_t a, uint32_t b, float acc) {
  typedef short s16x2 __attribute__((ext_vector_type(2)));
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(s16x2, a), __builtin_bit_cast(s16x2, b), acc, false);
}
template <>
__device__ __forceinline__ float dot2_acc<f16_t>(uint32_t a, uint32_t b, float acc) {
  typedef _Float16 h16x2 __attribute__((ext_vector_type(2)));
  return __builtin_amdgcn_fdot2(__builtin_bit_cast(h16x2, a), __builtin_bit_cast(h16x2, b), acc, false);
}

// Raw buffer resource over [base, base + bytes): loads past the end return 0, and a
// per-iteration offset rides in the scalar offset, so the loop does no 64-bit
// address arithmetic.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, 0x00020000);
}

// Over the scales, their last dword counted whole: a dword that reaches past the descriptor
// comes back as zero, and with it the last of an odd number of 16-bit scales. (The array is
// then 4-byte aligned, host-checked, so that the dword lies in one page.)
__device__ __forceinline__ __amdgpu_buffer_rsrc_t scale_rsrc(const W4Params& p, int esize) {
  return buffer_rsrc(p.sc, ((uint32_t)((int64_t)p.n * p.groups * esize) + 3u) & ~3u);
}

constexpr int kOutOfRange = 0x40000000;  // buffer offset past any operand (< 2^31 bytes)

// Eight int4 weights (one word: keys 8j .. 8j + 7 of a row) -> the MFMA B fragment
// T((q - z) * s) in key order, computed as fma(q, s, -z s) in fp32 and rounded once
// to the activation type. (The reference rounds (q - z) * s to the scales' dtype and
// then to the activation dtype, quant_ref.py:112-116,132; with fp16 scales and bf16
// activations the single rounding differs from that double rounding by at most one
// bf16 ulp of a weight.) Per word: two masks, eight byte converts (v_cvt_f32_ubyteN),
// eight FMAs and four packs.
template <typename T>
__device__ __forceinline__ u32x4 dequant_word(uint32_t w, float s, float nzs) {
  // the masks as asm, so that the compiler does not fold each (lo >> 8b) & 0xFF into a
  // 4-bit field extract and lose the byte converts' own byte select
  uint32_t lo, hi;
  asm("v_and_b32 %0, 0x0f0f0f0f, %1" : "=v"(lo) : "v"(w));
  asm("v_and_b32 %0, 0x0f0f0f0f, %1" : "=v"(hi) : "v"(w >> 4));
  u32x4 r;
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const float qa = (float)((lo >> (8 * b)) & 0xFFu), qb = (float)((hi >> (8 * b)) & 0xFFu);
    r[b] = Elem<T>::pack2(fmaf(qa, s, nzs), fmaf(qb, s, nzs));
  }
  return r;
}

// Scale of SD (a dtype code) from its raw bits (the low 16 bits for 16-bit scales).
template <int SD>
__device__ __forceinline__ float scale_from_bits(uint32_t b) {
  if constexpr (SD == SS_DTYPE_F16) return (float)__builtin_bit_cast(f16_t, (uint16_t)(b & 0xFFFFu));
  if constexpr (SD == SS_DTYPE_BF16) return __builtin_bit_cast(float, b << 16);
  return __builtin_bit_cast(float, b);
}

// Buffer loads for the wide kernel, written as asm: the compiler inserts no vmcnt wait
// of its own for them (its count of loads in flight, merged around the loop's back
// edge, made it wait for nearly every prefetched stage at the top of each stage). The
// kernel waits itself, with vm_wait_tied, whose register operands keep every use of a
// loaded value behind the wait. Descriptors are plain SGPR quads over [base, base + bytes):
// offsets past the end read zeros without a memory access.
typedef int i32x4w __attribute__((ext_vector_type(4)));
__device__ __forceinline__ i32x4w wide_rsrc(const void* base, uint32_t bytes) {
  const uint64_t a = (uint64_t)base;
  return i32x4w{(int)(uint32_t)a, (int)((uint32_t)(a >> 32) & 0xFFFF), (int)bytes, 0x00020000};
}
__device__ __forceinline__ u32x4 asm_load_b128_nt(i32x4w rs, int voff, int soff) {
  u32x4 v;
  asm volatile("buffer_load_dwordx4 %0, %1, %2, %3 offen nt" : "=v"(v) : "v"(voff), "s"(rs), "s"(soff));
  return v;
}
__device__ __forceinline__ uint32_t asm_load_b32(i32x4w rs, int voff) {
  uint32_t v;
  asm volatile("buffer_load_dword %0, %1, %2, 0 offen" : "=v"(v) : "v"(voff), "s"(rs));
  return v;
}
__device__ __forceinline__ uint32_t asm_load_u16(i32x4w rs, int voff) {
  uint32_t v;
  asm volatile("buffer_load_ushort %0, %1, %2, 0 offen" : "=v"(v) : "v"(voff), "s"(rs));
  return v;
}

// 16 bytes per lane from rs + voff + soff straight into LDS at lds + 16 * lane
// (buffer_load_dwordx4 ... lds; M0 holds the LDS destination). The s_nop: M0 is
// written just before by the compiler, and the load may read it one wait state later.
typedef __attribute__((address_space(3))) char* LdsW;
__device__ __forceinline__ void asm_dma_b128(i32x4w rs, LdsW lds, int voff, int soff) {
  const uint32_t m0 = (uint32_t)(uintptr_t)lds;
  asm volatile("s_nop 1\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds"
               :
               : "v"(voff), "s"(rs), "s"(soff), "{m0}"(m0)
               : "memory");
}

}  // namespace
}  // namespace ss
