// mm_operand.hpp — Q4_K / Q6_K weight tiles as matrix-core A operands, shared
// by the batched matmuls (k_batch.hip, k_head.hip) and the prefill matmul
// (k_prefill.hip): the loads of one 16-row tile and super-block and their conversion to f16
// sc * q values in the v_mfma_f32_16x16x32_f16 operand order.
#pragma once
#include <utility>

#include "g4_internal.hpp"

namespace g4mm {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x3a __attribute__((ext_vector_type(3), aligned(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));  // native vector: stays in registers

__device__ __forceinline__ uint32_t pack_h2(_Float16 a, _Float16 b) {
  h2 v = {a, b};
  return __builtin_bit_cast(uint32_t, v);
}

// f(0), f(1), ... f(N - 1), each index a compile-time constant.
template <typename F, int... J>
__device__ __forceinline__ void static_for_seq(F&& f, std::integer_sequence<int, J...>) {
  (f(std::integral_constant<int, J>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_seq(f, std::make_integer_sequence<int, N>{});
}

// Waits until at most N of the wave's memory loads are in flight.
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt field");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}
// Barrier after which LDS written before it (global -> LDS loads: by waves
// that waited for them) is readable; waits for no load in flight, unlike
// __syncthreads's fence.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// A logit's softcap (shaders/logit_softcap.wgsl), none for cap 0.
__device__ __forceinline__ float epilogue(float y, float cap) {
  if (cap > 0.f) {
    const float t = fminf(fmaxf(y / cap, -15.0f), 15.0f);
    return tanhf(t) * cap;
  }
  return y;
}

template <int QT>
struct Blk;
template <> struct Blk<0> { static constexpr int BYTES = 144; };
template <> struct Blk<1> { static constexpr int BYTES = 210; };

// Weight registers of one 16-row tile and super-block. A side (row lane%16,
// k-group q = lane/16): codes and sub-block scales; D side (rows 4q + i): d
// (Q4_K: d | dmin << 16).
template <int QT>
struct WRegs;
template <> struct WRegs<0> {
  uint2 qs[4];
  uint4 hdr;
  uint32_t dd[4];
};
template <> struct WRegs<1> {
  uint2 ql[4], qh[2];
  uint4 sc;
  uint32_t dd[4];
};

// What load_w leaves in registers: the weights as loaded. Q4_K blocks are
// 16-byte aligned and load straight into WRegs; a Q6_K block (210 bytes) may
// sit 2 bytes off a dword, so its pieces are loaded as the aligned dwords
// around them and shifted into place by w_decode where they are used (a
// shift at the load would wait for the load there, also for the weights of
// a block that is only prefetched).
template <int QT>
struct WLoad;
template <> struct WLoad<0> {
  WRegs<0> r;
};
template <> struct WLoad<1> {
  u32x3a ql[4], qh[2];
  uint32_t s0, s1, s2, s3, s4;  // the dwords around the 16 scale bytes
  uint32_t dd[4];
  uint32_t sh;                  // the block's byte offset within its dword (0 or 2)
};

__device__ __forceinline__ void load_w(WLoad<0>& ld, const uint8_t* W, uint32_t M, uint32_t bpr, uint32_t rbase,
                                       uint32_t kb, int l) {
  WRegs<0>& r = ld.r;
  constexpr int BY = 144;
  const int q = l >> 4;
  const uint32_t ra = min(rbase + (uint32_t)(l & 15), M - 1);
  const uint8_t* blk = W + ((size_t)ra * bpr + kb) * BY;
  r.hdr = *(const uint4*)blk;
#pragma unroll
  for (int g = 0; g < 4; ++g) r.qs[g] = *(const uint2*)(blk + 16 + 32 * g + 8 * q);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t rd = min(rbase + 4u * q + i, M - 1);
    r.dd[i] = *(const uint32_t*)(W + ((size_t)rd * bpr + kb) * BY);
  }
}

__device__ __forceinline__ void load_w(WLoad<1>& r, const uint8_t* W, uint32_t M, uint32_t bpr, uint32_t rbase,
                                       uint32_t kb, int l) {
  constexpr int BY = 210;
  const int q = l >> 4;
  const uint32_t ra = min(rbase + (uint32_t)(l & 15), M - 1);
  const uint8_t* blk = W + ((size_t)ra * bpr + kb) * BY;
  // every piece sits at a multiple of 8 bytes into the block: one shift for all
  r.sh = (uint32_t)((uintptr_t)blk & 3);
  const uint8_t* b4 = blk - r.sh;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    r.ql[2 * h] = *(const u32x3a*)(b4 + 64 * h + 8 * q);
    r.ql[2 * h + 1] = *(const u32x3a*)(b4 + 64 * h + 32 + 8 * q);
    r.qh[h] = *(const u32x3a*)(b4 + 128 + 32 * h + 8 * q);
  }
  // sc[16] at bytes 192..207: four dwords from the one holding byte 192 and
  // a fifth (bytes 206..209) that only a block at 2 mod 4 needs
  const uint32_t* p4 = (const uint32_t*)(b4 + 192);
  r.s0 = p4[0];
  r.s1 = p4[1];
  r.s2 = p4[2];
  r.s3 = p4[3];
  r.s4 = *(const uint32_t*)((const uint8_t*)p4 + 12 + 2 * r.sh);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t rd = min(rbase + 4u * q + i, M - 1);
    r.dd[i] = *(const uint16_t*)(W + ((size_t)rd * bpr + kb) * BY + 208);
  }
}

__device__ __forceinline__ const WRegs<0>& w_decode(const WLoad<0>& ld) { return ld.r; }
__device__ __forceinline__ WRegs<1> w_decode(const WLoad<1>& ld) {
  WRegs<1> r;
  const uint32_t sh = ld.sh;
  auto piece = [&](const u32x3a& w) {
    return make_uint2(__builtin_amdgcn_alignbyte(w.y, w.x, sh), __builtin_amdgcn_alignbyte(w.z, w.y, sh));
  };
#pragma unroll
  for (int i = 0; i < 4; ++i) r.ql[i] = piece(ld.ql[i]);
#pragma unroll
  for (int h = 0; h < 2; ++h) r.qh[h] = piece(ld.qh[h]);
  r.sc = make_uint4(__builtin_amdgcn_alignbyte(ld.s1, ld.s0, sh), __builtin_amdgcn_alignbyte(ld.s2, ld.s1, sh),
                    __builtin_amdgcn_alignbyte(ld.s3, ld.s2, sh), __builtin_amdgcn_alignbyte(ld.s4, ld.s3, sh));
#pragma unroll
  for (int i = 0; i < 4; ++i) r.dd[i] = ld.dd[i];
  return r;
}

// f16 pairs (1024 + b_i, 1024 + b_j) from two bytes of `codes`: v_perm_b32
// takes selector bytes 0-3 from its second operand and 4-7 from its first.
__device__ __forceinline__ h2 biased_pair(uint32_t codes, uint32_t sel) {
  return __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, codes, sel));
}
constexpr uint32_t kSel01 = 0x04010400u, kSel23 = 0x04030402u;

__device__ __forceinline__ h8 cat(h2 a, h2 b, h2 c, h2 d) { return h8{a.x, a.y, b.x, b.y, c.x, c.y, d.x, d.y}; }

// Q4_K 6-bit scale and min of sub-block j (src/gguf.ts:175-182).
__device__ __forceinline__ void q4k_sc_mn(const uint4& hdr, int j, uint32_t& sc, uint32_t& mn) {
  const int sh = 8 * (j & 3);
  if (j < 4) {
    sc = (hdr.y >> sh) & 63u;
    mn = (hdr.z >> sh) & 63u;
  } else {
    sc = ((hdr.w >> sh) & 15u) | (((hdr.y >> sh) >> 6 & 3u) << 4);
    mn = ((hdr.w >> sh) >> 4 & 15u) | (((hdr.z >> sh) >> 6 & 3u) << 4);
  }
}

// Weight operand of sub-block s: 8 f16 values sc * q of row lane%16, k = 8q .. 8q+7.
__device__ __forceinline__ h8 a_operand(const WRegs<0>& r, int s, int) {
  const uint2 raw = r.qs[s >> 1];
  const uint32_t c0 = (s & 1) ? (raw.x >> 4) & 0x0f0f0f0fu : raw.x & 0x0f0f0f0fu;
  const uint32_t c1 = (s & 1) ? (raw.y >> 4) & 0x0f0f0f0fu : raw.y & 0x0f0f0f0fu;
  uint32_t sc, mn;
  q4k_sc_mn(r.hdr, s, sc, mn);
  const _Float16 f = (_Float16)(float)sc;
  const _Float16 fb = (_Float16)(-1024.0f * (float)sc);  // exact: sc <= 63
  const h2 mul = {f, f}, bias = {fb, fb};
  // (1024 + c) * sc - 1024 * sc = c * sc, one rounding of an exact value
  return cat(__builtin_elementwise_fma(biased_pair(c0, kSel01), mul, bias),
             __builtin_elementwise_fma(biased_pair(c0, kSel23), mul, bias),
             __builtin_elementwise_fma(biased_pair(c1, kSel01), mul, bias),
             __builtin_elementwise_fma(biased_pair(c1, kSel23), mul, bias));
}

// Q6_K sub-block s: half h = s/4, run pair k' = s%4 (src/gguf.ts:344-361);
// this lane's 8 codes lie in run q/2 of the sub-block.
__device__ __forceinline__ h8 a_operand(const WRegs<1>& r, int s, int q) {
  const int h = s >> 2, kp = s & 3;
  const uint2 ql = r.ql[2 * h + (kp & 1)];
  const uint2 qh = r.qh[h];
  const uint32_t lo0 = kp < 2 ? (ql.x & 0x0f0f0f0fu) : ((ql.x >> 4) & 0x0f0f0f0fu);
  const uint32_t lo1 = kp < 2 ? (ql.y & 0x0f0f0f0fu) : ((ql.y >> 4) & 0x0f0f0f0fu);
  const uint32_t c0 = lo0 | (((qh.x >> (2 * kp)) & 0x03030303u) << 4);
  const uint32_t c1 = lo1 | (((qh.y >> (2 * kp)) & 0x03030303u) << 4);
  const int is = 8 * h + 2 * kp + (q >> 1);
  const uint32_t wd = (is < 4) ? r.sc.x : (is < 8) ? r.sc.y : (is < 12) ? r.sc.z : r.sc.w;
  const int scv = (int)(int8_t)((wd >> (8 * (is & 3))) & 0xffu);
  const _Float16 f = (_Float16)(float)scv;
  const h2 mul = {f, f};
  const h2 off = {(_Float16)-1056.0f, (_Float16)-1056.0f};
  // (1024 + c) - 1056 = c - 32 exactly, then one rounding of (c - 32) * sc
  return cat((biased_pair(c0, kSel01) + off) * mul, (biased_pair(c0, kSel23) + off) * mul,
             (biased_pair(c1, kSel01) + off) * mul, (biased_pair(c1, kSel23) + off) * mul);
}

// Min operand of a Q4_K super-block: slots 8q .. 8q+3 hold the min of
// sub-block 2q, slots 8q+4 .. +7 that of sub-block 2q+1.
__device__ __forceinline__ h8 min_operand(const WRegs<0>& r, int q) {
  uint32_t sc0, m0, sc1, m1;
  q4k_sc_mn(r.hdr, 2 * q, sc0, m0);
  q4k_sc_mn(r.hdr, 2 * q + 1, sc1, m1);
  const _Float16 a = (_Float16)(float)m0, b = (_Float16)(float)m1;
  return h8{a, a, a, a, b, b, b, b};
}

}  // namespace g4mm
