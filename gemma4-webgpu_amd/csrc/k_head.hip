// k_head.hip — matmul of a tall Q6_K matrix (the LM head) and up to 32
// activation vectors on the gfx950 matrix cores (the logits of
// src/engine.ts:1686-1717 for several sequences at once).
//
// k_batch.hip's waves (mmf_kernel) read their 16 rows' blocks straight into registers, 14
// loads of 16 scattered rows per super-block, and each of its thousands of
// workgroups copies every operand into LDS: 2.8 TB/s at 16 vectors. Here
// persistent workgroups walk tiles of 16 whole rows, which are one
// contiguous run of bytes and arrive by 1 KB global -> LDS loads in a ring of
// D tiles; wave w owns super-block w of the width for every tile, so its
// vectors' operands stay in registers (64 per 16 vectors) and the waves share
// nothing but the tile. Their partial sums meet through LDS, every thread
// adding one output's in super-block order before the next tile is
// multiplied: one barrier per tile. A tile costs a wave 250 VALU instructions
// (40 us of 262144 x 1536); the chain from barrier to barrier bounds it, above
// the 64 us of its bytes.
#include "mm_operand.hpp"

namespace {

using namespace g4mm;
using g4d::Ops;

struct TallArgs {
  const uint8_t* W;    // [M] rows of NSB Q6_K blocks
  float* Y;            // [B][M]
  uint32_t M, B;
  float cap;           // softcap when > 0
  const uint8_t* ops;  // [NSB][Ops::bytes(NTV)]
};

template <int NSB, int NTV>
struct Mlh {
  static constexpr uint32_t RB = NSB * Blk<1>::BYTES, TB = 16 * RB;  // bytes of a row, of a tile
  static constexpr int NP = (TB + 1023) / 1024, PW = (NP + NSB - 1) / NSB;  // 1 KB pieces, of a wave
  static constexpr uint32_t BUF = NP * 1024;
  static constexpr int WGS = NTV == 1 ? 2 : 1;  // workgroups per CU
  static constexpr int D = NTV == 2 || BUF <= 16384 ? 4 : (BUF <= 20480 ? 3 : 2);
  static constexpr uint32_t RED = NSB * NTV * 1024;  // a tile's partial sums
  static_assert(WGS * (D * BUF + 2 * RED) <= 160 * 1024, "LDS");
};

// 16 bytes per lane from src to LDS at dst + 16 lane, non-temporal. Written as
// the instruction itself because the compiler, which knows the builtin's LDS
// write, waits for every such load before any pair of LDS reads it merges
// (read2 loses the object they belong to); the waits are the caller's
// wait_vmcnt and lds_barrier. (m0 takes the LDS address, with one wait state
// after its write. It is a reserved register, which the compiler sets at each
// use of its own and never keeps a value in, so a clobber entry says nothing;
// nothing else in this file's code uses it.)
__device__ __forceinline__ void to_lds_unwaited(const void* src, uint8_t* dst) {
  const uint32_t at = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)dst);
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off nt" ::"v"(src), "s"(at) : "memory");
}
// A lane's row of a tile in LDS (blk: its block; sh: the block's offset within
// its dword, uniform over the wave) as matrix-core weight registers.
__device__ __forceinline__ WRegs<1> lds_weights(const uint8_t* blk, int q, uint32_t sh) {
  WRegs<1> r;
  const uint8_t* b4 = blk - sh;
  auto piece = [&](uint32_t o) {
    const uint32_t* p = (const uint32_t*)(b4 + o);
    const uint32_t x = p[0], y = p[1], z = p[2];
    return make_uint2(__builtin_amdgcn_alignbyte(y, x, sh), __builtin_amdgcn_alignbyte(z, y, sh));
  };
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    r.ql[2 * h] = piece(64u * h + 8u * q);
    r.ql[2 * h + 1] = piece(64u * h + 32u + 8u * q);
    r.qh[h] = piece(128u + 32u * h + 8u * q);
  }
  const uint32_t* p = (const uint32_t*)(b4 + 192);
  const uint32_t s0 = p[0], s1 = p[1], s2 = p[2], s3 = p[3], s4 = p[4];  // (s4: d's dword)
  r.sc = make_uint4(__builtin_amdgcn_alignbyte(s1, s0, sh), __builtin_amdgcn_alignbyte(s2, s1, sh),
                    __builtin_amdgcn_alignbyte(s3, s2, sh), __builtin_amdgcn_alignbyte(s4, s3, sh));
  return r;
}

template <int NSB, int NTV>
__global__ __launch_bounds__(64 * NSB, NTV == 1 ? 3 : 2) void mlh_kernel(TallArgs a) {
  using P = Mlh<NSB, NTV>;
  constexpr int D = P::D;
  __shared__ __align__(16) uint8_t r0[P::BUF], r1[P::BUF], r2[P::BUF], r3[D == 4 ? P::BUF : 16];
  __shared__ __align__(16) f4 red[2 * NSB * NTV * 64];
  uint8_t* const ring[4] = {r0, r1, r2, r3};
  const int tid = threadIdx.x, l = tid & 63, q = l >> 4, c = l & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint8_t* const W = a.W;
  float* const Y = a.Y;
  const uint32_t M = a.M, tiles = (M + 15) / 16, G = gridDim.x;
  const uint32_t n = (tiles - blockIdx.x + G - 1) / G;  // this workgroup's tiles: blockIdx.x + G i (G <= tiles)

  // a tile's first row: the last tile of a matrix whose rows are no multiple of
  // 16 starts early, its first rows the same as the tile's before it
  auto row0 = [&](uint32_t i) { return min((blockIdx.x + G * i) * 16u, M - 16u); };
  // tile i into its slot; past the end the last one again, so that every turn
  // issues the same number of loads (16 rows are a multiple of 16 bytes; the
  // lanes past a tile's end read its last 16)
  auto stage = [&](uint32_t i, uint8_t* buf) {
    const uint8_t* src = W + (size_t)row0(min(i, n - 1u)) * P::RB;
#pragma unroll
    for (int k = 0; k < P::PW; ++k) {
      const uint32_t pc = min((uint32_t)(w + k * NSB), (uint32_t)P::NP - 1u);
      to_lds_unwaited(src + min(pc * 1024u + l * 16u, P::TB - 16u), buf + pc * 1024u);
    }
  };
  static_for<D - 1>([&](auto ic) { stage(decltype(ic)::value, ring[decltype(ic)::value]); });

  // this wave's super-block of every vector
  const uint8_t* ob = a.ops + (size_t)w * Ops::bytes(NTV);
  h8 bh[8][NTV], bl[8][NTV];
  float fs[NTV];
#pragma unroll
  for (int t = 0; t < NTV; ++t) {
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      bh[s][t] = *(const h8*)(ob + t * Ops::MAIN_T + s * 2048 + l * 16);
      bl[s][t] = *(const h8*)(ob + t * Ops::MAIN_T + s * 2048 + 1024 + l * 16);
    }
    fs[t] = *(const float*)(ob + Ops::scale_off(NTV) + t * 64 + c * 4);
  }
  wait_vmcnt<0>();

  // adds tile i's partial sums in super-block order and stores its outputs,
  // one per thread: output o is row o % 16 of vector o / 16
  auto reduce = [&](uint32_t i) {
#pragma unroll
    for (int o0 = 0; o0 < 256 * NTV; o0 += 64 * NSB) {
      const int o = o0 + tid, v = o >> 4, r = o & 15;
      if (o >= 256 * NTV) break;
      const float* x = (const float*)(red + (i & 1u) * NSB * NTV * 64) + ((v >> 4) * 64 + (r >> 2) * 16 + (v & 15)) * 4 +
                       (r & 3);
      float y = x[0];
#pragma unroll
      for (int k = 1; k < NSB; ++k) y += x[k * NTV * 256];
      if ((uint32_t)v < a.B) Y[(size_t)v * M + row0(i) + r] = epilogue(y, a.cap);
    }
  };

  for (uint32_t i0 = 0; i0 < n; i0 += D)
    static_for<D>([&](auto ic) {
      constexpr int I = decltype(ic)::value;
      const uint32_t i = i0 + I;
      if (i >= n) return;  // (uniform)
      // tile i was requested D - 1 turns ago; D - 2 later tiles may be in flight
      // (a store among them makes the wait stricter)
      wait_vmcnt<P::PW*(D - 2)>();
      lds_barrier();  // the tile is in LDS, the last one's partial sums are; its slot is free
      stage(i + D - 1, ring[(I + D - 1) % D]);
      __builtin_amdgcn_sched_barrier(0);
      if (i > 0) reduce(i - 1);
      const uint8_t* tile = ring[I] + w * Blk<1>::BYTES;
      const WRegs<1> wr = lds_weights(tile + c * P::RB, q, (uint32_t)(w * Blk<1>::BYTES) & 3u);
      float d[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) d[k] = g4d::f16_bits_to_f32(*(const uint16_t*)(tile + (4 * q + k) * P::RB + 208));
      f4 C[NTV], Cl[NTV];
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        const h8 A = a_operand(wr, s, q);
#pragma unroll
        for (int t = 0; t < NTV; ++t) {
          const f4 z = f4{0.f, 0.f, 0.f, 0.f};
          C[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A, bh[s][t], s == 0 ? z : C[t], 0, 0, 0);
          Cl[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A, bl[s][t], s == 0 ? z : Cl[t], 0, 0, 0);
        }
      }
#pragma unroll
      for (int t = 0; t < NTV; ++t) {
        f4 y;
#pragma unroll
        for (int k = 0; k < 4; ++k) y[k] = fs[t] * d[k] * (C[t][k] + Cl[t][k]);
        red[(((i & 1u) * NSB + w) * NTV + t) * 64 + l] = y;
      }
    });
  wait_vmcnt<0>();  // no load into this workgroup's LDS outlives it
  lds_barrier();
  reduce(n - 1);
}

template <int NSB, int NTV>
int mlh_launch(g4_ctx* ctx, const TallArgs& a) {
  const uint32_t cus = (uint32_t)(ctx->num_cus > 0 ? ctx->num_cus : 256);
  hipLaunchKernelGGL((mlh_kernel<NSB, NTV>), dim3(Mlh<NSB, NTV>::WGS * cus), dim3(64 * NSB), 0, ctx->stream, a);
  G4_LAUNCHED(ctx, "mlh");
  return G4_OK;
}

}  // namespace

int g4_internal_tall_q6k(g4_ctx* ctx, const uint8_t* W, float* Y, uint32_t M, uint32_t K, const uint8_t* ops,
                         uint32_t B, float cap) {
  const TallArgs a{W, Y, M, B, cap, ops};
  if (K == 1536) return B <= 16 ? mlh_launch<6, 1>(ctx, a) : mlh_launch<6, 2>(ctx, a);
  return B <= 16 ? mlh_launch<8, 1>(ctx, a) : mlh_launch<8, 2>(ctx, a);
}
