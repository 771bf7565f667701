// k_prefill.hip — quantized matmuls for a whole prompt (hundreds to
// thousands of activation vectors) on the gfx950 matrix cores.
//
// The reference prefills one token at a time (src/engine.ts:1923-1938); the
// ragged step's matmul (k_batch.hip) takes 64 vectors a launch and gives each
// wave one 16-row tile, so every 64 tokens re-read and re-decode every
// weight, and a wave reads 4 KB of activation operands from LDS for each
// 1 KB weight operand. Here one pass takes the prompt:
//  * unpack_kernel decodes a launch's matrices once into matrix-core operand
//    order in a scratch buffer (f16 sc * q, the values k_batch.hip's waves
//    form in registers; the f16 row d's and the Q4_K mins beside them). It
//    costs one write and one read of 2 B per weight: 7 % of a 1900-token
//    pass, 13 % of a 512-token one; decoding in the matmul instead would
//    repeat per 64 tokens and take about as many VALU cycles as the products
//    take matrix-core cycles.
//  * pf_gemm_kernel: a workgroup (4 waves) owns 64 RT rows (RT 16-row tiles
//    per wave) x 64 vectors. The weight operands go from memory (L2) straight
//    into registers, 1 KB contiguous per wave load; the activation operands
//    (f16 hi + lo, twice the bytes) are shared by the waves through LDS. With
//    RT = 4 a wave issues 32 MFMAs per 8 KB of LDS reads, half the LDS rate;
//    with all operands in LDS the reads would take as long as the products.
//    Both streams run three to four 32-k sub-blocks ahead (about 1.5 us): a
//    form with the next 64 k in flight, whose loads the compiler moved next
//    to their use, spent 13 us per super-block, eight times its products,
//    waiting for memory (gate/up 2 x 6144 x 1536 at 1900 vectors 241 -> 156
//    us, o 101 -> 55, down 12288 wide 159 -> 138: 1040 TFLOP/s of f16 products).
// The arithmetic is that of mmf_kernel: x * 2^e as f16 hi + lo, exact f16
// sc * q (Q6_K rounds once above 2048), f32 accumulation over half a
// super-block, then d and 2^-e in f32 (the min term with the super-block's
// second half). mmf_kernel keeps the hi and the lo sums of a super-block apart,
// which there are no registers for here; the lo products before the hi ones and
// half the chain match its accuracy. Relative error against float64, 64 vectors
// x 1536, Q4_K and Q6_K with exact operands: mmf_kernel 2.7e-7 and 1.23e-7, this
// 2.7e-7 and 1.24e-7, whole super-blocks with hi first 3.4e-7 and 1.6e-7 (gate/up
// 2 x 12288 at 1900 vectors 331 us so, 329 as it is; o 55.5 and 56; q/k/v 66 both).
#include <algorithm>

#include "mm_operand.hpp"

namespace {

using namespace g4mm;
using g4d::PfOps;

constexpr int NT = 256;
constexpr int kMaxSeg = 4;

struct PfSeg {
  const uint8_t* W;
  float* Y;       // [ksplit][T][rows]
  uint32_t rows;
  uint32_t rt0;   // first row tile
};

// Unpacked weights of one launch: rtn row tiles of 16 rows (each segment
// padded to whole tiles, the padding repeating its last row).
struct PfWeights {
  uint8_t* A;  // [rtn][K/32][64 lanes] 16 B: f16 sc * q of row lane % 16, k = 32s + 8 (lane / 16) .. +7
  uint8_t* X;  // [rtn][K/256][Aux<QT>::BYTES]: see Aux
};
// A row tile and super-block's values beside the operands: d [16 rows] f32;
// Q4_K also 64 dmin [16 rows] f32 and per lane the f16 mins of row lane % 16,
// sub-blocks 2 (lane / 16) and + 1. CH: its 16-byte pieces.
template <int QT>
struct Aux {
  static constexpr uint32_t BYTES = QT == 0 ? 384 : (QT == 1 ? 64 : 0);
  static constexpr uint32_t DM = 64, MN = 128, CH = BYTES / 16;
};
uint32_t aux_bytes(int wtype) { return wtype == 0 ? Aux<0>::BYTES : (wtype == 1 ? Aux<1>::BYTES : 0u); }

struct PfArgs {
  PfSeg s[kMaxSeg];
  int n;
  PfWeights w;
  uint32_t rtn, K, nsb;  // row tiles; width; super-blocks of the width
  const uint8_t* ops;    // [T / 64][nsb][PfOps::BYTES]
  const uint8_t* ops_lo; // f16 matrices: the third term, [T / 64][nsb][PfOps::LO_BYTES], or null
  uint32_t T, ntt;       // vectors, tiles of 64
  uint32_t ksplit, kc;
  uint32_t groups, items;
  uint8_t* ops_out;  // gate/up: the product's operands [T / 64][rows / 256][PfOps::BYTES]
};

template <int QT>
__global__ __launch_bounds__(NT) void unpack_kernel(PfArgs a) {
  const int l = threadIdx.x & 63, q = l >> 4, c = l & 15;
  const uint32_t u = blockIdx.x * 4u + (threadIdx.x >> 6);  // (row tile, super-block)
  if (u >= a.rtn * a.nsb) return;
  const uint32_t rt = u / a.nsb, sb = u % a.nsb;
  const uint8_t* W = a.s[0].W;
  uint32_t M = a.s[0].rows, rt0 = 0;
#pragma unroll
  for (int i = 1; i < kMaxSeg; ++i)
    if (i < a.n && rt >= a.s[i].rt0) {
      W = a.s[i].W;
      M = a.s[i].rows;
      rt0 = a.s[i].rt0;
    }
  const uint32_t rbase = (rt - rt0) * 16u;
  u32x4* out = (u32x4*)a.w.A + ((size_t)rt * (a.K / 32) + sb * 8u) * 64u + l;
  if constexpr (QT == 2) {  // f16 rows: only the order changes
    const u32x4* row = (const u32x4*)(W + ((size_t)min(rbase + (uint32_t)c, M - 1) * a.K + sb * 256u + 8u * q) * 2u);
#pragma unroll
    for (int s = 0; s < 8; ++s) out[s * 64] = row[s * 4];
  } else {
    WLoad<QT> ld;
    load_w(ld, W, M, a.nsb, rbase, sb, l);
    const auto& wr = w_decode(ld);
#pragma unroll
    for (int s = 0; s < 8; ++s) out[s * 64] = __builtin_bit_cast(u32x4, a_operand(wr, s, q));
    float4 d, dm = make_float4(0.f, 0.f, 0.f, 0.f);
    float* dp = (float*)&d;
    float* dmp = (float*)&dm;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      dp[i] = g4d::f16_bits_to_f32(wr.dd[i] & 0xffffu);
      if constexpr (QT == 0) dmp[i] = g4d::f16_bits_to_f32(wr.dd[i] >> 16) * 64.0f;
    }
    uint8_t* x = a.w.X + ((size_t)rt * a.nsb + sb) * Aux<QT>::BYTES;
    if (c == 0) *(float4*)(x + 16 * q) = d;
    if constexpr (QT == 0) {
      if (c == 0) *(float4*)(x + Aux<0>::DM + 16 * q) = dm;
      const h8 m = min_operand(wr, q);
      *(uint32_t*)(x + Aux<0>::MN + 4 * l) = pack_h2(m[0], m[4]);
    }
  }
}

// One 32-k sub-block of the four vector tiles in LDS (f16 hi and lo, 2 KB a
// tile), in a ring of four, and the values a super-block's sums need, in
// turn: the vectors' part (their sub-block sums and 2^-e) and each wave's own
// row tiles'. Separate LDS objects: the compiler then waits for a
// global -> LDS load only where its own object is read.
constexpr uint32_t SUB = 4 * 2048;
constexpr uint32_t VAUX_LDS = 5120;  // an operand block's sums and scales (4608 B), in whole 1 KB loads
constexpr uint32_t WAUX_LDS = 2048;  // a wave's row tiles' Aux values, likewise

__device__ __forceinline__ void to_lds(const void* src, uint8_t* dst) {  // 16 bytes per lane, dst + 16 lane
  __builtin_amdgcn_global_load_lds(src, (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}

// MODE 0: row group g is row tiles 4 RT g .. +4 RT - 1 of the segments in
// order, RT consecutive tiles per wave. MODE 1 (gate/up, RT 4): segments 0
// and 1 have the same rows; a row group is 128 rows of both, a wave's tiles
// 0-1 the gate's and 2-3 the up's same 32 rows, so gelu(gate) * up needs no
// exchange; the product leaves as the down projection's operands, one
// 32-row sub-block per wave, one 2^e per vector and 128 rows (the four
// waves' maxima meet in LDS). SG: scale groups per super-block of the
// operands read (2 for that product, 1 otherwise: both halves equal). TERMS 3
// (f16 matrices): the vectors with their third term, each sub-block's products
// added in f32 to the super-block's sums (even and odd ones apart), for the
// accuracy of the f32 matvec (hmv_kernel) that f16 matrices take in a step:
// relative error against float64, 256 x 1536 and 1536 x 256, matvec 9.2e-8 and
// 7.8e-8, three terms 9.4e-8 and 6.9e-8, two terms 1.6e-7 and 1.5e-7. At 1900
// vectors the 8960-row model projection 123 -> 208 us for it, a layer's gate and
// proj 14 -> 17 and 14 -> 16 (as matvecs all of them took 9.5 ms of that prompt).
template <int QT, int RT, int MODE, int SG, int TERMS = 2>
__global__ __launch_bounds__(NT, 2) void pf_gemm_kernel(PfArgs a) {
  static_assert(MODE == 0 || RT == 4, "gate/up: two tiles of each");
  static_assert(TERMS == 2 || (QT == 2 && RT == 2 && MODE == 0 && SG == 1), "three terms: f16 rows");
  constexpr int FL = TERMS == 3 ? 8 : 4;  // sub-blocks summed before d and 2^-e
  __shared__ __align__(16) uint8_t b0[SUB], b1[SUB], b2[SUB], b3[SUB];
  __shared__ __align__(16) uint8_t vaux[2 * VAUX_LDS], waux[QT == 2 ? 16 : 2 * 4 * WAUX_LDS];
  constexpr uint32_t SUB3 = TERMS == 3 ? 4 * 1024 : 16;
  __shared__ __align__(16) uint8_t c0[SUB3], c1[SUB3], c2[SUB3], c3[SUB3];
  uint8_t* const ring[4] = {b0, b1, b2, b3};
  uint8_t* const ring3[4] = {c0, c1, c2, c3};
  const int tid = threadIdx.x, l = tid & 63, q = l >> 4, c = l & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  // Workgroups go to the XCDs in turn (linear id mod 8): XCD x takes the
  // x-th eighth of the items, in which the vector tiles of one row group and
  // K chunk are neighbours, so the group's operands come from that XCD's L2.
  const uint32_t per = (a.items + 7u) / 8u;
  const uint32_t item = (blockIdx.x & 7u) * per + (blockIdx.x >> 3);
  if (item >= a.items) return;  // (uniform)
  const uint32_t tt = item % a.ntt, gc = item / a.ntt, chunk = gc % a.ksplit, g = gc / a.ksplit;
  const uint32_t sb0 = chunk * a.kc;
  const uint32_t nsub = a.K / 32;

  uint32_t rt[RT];
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    if constexpr (MODE == 0) rt[r] = min((g * 4u + w) * RT + r, a.rtn - 1);  // (past the last tile: not stored)
    else rt[r] = (r >= 2 ? a.s[1].rt0 : 0u) + g * 8u + w * 2u + (r & 1);
  }
  const u32x4* Ap[RT];  // (uniform)
#pragma unroll
  for (int r = 0; r < RT; ++r) Ap[r] = (const u32x4*)a.w.A + ((size_t)rt[r] * nsub + sb0 * 8u) * 64u;
  const uint8_t* Bg = a.ops + ((size_t)tt * a.nsb + sb0) * PfOps::BYTES;
  const uint8_t* Bl = TERMS == 3 ? a.ops_lo + ((size_t)tt * a.nsb + sb0) * PfOps::LO_BYTES : nullptr;
  const uint32_t nwalk = a.kc * 8u;  // sub-blocks of the walk

  f4 acc[RT][4], C[RT][TERMS == 3 ? 8 : 4];  // (three terms: the even and the odd sub-blocks' sums)
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[r][t] = f4{0.f, 0.f, 0.f, 0.f};

  // sub-block u of the walk: 8 or 12 pieces of 1 KB, each wave its vector
  // tile's two or three; past the end the last one again, so that every turn issues
  // the same number of loads
  auto stage = [&](uint32_t u, uint8_t* buf, uint8_t* buf3) {
    const uint32_t v = min(u, nwalk - 1u);
    const uint8_t* src = Bg + (size_t)(v >> 3) * PfOps::BYTES + w * PfOps::MAIN_T + (v & 7u) * 2048u + l * 16;
    to_lds(src, buf + w * 2048);
    to_lds(src + 1024, buf + w * 2048 + 1024);
    if constexpr (TERMS == 3)
      to_lds(Bl + (size_t)(v >> 3) * PfOps::LO_BYTES + w * 8192u + (v & 7u) * 1024u + l * 16, buf3 + w * 1024);
  };
  // the values super-block j's sums need
  auto stage_aux = [&](uint32_t j) {
    const uint32_t jc = min(j, a.kc - 1u);
    const uint8_t* src = Bg + (size_t)jc * PfOps::BYTES + PfOps::SUMS;
    uint8_t* vb = vaux + (j & 1u) * VAUX_LDS;
    to_lds(src + w * 1024 + l * 16, vb + w * 1024);
    if (w == 0) to_lds(src + 4096 + min(l, 31) * 16, vb + 4096);
    if constexpr (QT != 2) {
      constexpr uint32_t CH = Aux<QT>::CH;
#pragma unroll
      for (uint32_t i = 0; i < (RT * CH + 63) / 64; ++i) {
        const uint32_t ch = min(64u * i + l, RT * CH - 1), r = ch / CH;
        uint32_t t = rt[0];
#pragma unroll
        for (int k = 1; k < RT; ++k) t = r == (uint32_t)k ? rt[k] : t;
        to_lds(a.w.X + ((size_t)t * a.nsb + sb0 + jc) * Aux<QT>::BYTES + (ch - r * CH) * 16u,
               waux + ((j & 1u) * 4u + w) * WAUX_LDS + i * 1024u);
      }
    }
  };

  // weight operands: a ring of four sub-blocks in registers
  u32x4 A[4][RT];
  stage_aux(0);
#pragma unroll
  for (int s = 0; s < 3; ++s) stage(s, ring[s], ring3[s]);
#pragma unroll
  for (int s = 0; s < 4; ++s)
#pragma unroll
    for (int r = 0; r < RT; ++r) A[s][r] = Ap[r][s * 64 + l];
  // (the walk's first waits: known complete here, they cost the loop none)
  wait_vmcnt<0>();

  for (uint32_t j = 0; j < a.kc; ++j) {
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      // Sub-block s of the vectors, requested three turns ago, has arrived
      // once at most what was issued after it is in flight: two turns' TERMS
      // LDS loads and three turns' RT weight loads (the others only make the
      // wait stricter). Every wave has also left sub-block s - 1, whose
      // buffer takes sub-block s + 3.
      wait_vmcnt<2 * TERMS + 3 * RT>();
      lds_barrier();
      if (s == 4) stage_aux(j + 1);
      stage(j * 8u + s + 3, ring[(s + 3) & 3], ring3[(s + 3) & 3]);
      __builtin_amdgcn_sched_barrier(0);
      const uint8_t* base = ring[s & 3] + l * 16;
      const bool first = s % FL == 0;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const h8 bh = *(const h8*)(base + t * 2048), bl = *(const h8*)(base + t * 2048 + 1024);
        auto mul = [&](int r, h8 b, f4 z) {
          return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, A[s & 3][r]), b, z, 0, 0, 0);
        };
        const f4 zero = f4{0.f, 0.f, 0.f, 0.f};
        if constexpr (TERMS == 3) {
          const h8 b3 = *(const h8*)(ring3[s & 3] + t * 1024 + l * 16);
          f4 z[RT];
#pragma unroll
          for (int r = 0; r < RT; ++r) z[r] = mul(r, b3, zero);
#pragma unroll
          for (int r = 0; r < RT; ++r) z[r] = mul(r, bl, z[r]);
#pragma unroll
          for (int r = 0; r < RT; ++r) z[r] = mul(r, bh, z[r]);
#pragma unroll
          for (int r = 0; r < RT; ++r) C[r][4 * (s & 1) + t] = s < 2 ? z[r] : C[r][4 * (s & 1) + t] + z[r];
        } else {
#pragma unroll
          for (int r = 0; r < RT; ++r) C[r][t] = mul(r, bl, first ? zero : C[r][t]);
#pragma unroll
          for (int r = 0; r < RT; ++r) C[r][t] = mul(r, bh, C[r][t]);
        }
      }
      // the next tile's operands are read while one is multiplied
      __builtin_amdgcn_sched_group_barrier(0x100, 2 * TERMS, 0);  // LDS reads
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        __builtin_amdgcn_sched_group_barrier(0x008, TERMS * RT, 0);  // MFMAs
        if (t < 2) __builtin_amdgcn_sched_group_barrier(0x100, TERMS, 0);
      }
      {  // the weight operands four sub-blocks on (past the end: the last again)
        const uint32_t off = min(j * 8u + s + 4, nwalk - 1u) * 64u + l;
#pragma unroll
        for (int r = 0; r < RT; ++r) A[s & 3][r] = Ap[r][off];
      }
      __builtin_amdgcn_sched_barrier(0);
      // these sub-blocks' products times d and 2^-e; the super-block's (or its
      // half's) min term with its last ones
      if (s % FL == FL - 1) {
        const int hf = SG == 2 ? s >> 2 : 0;
        const bool mins = QT == 0 && (s == 7 || (SG == 2 && s == 3));
        const uint8_t* vb = vaux + (j & 1u) * VAUX_LDS;
        const uint8_t* wb = waux + (QT == 2 ? 0u : ((j & 1u) * 4u + w) * WAUX_LDS);
        float fs[4];
        h8 bm[QT == 0 ? 4 : 1];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          fs[t] = *(const float*)(vb + (PfOps::SCALE - PfOps::SUMS) + t * 128 + hf * 64 + c * 4);
          if (mins) bm[t] = *(const h8*)(vb + t * 1024 + l * 16);
        }
#pragma unroll
        for (int r = 0; r < RT; ++r) {
          if constexpr (QT == 2) {
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
              for (int i = 0; i < 4; ++i)
                acc[r][t][i] += fs[t] * (TERMS == 3 ? C[r][t][i] + C[r][TERMS == 3 ? 4 + t : t][i] : C[r][t][i]);
          } else {
            const uint8_t* xr = wb + r * Aux<QT>::BYTES;
            const f4 d = *(const f4*)(xr + 16 * q);
            f4 dm = f4{0.f, 0.f, 0.f, 0.f};
            h8 am = h8{};
            if (mins) {
              dm = *(const f4*)(xr + Aux<0>::DM + 16 * q);
              const h2 mn = *(const h2*)(xr + Aux<0>::MN + 4 * l);
              // slots 8q .. 8q + 7 are sub-blocks 2q and 2q + 1: a half is two lane groups
              if (SG == 1 || (q >> 1) == hf) am = h8{mn.x, mn.x, mn.x, mn.x, mn.y, mn.y, mn.y, mn.y};
            }
#pragma unroll
            for (int t = 0; t < 4; ++t) {
              f4 cm = f4{0.f, 0.f, 0.f, 0.f};
              if (mins) cm = __builtin_amdgcn_mfma_f32_16x16x32_f16(am, bm[t], cm, 0, 0, 0);
#pragma unroll
              for (int i = 0; i < 4; ++i)
                acc[r][t][i] += mins ? fs[t] * (d[i] * C[r][t][i] - dm[i] * cm[i]) : fs[t] * d[i] * C[r][t][i];
            }
          }
        }
      }
    }
  }
  wait_vmcnt<0>();  // no load into this workgroup's LDS outlives it
  lds_barrier();

  // ---- outputs: lane (q, c) holds rows 4q + i of a row tile, vector 64 tt + 16t + c ----
  if constexpr (MODE == 0) {
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      const uint32_t rr = (g * 4u + w) * RT + r;
      if (rr >= a.rtn) continue;  // (uniform over the wave)
      float* Y = a.s[0].Y;
      uint32_t M = a.s[0].rows, rt0 = 0;
#pragma unroll
      for (int i = 1; i < kMaxSeg; ++i)
        if (i < a.n && rr >= a.s[i].rt0) {
          Y = a.s[i].Y;
          M = a.s[i].rows;
          rt0 = a.s[i].rt0;
        }
      const uint32_t row = (rr - rt0) * 16u + 4u * q;
      Y += (size_t)chunk * a.T * M;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const uint32_t v = tt * 64u + 16u * t + c;
        if (v >= a.T) continue;
        float* dst = Y + (size_t)v * M + row;
        if ((M & 3) == 0 && row + 3 < M) {
          *(f4*)dst = acc[r][t];
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (row + i < M) dst[i] = acc[r][t][i];
        }
      }
    }
  } else {
    f4 y[2][4];
    float* mx = (float*)b0;  // [wave][t][16]
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const bool live = tt * 64u + 16u * t + c < a.T;
      float m = 0.f;
#pragma unroll
      for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          y[r][t][i] = live ? g4d::gelu_tanh(acc[r][t][i]) * acc[r + 2][t][i] : 0.f;
          m = fmaxf(m, fabsf(y[r][t][i]));
        }
      m = g4d::xmax32(g4d::xmax16(m));
      if (q == 0) mx[(w * 4 + t) * 16 + c] = m;
    }
    __syncthreads();
    const uint32_t hf = g & 1u, s = hf * 4u + w;  // this wave's sub-block of super-block g / 2
    uint8_t* ob = a.ops_out + ((size_t)tt * (a.s[0].rows / 256u) + (g >> 1)) * PfOps::BYTES;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const float am = fmaxf(fmaxf(mx[t * 16 + c], mx[(4 + t) * 16 + c]),
                             fmaxf(mx[(8 + t) * 16 + c], mx[(12 + t) * 16 + c]));
      int ex = 0;
      (void)frexpf(am, &ex);
      const int k = am > 0.f ? min(max(14 - ex, -120), 120) : 0;
      const float sc = ldexpf(1.0f, k);
      float sum = 0.f;
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        _Float16 hi[4], lo[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float xs = y[r][t][i] * sc;
          sum += xs;
          hi[i] = (_Float16)xs;
          lo[i] = (_Float16)(xs - (float)hi[i]);
        }
        // rows 16r + 4q + i of the sub-block: 8-element group 2r + q / 2, half q % 2 of it
        uint8_t* slot = ob + t * PfOps::MAIN_T + s * 2048u + (c + 16u * (2u * r + (q >> 1))) * 16u + (q & 1) * 8u;
        *(u32x2*)slot = u32x2{pack_h2(hi[0], hi[1]), pack_h2(hi[2], hi[3])};
        *(u32x2*)(slot + 1024) = u32x2{pack_h2(lo[0], lo[1]), pack_h2(lo[2], lo[3])};
      }
      sum = g4d::xsum32(g4d::xsum16(sum)) * 0.015625f;  // the sub-block's sum * 2^-6
      if (q == 0) {
        const _Float16 p0 = (_Float16)sum;
        const float r1 = sum - (float)p0;
        const _Float16 p1 = (_Float16)r1;
        const _Float16 p2 = (_Float16)(r1 - (float)p1);
        *(u32x2*)(ob + PfOps::SUMS + t * 1024 + (c + 16u * (s >> 1)) * 16u + (s & 1u) * 8u) =
            u32x2{pack_h2(p0, p1), pack_h2(p2, (_Float16)0.f)};
        if (w == 0) *(float*)(ob + PfOps::SCALE + t * 128 + hf * 64u + c * 4) = ldexpf(1.0f, -k);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// host
// ---------------------------------------------------------------------------

// Bytes of a launch's unpacked weights: the operands, then the Aux values.
size_t w_operands(uint32_t rtn, uint32_t K) { return (size_t)rtn * (K / 32) * 1024; }
size_t w_bytes(int wtype, uint32_t rtn, uint32_t K) {
  return w_operands(rtn, K) + (size_t)rtn * (K / 256) * aux_bytes(wtype);
}

int check_pf(const char* fn, int wtype, const void* const* weights, const uint32_t* rows, int nseg, uint32_t N,
             const void* ops, uint32_t T, const void* wops, size_t wops_bytes, uint32_t& rtn) {
  G4_REQUIRE(wtype >= 0 && wtype <= 2, "%s: wtype must be 0 (Q4_K), 1 (Q6_K) or 2 (f16)", fn);
  G4_REQUIRE(nseg >= 1 && nseg <= kMaxSeg && weights && rows, "%s: 1..%d segments", fn, kMaxSeg);
  G4_REQUIRE(N >= 256 && N % 256 == 0 && N <= 65536, "%s: N=%u must be a multiple of 256", fn, N);
  G4_REQUIRE(T >= 1 && T <= 65535, "%s: %u vectors outside 1..65535", fn, T);
  G4_REQUIRE(ops && ((uintptr_t)ops & 15) == 0 && wops && ((uintptr_t)wops & 15) == 0,
             "%s: operands must be non-null and 16-byte aligned", fn);
  rtn = 0;
  for (int i = 0; i < nseg; ++i) {
    G4_REQUIRE(weights[i] && rows[i] > 0 && rows[i] <= (1u << 20), "%s: segment %d empty or too tall", fn, i);
    G4_REQUIRE(((uintptr_t)weights[i] & (wtype == 1 ? 3 : 15)) == 0,
               "%s: weights misaligned (Q4_K and f16 16 B, Q6_K 4 B)", fn);
    rtn += ceil_div(rows[i], 16);
  }
  G4_REQUIRE(wops_bytes >= w_bytes(wtype, rtn, N), "%s: weight operand buffer of %zu bytes, %zu needed", fn,
             wops_bytes, w_bytes(wtype, rtn, N));
  return G4_OK;
}

PfArgs pf_args(const void* const* weights, float* const* outputs, const uint32_t* rows, int nseg, uint32_t N,
               const void* ops, uint32_t T, void* wops, uint32_t rtn) {
  PfArgs a{};
  uint32_t rt0 = 0;
  for (int i = 0; i < nseg; ++i) {
    a.s[i] = PfSeg{(const uint8_t*)weights[i], outputs ? outputs[i] : nullptr, rows[i], rt0};
    rt0 += ceil_div(rows[i], 16);
  }
  a.n = nseg;
  a.w = PfWeights{(uint8_t*)wops, (uint8_t*)wops + w_operands(rtn, N)};
  a.rtn = rtn;
  a.K = N;
  a.nsb = N / 256;
  a.ops = (const uint8_t*)ops;
  a.T = T;
  a.ntt = ceil_div(T, 64);
  a.ksplit = 1;
  a.kc = a.nsb;
  return a;
}

int unpack(g4_ctx* ctx, int wtype, const PfArgs& a) {
  const dim3 grid(ceil_div((uint64_t)a.rtn * a.nsb, 4));
  if (wtype == 0) hipLaunchKernelGGL(unpack_kernel<0>, grid, dim3(NT), 0, ctx->stream, a);
  else if (wtype == 1) hipLaunchKernelGGL(unpack_kernel<1>, grid, dim3(NT), 0, ctx->stream, a);
  else hipLaunchKernelGGL(unpack_kernel<2>, grid, dim3(NT), 0, ctx->stream, a);
  G4_LAUNCHED(ctx, "prefill_unpack");
  return G4_OK;
}

template <int RT, int MODE, int SG, int F16_TERMS = 2>
int gemm_qt(g4_ctx* ctx, int wtype, PfArgs a, uint32_t groups) {
  a.groups = groups;
  a.items = groups * a.ksplit * a.ntt;
  const dim3 grid(ceil_div(a.items, 8) * 8);
  if (wtype == 0) {
    if constexpr (RT == 4 && SG == 2) return G4_ERR_UNSUPPORTED;  // (pick_plan)
    else hipLaunchKernelGGL((pf_gemm_kernel<0, RT, MODE, SG>), grid, dim3(NT), 0, ctx->stream, a);
  } else if (wtype == 1) hipLaunchKernelGGL((pf_gemm_kernel<1, RT, MODE, SG>), grid, dim3(NT), 0, ctx->stream, a);
  else hipLaunchKernelGGL((pf_gemm_kernel<2, RT, MODE, SG, F16_TERMS>), grid, dim3(NT), 0, ctx->stream, a);
  G4_LAUNCHED(ctx, "prefill_gemm");
  return G4_OK;
}

// Row tiles per wave (4 or 2) and K split of a launch: the pair with the
// least estimated time, in units of one super-block of a RT = 4 workgroup
// (half as much with RT = 2, a fifth more per tile as the operands read from
// LDS serve half the rows), over rounds of two workgroups per CU, plus the
// split's partial sums (their write and the next launch's read).
struct Plan {
  int rt;
  uint32_t ks;
};
Plan pick_plan(const g4_ctx* ctx, const PfArgs& a, uint32_t max_split, bool two_only) {
  const uint32_t slots = 2u * (uint32_t)(ctx->num_cus > 0 ? ctx->num_cus : 256);
  Plan best{2, 1};
  double bt = 1e30;
  for (int rt = two_only ? 2 : 4; rt >= 2; rt -= 2)
    for (uint32_t ks = 1; ks <= a.nsb && ks <= max_split; ++ks) {
      if (a.nsb % ks) continue;
      const uint32_t items = ceil_div(a.rtn, 4u * rt) * a.ntt * ks, rounds = ceil_div(items, slots);
      const double sb = rt == 4 ? 1.0 : 0.6;
      // a last round that leaves one workgroup per CU runs it about 1.6 times as fast
      const uint32_t rest = items - (rounds - 1) * slots;
      const double eff = rounds - 1 + (rest <= slots / 2 ? 0.62 : 1.0);
      const double t = eff * (a.nsb / ks * sb + 1.0) + (ks > 1 ? ks * (double)a.T * a.rtn * 16.0 * 1e-7 : 0.0);
      if (t < bt) {
        bt = t;
        best = Plan{rt, ks};
      }
    }
  return best;
}

}  // namespace

extern "C" {

int g4_prefillWeightBytes(int wtype, uint32_t rows, uint32_t N, size_t* bytes) {
  G4_REQUIRE(bytes && wtype >= 0 && wtype <= 2 && rows > 0 && rows <= (1u << 22) && N >= 256 && N % 256 == 0 &&
                 N <= 65536,
             "g4_prefillWeightBytes: bad shape");
  *bytes = w_bytes(wtype, ceil_div(rows, 16), N);
  return G4_OK;
}

int g4_prefillOperandBytes(uint32_t N, uint32_t vectors, size_t* bytes) {
  G4_REQUIRE(bytes && N >= 256 && N % 256 == 0 && N <= 65536 && vectors >= 1 && vectors <= 65535,
             "g4_prefillOperandBytes: bad shape");
  *bytes = (size_t)ceil_div(vectors, 64) * (N / 256) * PfOps::BYTES;
  return G4_OK;
}

int g4_prefillOperandLoBytes(uint32_t N, uint32_t vectors, size_t* bytes) {
  G4_REQUIRE(bytes && N >= 256 && N % 256 == 0 && N <= 65536 && vectors >= 1 && vectors <= 65535,
             "g4_prefillOperandLoBytes: bad shape");
  *bytes = (size_t)ceil_div(vectors, 64) * (N / 256) * PfOps::LO_BYTES;
  return G4_OK;
}

int g4_prefillMatmul(g4_ctx* ctx, int wtype, const void* const* weights, float* const* outputs, const uint32_t* rows,
                     int nseg, uint32_t N, const void* ops, int product_ops, uint32_t vectors, void* wops,
                     size_t wops_bytes, uint32_t max_ksplit, uint32_t* ksplit) {
  return g4_prefillMatmulLo(ctx, wtype, weights, outputs, rows, nseg, N, ops, nullptr, product_ops, vectors, wops,
                            wops_bytes, max_ksplit, ksplit);
}

int g4_prefillMatmulLo(g4_ctx* ctx, int wtype, const void* const* weights, float* const* outputs,
                       const uint32_t* rows, int nseg, uint32_t N, const void* ops, const void* ops_lo,
                       int product_ops, uint32_t vectors, void* wops, size_t wops_bytes, uint32_t max_ksplit,
                       uint32_t* ksplit) {
  G4_ENTER(ctx);
  uint32_t rtn;
  int rc = check_pf(__func__, wtype, weights, rows, nseg, N, ops, vectors, wops, wops_bytes, rtn);
  if (rc) return rc;
  G4_REQUIRE(outputs && ksplit && max_ksplit >= 1, "g4_prefillMatmul: null outputs, null ksplit or max_ksplit 0");
  for (int i = 0; i < nseg; ++i)
    G4_REQUIRE(outputs[i] && ((uintptr_t)outputs[i] & 15) == 0, "g4_prefillMatmul: output %d null or misaligned", i);
  G4_REQUIRE(!ops_lo || (wtype == 2 && !product_ops && ((uintptr_t)ops_lo & 15) == 0),
             "g4_prefillMatmul: ops_lo goes with f16 rows, not with product_ops, 16-byte aligned");
  PfArgs a = pf_args(weights, outputs, rows, nseg, N, ops, vectors, wops, rtn);
  rc = unpack(ctx, wtype, a);
  if (rc) return rc;
  a.ops_lo = (const uint8_t*)ops_lo;
  // (Q4_K over a product's operands: with four row tiles the two scale groups'
  // min products spill 289 registers; so do the sums of three terms)
  const Plan p = pick_plan(ctx, a, max_ksplit, (wtype == 0 && product_ops) || ops_lo);
  a.ksplit = p.ks;
  a.kc = a.nsb / p.ks;
  *ksplit = p.ks;
  const uint32_t groups = ceil_div(rtn, 4u * (uint32_t)p.rt);
  if (ops_lo) return gemm_qt<2, 0, 1, 3>(ctx, wtype, a, groups);
  if (product_ops) return p.rt == 4 ? gemm_qt<4, 0, 2>(ctx, wtype, a, groups) : gemm_qt<2, 0, 2>(ctx, wtype, a, groups);
  return p.rt == 4 ? gemm_qt<4, 0, 1>(ctx, wtype, a, groups) : gemm_qt<2, 0, 1>(ctx, wtype, a, groups);
}

int g4_prefillGateUp(g4_ctx* ctx, int wtype, const void* w_gate, const void* w_up, const void* ops, void* product_ops,
                     uint32_t M, uint32_t N, uint32_t vectors, void* wops, size_t wops_bytes) {
  G4_ENTER(ctx);
  const void* weights[2] = {w_gate, w_up};
  const uint32_t rows[2] = {M, M};
  uint32_t rtn;
  int rc = check_pf(__func__, wtype, weights, rows, 2, N, ops, vectors, wops, wops_bytes, rtn);
  if (rc) return rc;
  G4_REQUIRE(M % 256 == 0, "g4_prefillGateUp: M=%u must be a multiple of 256", M);
  G4_REQUIRE(product_ops && ((uintptr_t)product_ops & 15) == 0, "g4_prefillGateUp: product operands null or misaligned");
  PfArgs a = pf_args(weights, nullptr, rows, 2, N, ops, vectors, wops, rtn);
  a.ops_out = (uint8_t*)product_ops;
  rc = unpack(ctx, wtype, a);
  if (rc) return rc;
  return gemm_qt<4, 1, 1>(ctx, wtype, a, M / 128);
}

}  // extern "C"
