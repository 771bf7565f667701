// k_prefill_attn.hip — attention of a whole prompt's rows on the gfx950
// matrix cores: the rows are tokens of one sequence over one page list
// (batched prefill; the reference runs attn_score / softmax / attn_output once
// per prompt token, src/engine.ts:1556-1584).
//
// The ragged step's attention gives every row a workgroup set of its own, so
// each row reads its whole window: at 1900 tokens the same K/V rows up to
// 1900 times, 25-55 us per 64 rows and layer in three launches. Here a
// workgroup takes 8 tokens x the 8 query heads of a KV head and walks their
// common window once:
//  * a wave holds 16 columns (2 tokens x 8 heads) of q in registers as f16 hi
//    and lo operands and their output sums; K and V rows go through LDS in
//    steps of 32 positions, K as stored, V transposed;
//  * scores S[pos][col] = K q with v_mfma_f32_16x16x32_f16, lo apart from hi;
//    the online softmax runs per column; two 16-position score tiles are the
//    32-deep A operand of the PV product as they lie in registers (V's
//    positions are stored in that order), P as f16 hi + lo;
//  * q is scaled by a power of two that brings its column's (and half's)
//    largest element to 2^13 .. 2^14, P (at most 1) by 2^14: hi + lo then hold
//    22 bits of every element down to 2^-16 of the largest, and no f32 q
//    overflows f16. Unscaled, a P below 2^-25 left the product (not the sum
//    it is divided by): one key 14 above 1900 others, whose V is small, cost
//    3e-5 of the result;
//  * sums over steps and over more than 32 dims (64 at head dim 256) are f32
//    additions: a product that adds to a running accumulator does so with about
//    twice an addition's error. Relative error against float64, 100 rows to
//    1900 positions, scores of spread 2: head dim 256 3.5e-7 and 512 3.5e-7,
//    where the ragged step's attention has 5.6e-7 (mq_attn_kernel) and 3.5e-7
//    (attn_kernel); chained products on unscaled pairs had 8e-7 and 7e-7. Cost
//    of both at 1900 rows: head dim 256, window 512 53 -> 55 us, 512 225 -> 237;
//  * head dim 512: two waves share a column tile, each 256 dims; their score
//    halves are added through LDS (same order in both);
//  * a token's V rows are those of its own window only: in the steps at the
//    ends of the workgroup's windows a wave multiplies V once for each of its
//    two tokens, with the rows outside that token's window zeroed (P is 0
//    there, but 0 x Inf is NaN: one non-finite row would reach tokens before
//    it). These steps go first, in a loop of their own: as a branch of one loop
//    they cost it 30 spilled registers.
// A wave's LDS reads take as long as its products (1 KB per two MFMAs), which
// bounds the kernel; a window of few tokens over a long cache is split over
// workgroups (partials merged in split order by merge_kernel).
#include <algorithm>
#include <type_traits>

#include "mm_operand.hpp"

namespace {

using namespace g4mm;

typedef _Float16 h4 __attribute__((ext_vector_type(4)));

constexpr int TOK = 8;     // tokens of a workgroup
constexpr int HEADS = 8;   // query heads per KV head
constexpr uint32_t kMaxSplit = 16;
constexpr float kPScale = 16384.f;  // P's power of two

struct PaArgs {
  const float* q;  // [T][nqh][HD], normed and roped
  const uint16_t* kc;
  const uint16_t* vc;
  const int32_t* page_table;  // [max_pages]
  uint32_t page_size, max_pages, num_pages;
  const uint32_t* lens;  // [T]: row v attends to positions below lens[v]
  uint32_t T, nqh, nkh, cap, window;
  float scale;
  uint32_t nsplit;
  float* ws;   // nsplit > 1: m and l [2][nsplit][T][nqh], then o [nsplit][T][nqh][HD]
  float* out;  // [T][nqh][HD]
};

template <int HD>
struct Shape {
  static constexpr int NH = HD / 256;            // waves per column tile
  static constexpr int NT = 256 * NH;
  static constexpr int STEP = 32;                // (64 at head dim 256: the prefetched rows spill)
  static constexpr int NPT = STEP / 16;          // score tiles of a step
  static constexpr int KS = HD + 8;              // K row stride (halves)
  static constexpr int VS = STEP + 8;            // transposed V row stride (halves)
  static constexpr int NB = STEP / 8;            // 16-byte blocks of a transposed row
  static constexpr int PK = STEP * HD / 8 / NT;  // 16-byte pieces of K per thread and step
  static constexpr int PV = PK / 4;              // 4-position x 8-dim pieces of V
};

// The softmax works in powers of two (scores times log2 e, in one product with
// the scale): P = exp2(fma(score, scale, -max)) rounds its exponent once.
constexpr float kLog2e = 1.44269504f;
__device__ __forceinline__ float exp2_h(float x) { return __builtin_amdgcn_exp2f(x); }

template <int HD>
__global__ __launch_bounds__(Shape<HD>::NT, 2) void pf_attn_kernel(PaArgs a) {
  using S_ = Shape<HD>;
  constexpr int STEP = S_::STEP, NPT = S_::NPT, KS = S_::KS, VS = S_::VS, NB = S_::NB;
  __shared__ __align__(16) _Float16 kt[STEP * KS];
  __shared__ __align__(16) _Float16 vt[HD * VS];
  __shared__ __align__(16) f4 xs[HD == 512 ? 8 * NPT * 64 : 1];  // score halves
  const int tid = threadIdx.x, l = tid & 63, q = l >> 4, c = l & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wc = w & 3, wd = w >> 2;  // column tile, 256-dim half
  const uint32_t kvh = blockIdx.y;
  // the last tiles of a prompt have the longest windows: they start first
  const uint32_t tile = gridDim.x - 1 - blockIdx.x, split = blockIdx.z;
  const uint32_t t0 = tile * TOK;

  // the tokens' windows (uniform loads): the wave's two, their union and common part over the workgroup
  uint32_t lo = 0xffffffffu, hi = 0, wlo[2] = {0, 0}, whi[2] = {0, 0}, ilo = 0, ihi = 0xffffffffu;
#pragma unroll
  for (int i = 0; i < TOK; ++i) {
    const uint32_t L = min(a.lens[min(t0 + i, a.T - 1)], a.cap);
    const uint32_t s = a.window && L > a.window ? L - a.window : 0u;
    lo = min(lo, s);
    hi = max(hi, L);
    ilo = max(ilo, s);
    ihi = min(ihi, L);
    if ((i >> 1) == wc) {
      wlo[i & 1] = s;
      whi[i & 1] = L;
    }
  }
  const uint32_t clo = wlo[c >> 3], chi = whi[c >> 3];  // this column's
  const uint32_t steps = hi > lo ? (hi - lo + STEP - 1) / STEP : 0u;
  const uint32_t per = (steps + a.nsplit - 1) / a.nsplit;
  const uint32_t s0 = min(split * per, steps), s1 = min(s0 + per, steps);
  // Steps e0 .. e1 - 1 lie inside every token's window. The others, at its
  // ends, go first: turn k of the n is step step_of(k).
  const uint32_t n = s1 - s0;
  const uint32_t e0 = min(max((ilo - lo + STEP - 1) / STEP, s0), s1);
  const uint32_t e1 = max(min(ihi > lo ? (ihi - lo) / STEP : 0u, s1), e0);
  const uint32_t ends = n - (e1 - e0);
  auto step_of = [&](uint32_t k) { return k < e0 - s0 ? s0 + k : (k < ends ? e1 + (k - (e0 - s0)) : e0 + (k - ends)); };
  const uint32_t last = hi ? hi - 1 : 0u;  // rows past the window repeat its last position (masked)

  auto row_of = [&](uint32_t pos) -> size_t {
    int32_t pg = a.page_table[pos / a.page_size];
    pg = pg < 0 ? 0 : (pg >= (int32_t)a.num_pages ? (int32_t)a.num_pages - 1 : pg);
    return ((size_t)pg * a.page_size + pos % a.page_size) * a.nkh + kvh;
  };
  u32x4 kp[S_::PK], vp[4 * S_::PV];
  auto load_step = [&](uint32_t st) {
    const uint32_t p0 = lo + st * STEP;
#pragma unroll
    for (int i = 0; i < S_::PK; ++i) {
      const uint32_t pc = (uint32_t)tid + (uint32_t)S_::NT * i, r = pc / (HD / 8), d = pc % (HD / 8) * 8;
      kp[i] = *(const u32x4*)(a.kc + row_of(min(p0 + r, last)) * HD + d);
    }
#pragma unroll
    for (int i = 0; i < S_::PV; ++i) {  // positions 4 (pc / (HD / 8)) .. + 3
      const uint32_t pc = (uint32_t)tid + (uint32_t)S_::NT * i, r = pc / (HD / 8) * 4, d = pc % (HD / 8) * 8;
#pragma unroll
      for (int k = 0; k < 4; ++k) vp[4 * i + k] = *(const u32x4*)(a.vc + row_of(min(p0 + r + k, last)) * HD + d);
    }
  };
  // Transposed V: row d holds the step's positions in the order of the PV
  // operand, index 8q + j of each 32 for position 4q + j (j < 4) and
  // 16 + 4q + j - 4; its 16-byte blocks are xored with d / 8 so that a
  // wave's stores of one position quad (8 dims apart) meet different banks.
  auto store_step = [&]() {
#pragma unroll
    for (int i = 0; i < S_::PK; ++i) {
      const uint32_t pc = (uint32_t)tid + (uint32_t)S_::NT * i, r = pc / (HD / 8), d = pc % (HD / 8) * 8;
      *(u32x4*)(kt + r * KS + d) = kp[i];
    }
#pragma unroll
    for (int i = 0; i < S_::PV; ++i) {
      const uint32_t pc = (uint32_t)tid + (uint32_t)S_::NT * i, k = pc / (HD / 8), o = pc % (HD / 8);
      const uint32_t blk = k / 8 * 4 + k % 4, half = k % 8 / 4;
      _Float16* dst = vt + o * 8 * VS + ((blk ^ (o & (NB - 1))) * 8 + half * 4);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const uint32_t sh = (e & 1) * 16, m = e >> 1;
        const uint32_t x0 = (vp[4 * i][m] >> sh) & 0xffffu, x1 = (vp[4 * i + 1][m] >> sh) & 0xffffu;
        const uint32_t x2 = (vp[4 * i + 2][m] >> sh) & 0xffffu, x3 = (vp[4 * i + 3][m] >> sh) & 0xffffu;
        *(u32x2*)(dst + e * VS) = u32x2{x0 | (x1 << 16), x2 | (x3 << 16)};
      }
    }
  };

  // q of this wave's columns: dims 256 wd + 32 j + 8q .. + 7, times 2^k, hi and lo
  h8 qh[8], ql[8];
  float unscale;  // 2^-k
  {
    const uint32_t tok = min(t0 + 2u * wc + (c >> 3), a.T - 1);
    const float* qg = a.q + ((size_t)tok * a.nqh + kvh * HEADS + (c & 7)) * HD + 256 * wd + 8 * q;
    float x[8][8], am = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float4 x0 = *(const float4*)(qg + 32 * j), x1 = *(const float4*)(qg + 32 * j + 4);
      const float y[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        x[j][e] = y[e];
        am = fmaxf(am, fabsf(y[e]));
      }
    }
    const float up = g4d::f16_pair_scale(g4d::xmax32(g4d::xmax16(am)), unscale);
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float y = x[j][e] * up;
        qh[j][e] = (_Float16)y;
        ql[j][e] = (_Float16)(y - (float)qh[j][e]);
      }
  }
  const float s_scale = (HD == 256 ? a.scale * unscale : a.scale) * kLog2e;

  // V operands of the even and odd dim tiles (positions 4q .. + 3 and 16 + 4q .. + 3; rows 16 dt apart)
  const _Float16* vb[2];
#pragma unroll
  for (int k = 0; k < 2; ++k)
    vb[k] = vt + (256 * wd + c) * VS + ((uint32_t)q ^ ((2u * k + (c >> 3)) & (NB - 1))) * 8;

  f4 O[16];
#pragma unroll
  for (int dt = 0; dt < 16; ++dt) O[dt] = f4{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_run = 0.f;  // of column c

  auto turn = [&](uint32_t k, auto inside) __attribute__((always_inline)) {
    const uint32_t st = step_of(k);
    __syncthreads();  // every wave is done with the previous step's rows
    store_step();
    __syncthreads();
    if (k + 1 < n) load_step(step_of(k + 1));  // (uniform) in flight during this step

    const f4 zero = f4{0.f, 0.f, 0.f, 0.f};
    constexpr int CH = HD == 256 ? 2 : 4;
    f4 S[NPT];
#pragma unroll
    for (int p = 0; p < NPT; ++p) {
      f4 Sl = zero;
      S[p] = zero;
#pragma unroll
      for (int j = 0; j < 8; j += CH) {
        f4 t[CH];
#pragma unroll
        for (int e = 0; e < CH; ++e) {
          const h8 A = *(const h8*)(kt + (16 * p + c) * KS + 256 * wd + 32 * (j + e) + 8 * q);
          t[e] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A, qh[j + e], HD == 256 && e ? t[e - 1] : zero, 0, 0, 0);
          Sl = __builtin_amdgcn_mfma_f32_16x16x32_f16(A, ql[j + e], Sl, 0, 0, 0);
        }
        if constexpr (HD == 256) S[p] += t[1];
        else S[p] += (t[0] + t[1]) + (t[2] + t[3]);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)  // (a non-finite K element: the lo product may cancel the hi one's infinity)
        S[p][i] = fabsf(S[p][i]) < INFINITY ? S[p][i] + Sl[i] : S[p][i];
    }
    if constexpr (HD == 512) {
#pragma unroll
      for (int p = 0; p < NPT; ++p) xs[(w * NPT + p) * 64 + l] = S[p] * unscale;
      __syncthreads();
#pragma unroll
      for (int p = 0; p < NPT; ++p)
        S[p] = xs[(wc * NPT + p) * 64 + l] + xs[((wc + 4) * NPT + p) * 64 + l];
    }
    float mx = -INFINITY;
    const uint32_t pb = lo + st * STEP + 4u * q;
    auto live = [&](int p, int i) {
      const uint32_t pos = pb + 16u * p + i;
      return decltype(inside)::value || (pos >= clo && pos < chi);
    };
#pragma unroll
    for (int p = 0; p < NPT; ++p)
#pragma unroll
      for (int i = 0; i < 4; ++i) mx = fmaxf(mx, live(p, i) ? S[p][i] * s_scale : -INFINITY);
    mx = g4d::xmax32(g4d::xmax16(mx));
    const float m_new = fmaxf(m_run, mx), m_fin = m_new == -INFINITY ? 0.f : m_new;
    const float alpha = exp2_h(m_run - m_fin);  // (nothing live yet: 0, times sums of 0)
    float ps = 0.f;
    h8 ph[NPT / 2], pl[NPT / 2];
#pragma unroll
    for (int p = 0; p < NPT; ++p)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float e = live(p, i) ? exp2_h(fmaf(S[p][i], s_scale, -m_fin)) : 0.f;
        ps += e;
        const float es = e * kPScale;
        const _Float16 h = (_Float16)es;
        ph[p / 2][(p & 1) * 4 + i] = h;
        pl[p / 2][(p & 1) * 4 + i] = (_Float16)(es - (float)h);
      }
    ps = g4d::xsum32(g4d::xsum16(ps));
    l_run = l_run * alpha + ps;
    m_run = m_new;
    if (__ballot(alpha != 1.f)) {  // O's rows here are columns 4q + i
      float ar[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) ar[i] = __shfl(alpha, 4 * q + i, 64);
#pragma unroll
      for (int dt = 0; dt < 16; ++dt)
#pragma unroll
        for (int i = 0; i < 4; ++i) O[dt][i] *= ar[i];
    }
    static_assert(NPT == 2 && NB == 4, "one 32-position operand per step");
    if constexpr (decltype(inside)::value) {
#pragma unroll
      for (int dt = 0; dt < 16; ++dt) {
        const h8 B = *(const h8*)(vb[dt & 1] + dt * 16 * VS);
        const f4 t = __builtin_amdgcn_mfma_f32_16x16x32_f16(pl[0], B, zero, 0, 0, 0);
        O[dt] += __builtin_amdgcn_mfma_f32_16x16x32_f16(ph[0], B, t, 0, 0, 0);
      }
    } else {
      u32x4 keep[2];  // of this lane's eight positions, each token's
      const uint32_t p0 = lo + st * STEP;
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const uint32_t n0 = whi[k] > p0 ? min(whi[k] - p0, 32u) : 0u, n1 = wlo[k] > p0 ? min(wlo[k] - p0, 32u) : 0u;
        const uint32_t live = (uint32_t)(((1ull << n0) - 1) & ~((1ull << n1) - 1)) >> (4 * q);  // (bit = position)
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          const uint32_t two = live >> ((m < 2 ? 0 : 16) + 2 * (m & 1));
          keep[k][m] = (two & 1u) * 0xffffu | (two >> 1 & 1u) * 0xffff0000u;
        }
      }
#pragma unroll
      for (int dt = 0; dt < 16; ++dt) {
        const u32x4 B = *(const u32x4*)(vb[dt & 1] + dt * 16 * VS);
        f4 o[2];  // O's rows 4q + i are of token q / 2
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const h8 Bk = __builtin_bit_cast(h8, B & keep[k]);
          o[k] = __builtin_amdgcn_mfma_f32_16x16x32_f16(pl[0], Bk, zero, 0, 0, 0);
          o[k] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ph[0], Bk, o[k], 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) O[dt][i] += q < 2 ? o[0][i] : o[1][i];
      }
    }
  };
  if (n) load_step(step_of(0));
  for (uint32_t k = 0; k < ends; ++k) turn(k, std::false_type{});
  for (uint32_t k = ends; k < n; ++k) turn(k, std::true_type{});

  // columns 4q + i: token 2 wc + (4q + i) / 8, head (4q + i) % 8
  float inv[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float L = __shfl(l_run, 4 * q + i, 64);
    inv[i] = (a.nsplit > 1 ? 1.f : (L > 0.f ? 1.0f / L : 0.f)) * (1.f / kPScale);
  }
  const uint32_t tok = t0 + 2u * wc + (q >> 1);
  const size_t rows = (size_t)a.T * a.nqh;
  float* o = a.nsplit > 1 ? a.ws + 2 * a.nsplit * rows + split * rows * HD : a.out;
  if (tok < a.T) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const size_t row = (size_t)tok * a.nqh + kvh * HEADS + (4u * q + i) % 8u;
#pragma unroll
      for (int dt = 0; dt < 16; ++dt) o[row * HD + 256 * wd + 16 * dt + c] = O[dt][i] * inv[i];
    }
  }
  const uint32_t ctok = t0 + 2u * wc + (c >> 3);
  if (a.nsplit > 1 && wd == 0 && q == 0 && ctok < a.T) {
    const size_t row = split * rows + (size_t)ctok * a.nqh + kvh * HEADS + (c & 7);
    a.ws[row] = m_run;
    a.ws[a.nsplit * rows + row] = l_run;
  }
}

// out[row] from the row's nsplit partials, in split order: row = (token, head).
template <int HD>
__global__ __launch_bounds__(HD / 4) void merge_kernel(const float* ws, float* out, uint32_t rows, uint32_t nsplit) {
  const uint32_t row = blockIdx.x, d = threadIdx.x * 4;
  float M = -INFINITY;
  for (uint32_t s = 0; s < nsplit; ++s) M = fmaxf(M, ws[(size_t)s * rows + row]);
  float L = 0.f;
  float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
  const float* lw = ws + (size_t)nsplit * rows;
  const float* ow = ws + (size_t)2 * nsplit * rows;
  for (uint32_t s = 0; s < nsplit; ++s) {
    const float m = ws[(size_t)s * rows + row];
    const float wt = m == -INFINITY ? 0.f : exp2_h(m - M);
    const float4 v = *(const float4*)(ow + ((size_t)s * rows + row) * HD + d);
    L += wt * lw[(size_t)s * rows + row];
    o.x += wt * v.x;
    o.y += wt * v.y;
    o.z += wt * v.z;
    o.w += wt * v.w;
  }
  const float inv = L > 0.f ? 1.0f / L : 0.f;
  *(float4*)(out + (size_t)row * HD + d) = make_float4(o.x * inv, o.y * inv, o.z * inv, o.w * inv);
}

// Splits of each tile's window: enough that the launch has a workgroup per
// CU, while a split keeps at least eight steps.
uint32_t pick_split(const g4_ctx* ctx, const g4_paged_attn_fused_params& p) {
  const uint32_t step = 32;
  const uint32_t eff = p.sliding_window ? std::min(p.max_seq_len, p.sliding_window + TOK) : p.max_seq_len;
  const uint32_t steps = ceil_div(eff, step), tiles = ceil_div(p.num_seqs, TOK) * p.num_kv_heads;
  const uint32_t cus = (uint32_t)(ctx && ctx->num_cus > 0 ? ctx->num_cus : 256);
  return std::max(1u, std::min({kMaxSplit, steps / 8, cus / tiles}));
}

size_t split_bytes(const g4_paged_attn_fused_params& p, uint32_t ns) {
  return ns > 1 ? (size_t)ns * p.num_seqs * p.num_q_heads * (p.head_dim + 2) * sizeof(float) : 0;
}

}  // namespace

extern "C" {

int g4_prefillAttn_workspace_size(g4_paged_attn_fused_params p, size_t* bytes) {
  G4_REQUIRE(bytes && p.num_seqs >= 1 && p.num_seqs <= 65535 && p.num_kv_heads >= 1 && p.num_kv_heads <= 64 &&
                 p.num_q_heads == HEADS * p.num_kv_heads && (p.head_dim == 256 || p.head_dim == 512),
             "g4_prefillAttn: 8 query heads per KV head of dim 256 or 512, 1..65535 rows");
  // the most any window can ask for: tiles x splits stays near one workgroup
  // per CU (at most 256 here), a split adds at most TOK rows a tile
  *bytes = (size_t)std::max(256u, ceil_div(p.num_seqs, TOK) * p.num_kv_heads) * TOK * HEADS * (p.head_dim + 2) *
           sizeof(float);
  return G4_OK;
}

int g4_prefillAttn(g4_ctx* ctx, const float* q, const uint16_t* k_pool, const uint16_t* v_pool,
                   const int32_t* page_table, const uint32_t* lens, float* out, g4_paged_attn_fused_params p,
                   float scale, void* workspace, size_t workspace_bytes) {
  G4_ENTER(ctx);
  G4_REQUIRE(q && k_pool && v_pool && page_table && lens && out, "g4_prefillAttn: null buffer");
  size_t need;
  int rc = g4_prefillAttn_workspace_size(p, &need);
  if (rc) return rc;
  G4_REQUIRE((((uintptr_t)q | (uintptr_t)k_pool | (uintptr_t)v_pool | (uintptr_t)out | (uintptr_t)workspace) & 15) == 0,
             "g4_prefillAttn: buffers must be 16-byte aligned");
  G4_REQUIRE(p.page_size > 0 && p.max_pages > 0 && p.num_pages > 0 && p.max_seq_len > 0 &&
                 (uint64_t)p.max_seq_len <= (uint64_t)p.page_size * p.max_pages,
             "g4_prefillAttn: max_seq_len %u exceeds the page table (%u x %u)", p.max_seq_len, p.max_pages,
             p.page_size);
  uint32_t ns = pick_split(ctx, p);
  while (ns > 1 && (!workspace || split_bytes(p, ns) > workspace_bytes)) --ns;
  const PaArgs a{q,      k_pool, v_pool,         page_table,     p.page_size,   p.max_pages,      p.num_pages, lens,
                 p.num_seqs, p.num_q_heads, p.num_kv_heads, p.max_seq_len, p.sliding_window, scale, ns, (float*)workspace, out};
  const dim3 grid(ceil_div(p.num_seqs, TOK), p.num_kv_heads, ns);
  const uint32_t rows = p.num_seqs * p.num_q_heads;
  if (p.head_dim == 256) hipLaunchKernelGGL(pf_attn_kernel<256>, grid, dim3(Shape<256>::NT), 0, ctx->stream, a);
  else hipLaunchKernelGGL(pf_attn_kernel<512>, grid, dim3(Shape<512>::NT), 0, ctx->stream, a);
  G4_LAUNCHED(ctx, "prefill_attn");
  if (ns == 1) return G4_OK;
  if (p.head_dim == 256) hipLaunchKernelGGL(merge_kernel<256>, dim3(rows), dim3(64), 0, ctx->stream, a.ws, out, rows, ns);
  else hipLaunchKernelGGL(merge_kernel<512>, dim3(rows), dim3(128), 0, ctx->stream, a.ws, out, rows, ns);
  G4_LAUNCHED(ctx, "prefill_attn_merge");
  return G4_OK;
}

}  // extern "C"
