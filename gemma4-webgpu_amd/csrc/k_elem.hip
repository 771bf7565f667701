// k_elem.hip — norms, RoPE, activations, KV store, sampling, dequant and the
// seeded synthetic-input generators.
#include <math.h>

#include <algorithm>

#include "g4_internal.hpp"

namespace {

constexpr int NT = 256;

// ---------------------------------------------------------------------------
// norms (shaders/rms_norm.wgsl, fused_norm_add.wgsl,
// per_head_rms_norm_no_weight.wgsl)
// ---------------------------------------------------------------------------

// out = [residual +] in * w / sqrt(mean(in^2) + eps); one workgroup.
template <bool ADD>
__global__ __launch_bounds__(1024) void rms_norm_kernel(const float* in, const uint16_t* w,
                                                        const float* residual, float* out,
                                                        uint32_t n, float eps) {
  __shared__ float red[16];
  float ss = 0.f;
  for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) {
    const float v = in[i];
    ss += v * v;
  }
  ss = g4d::wave_sum(ss);
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nw = blockDim.x >> 6;
  if (lane == 0) red[wv] = ss;
  __syncthreads();
  float tot = 0.f;
  for (int i = 0; i < nw; ++i) tot += red[i];
  const float inv = 1.0f / sqrtf(tot / (float)n + eps);
  for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) {
    float v = in[i] * g4d::f16_bits_to_f32(w[i]) * inv;
    if (ADD) v = residual[i] + v;
    out[i] = v;
  }
}

// Per-head norm (+ weight) then rotate-half RoPE over pairs (i, i+HD/2);
// one workgroup per head (shaders/fused_per_head_norm_rope.wgsl:21-63).
// MODE 0: weightless norm only (v_norm). MODE 1: weighted norm + RoPE.
template <int MODE>
__global__ __launch_bounds__(NT) void head_norm_kernel(float* data, const uint16_t* weight, uint32_t num_heads,
                                                       uint32_t hd, float eps, uint32_t position,
                                                       const uint32_t* position_dev, float theta,
                                                       uint32_t apply_divisor, const uint16_t* rope_freqs) {
  __shared__ float red[4];
  __shared__ float x[512];
  const uint32_t head = blockIdx.x;
  if (head >= num_heads) return;
  float* v = data + (size_t)head * hd;
  float ss = 0.f;
  for (uint32_t i = threadIdx.x; i < hd; i += NT) {
    const float t = v[i];
    x[i] = t;
    ss += t * t;
  }
  ss = g4d::block_sum<4>(ss, red);
  const float inv = 1.0f / sqrtf(ss / (float)hd + eps);
  if (MODE == 0) {
    for (uint32_t i = threadIdx.x; i < hd; i += NT) v[i] = x[i] * inv;
    return;
  }
  for (uint32_t i = threadIdx.x; i < hd; i += NT) x[i] = x[i] * g4d::f16_bits_to_f32(weight[i]) * inv;
  __syncthreads();
  const uint32_t pos = position_dev ? *position_dev : position;
  const uint32_t half = hd / 2;
  for (uint32_t i = threadIdx.x; i < half; i += NT) {
    // f32 frequency and angle exactly as the shader forms them; cos/sin of
    // that f32 angle are evaluated in double and rounded once.
    float f = (float)(1.0 / pow((double)theta, (double)(2u * i) / (double)hd));
    if (apply_divisor) f = f / g4d::f16_bits_to_f32(rope_freqs[i]);
    const float angle = (float)pos * f;
    const float c = (float)cos((double)angle), s = (float)sin((double)angle);
    const float x0 = x[i], x1 = x[i + half];
    v[i] = x0 * c - x1 * s;
    v[i + half] = x0 * s + x1 * c;
  }
}

// ---------------------------------------------------------------------------
// activations (shaders/gelu_mul.wgsl, logit_softcap.wgsl)
// ---------------------------------------------------------------------------

__global__ __launch_bounds__(NT) void gelu_mul_kernel(const float* gate, const float* up, float* out, uint32_t n) {
  const uint32_t i = blockIdx.x * NT + threadIdx.x;
  if (i >= n) return;
  out[i] = g4d::gelu_tanh(gate[i]) * up[i];
}

__global__ void advance_kernel(uint32_t* p, uint32_t delta) {
  if (threadIdx.x == 0) p[0] += delta;
}

__global__ __launch_bounds__(NT) void advance_many_kernel(uint32_t* p, uint32_t n, uint32_t delta) {
  const uint32_t i = blockIdx.x * NT + threadIdx.x;
  if (i < n) p[i] += delta;
}

// Bound by its writes: 32 rows of 262144 words (a batch's logits) are 32 MB.
__global__ __launch_bounds__(NT) void repeat_row_kernel(uint32_t* rows, uint32_t words, uint32_t src, uint32_t first,
                                                        uint32_t count) {
  const uint32_t i = blockIdx.x * NT + threadIdx.x;
  if (i >= words) return;
  const uint32_t x = rows[(size_t)src * words + i];
  for (uint32_t r = 0; r < count; ++r) rows[((size_t)first + r) * words + i] = x;
}

__global__ __launch_bounds__(NT) void softcap_kernel(float* logits, uint32_t n, float cap) {
  const uint32_t i = blockIdx.x * NT + threadIdx.x;
  if (i >= n) return;
  float x = logits[i] / cap;
  x = fminf(fmaxf(x, -15.0f), 15.0f);
  logits[i] = tanhf(x) * cap;
}

// ---------------------------------------------------------------------------
// KV cache store (shaders/kv_cache_store.wgsl:9-17), f16 rows
// ---------------------------------------------------------------------------

__global__ __launch_bounds__(NT) void kv_store_kernel(const float* k_in, const float* v_in, uint16_t* kc,
                                                      uint16_t* vc, uint32_t total, uint32_t position,
                                                      const uint32_t* position_dev, uint32_t max_seq) {
  const uint32_t i = blockIdx.x * NT + threadIdx.x;
  if (i >= total) return;
  const uint32_t pos = position_dev ? *position_dev : position;
  if (pos >= max_seq) return;  // a row past the cache is dropped, never written out of bounds
  const size_t idx = (size_t)pos * total + i;
  kc[idx] = g4d::f32_to_f16_bits(k_in[i]);
  vc[idx] = g4d::f32_to_f16_bits(v_in[i]);
}

// ---------------------------------------------------------------------------
// argmax / topk256 (shaders/argmax.wgsl, topk256.wgsl)
// ---------------------------------------------------------------------------
// The candidate order (g4d::Cand, g4d::better) reproduces the reference's
// per-residue scan and tree merge; see g4_internal.hpp.
using g4d::Cand;
using g4d::better;
using g4d::wave_best;

constexpr int kArgmaxBlocks = 256;

// stage 1: workgroup (b, r) scans a contiguous chunk of row r
__global__ __launch_bounds__(NT) void argmax_partial(const float* logits, uint32_t n, Cand* part) {
  __shared__ Cand sm[4];
  logits += (size_t)blockIdx.y * n;
  part += (size_t)blockIdx.y * gridDim.x;
  const uint32_t chunk = (n + gridDim.x - 1) / gridDim.x;
  const uint32_t lo = blockIdx.x * chunk;
  const uint32_t hi = min(n, lo + chunk);
  Cand c{-1e30f, 0u};
  for (uint32_t i = lo + threadIdx.x; i < hi; i += NT) {
    const Cand d{logits[i], i};
    if (better(d, c)) c = d;
  }
  c = wave_best(c);
  if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = c;
  __syncthreads();
  if (threadIdx.x == 0) {
    Cand b = sm[0];
    for (int k = 1; k < 4; ++k)
      if (better(sm[k], b)) b = sm[k];
    part[blockIdx.x] = b;
  }
}

// stage 2: workgroup r reduces row r's partials; the initial candidate
// (-1e30, 0) mirrors the reference's default result. With `adv` non-null it
// also adds `delta` to adv[r] (the row's position: a captured decode step
// then needs no separate advance launch).
// One wave per row: its lanes issue the loads of 8 candidates each before
// comparing any (one memory round trip per 512 candidates), then the wave
// reduction; no LDS, no barrier.
constexpr int kFinalLoads = 8;
__global__ __launch_bounds__(64) void argmax_final(const Cand* part, int nparts, uint32_t* result, uint32_t* adv,
                                                   uint32_t delta) {
  part += (size_t)blockIdx.x * nparts;
  Cand c{-1e30f, 0u};
  for (int i0 = 0; i0 < nparts; i0 += 64 * kFinalLoads) {
    Cand d[kFinalLoads];
#pragma unroll
    for (int k = 0; k < kFinalLoads; ++k) {
      const int i = i0 + 64 * k + (int)threadIdx.x;
      d[k] = i < nparts ? part[i] : Cand{-1e30f, 0u};
    }
#pragma unroll
    for (int k = 0; k < kFinalLoads; ++k)
      if (better(d[k], c)) c = d[k];
  }
  c = wave_best(c);
  if (threadIdx.x == 0) {
    // a candidate that never beat the -1e30 initial value leaves index 0
    result[blockIdx.x] = (c.v > -1e30f) ? c.i : 0u;
    if (adv) adv[blockIdx.x] += delta;
  }
}

// topk256 (shaders/topk256.wgsl:8-20): for each residue class t = i mod 256
// the first strict maximum of the logits in class t, in index order, starting
// from (-1e30, 0), so NaN and values <= -1e30 are never kept. Two stages:
// slabs of the index range each keep their class maxima, then each class
// takes the best slab candidate under `tk_better` (larger value, then
// smaller index), which equals the in-order strict scan whatever the slab
// order (slabs hold disjoint index ranges and never hold NaN).
// Candidates are laid out [batch][256 classes][nparts], so a class's
// candidates are contiguous for the second stage. The fused LM head
// (k_gemv.hip) writes the same layout from its workgroups' stored rows.
constexpr int kTopkSlabs = 256;
constexpr int kTopkLoads = 8;   // loads a thread issues before comparing any

__device__ __forceinline__ bool tk_better(const Cand& a, const Cand& b) {
  return a.v > b.v || (a.v == b.v && a.i < b.i);
}

// stage 1: workgroup (s, b) scans rows [r0, r1) of 256 logits of batch row b
__global__ __launch_bounds__(NT) void topk_partial(const float* logits, uint32_t n, Cand* part) {
  const uint32_t t = threadIdx.x, ns = gridDim.x;
  logits += (size_t)blockIdx.y * n;
  part += (size_t)blockIdx.y * 256 * ns;
  const uint32_t rows = (n + 255) / 256;
  const uint32_t per = (rows + ns - 1) / ns;
  const uint32_t r0 = blockIdx.x * per, r1 = min(rows, r0 + per);
  Cand c{-1e30f, 0u};
  for (uint32_t rb = r0; rb < r1; rb += kTopkLoads) {
    float v[kTopkLoads];
#pragma unroll
    for (int k = 0; k < kTopkLoads; ++k) {  // clamped, unconditional loads
      const uint32_t i = min((rb + (uint32_t)k) * 256u + t, n - 1);
      v[k] = logits[i];
    }
#pragma unroll
    for (int k = 0; k < kTopkLoads; ++k) {
      const uint32_t i = (rb + (uint32_t)k) * 256u + t;
      if (rb + (uint32_t)k < r1 && i < n && v[k] > c.v) c = Cand{v[k], i};
    }
  }
  part[(size_t)t * ns + blockIdx.x] = c;
}

// stage 2: 16 lanes per class, grid (16, batch); each lane reduces every
// 16th candidate of its class (kTopkLoads loads in flight), then the 16
// lanes combine. result[b][2t] = value, [2t + 1] = index bits.
__global__ __launch_bounds__(NT) void topk_final(const Cand* part, int nparts, float* result) {
  const uint32_t cls = blockIdx.x * (NT / 16) + threadIdx.x / 16, j = threadIdx.x % 16;
  const Cand* p = part + ((size_t)blockIdx.y * 256 + cls) * nparts;
  Cand c{-1e30f, 0u};
  for (int k0 = (int)j; k0 < nparts; k0 += 16 * kTopkLoads) {
    Cand d[kTopkLoads];
#pragma unroll
    for (int k = 0; k < kTopkLoads; ++k) {
      const int i = k0 + 16 * k;
      d[k] = i < nparts ? p[i] : Cand{-1e30f, 0u};
    }
#pragma unroll
    for (int k = 0; k < kTopkLoads; ++k)
      if (tk_better(d[k], c)) c = d[k];
  }
#pragma unroll
  for (int o = 8; o > 0; o >>= 1) {
    const Cand d{__shfl_xor(c.v, o, 16), (uint32_t)__shfl_xor((int)c.i, o, 16)};
    if (tk_better(d, c)) c = d;
  }
  if (j == 0) {
    float* r = result + (size_t)blockIdx.y * 512;
    r[2 * cls] = c.v;
    r[2 * cls + 1] = __uint_as_float(c.i);
  }
}

// ---------------------------------------------------------------------------
// seeded synthetic inputs (counter-based SplitMix64, Box-Muller in f64)
// ---------------------------------------------------------------------------

__device__ __forceinline__ double normal_from(uint64_t w0, uint64_t w1) {
  const double u1 = (double)((w0 >> 11) + 1) * 0x1.0p-53;
  const double u2 = (double)(w1 >> 11) * 0x1.0p-53;
  return sqrt(-2.0 * log(u1)) * cos(6.283185307179586 * u2);
}

__global__ __launch_bounds__(NT) void fill_q4k_kernel(uint8_t* dst, uint64_t nblocks, uint64_t seed) {
  const uint64_t b = (uint64_t)blockIdx.x * NT + threadIdx.x;
  if (b >= nblocks) return;
  uint64_t w[22];
#pragma unroll
  for (int i = 0; i < 22; ++i) w[i] = g4d::splitmix64(seed, 32 * b + (uint64_t)i);
  uint32_t words[36];
  const uint16_t d = g4d::f32_to_f16_bits((float)(fabs(normal_from(w[0], w[1])) * 2e-3));
  const uint16_t dm = g4d::f32_to_f16_bits((float)(fabs(normal_from(w[2], w[3])) * 1e-3));
  words[0] = (uint32_t)d | ((uint32_t)dm << 16);
  words[1] = (uint32_t)w[4];
  words[2] = (uint32_t)(w[4] >> 32);
  words[3] = (uint32_t)w[5];
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    words[4 + 2 * k] = (uint32_t)w[6 + k];
    words[5 + 2 * k] = (uint32_t)(w[6 + k] >> 32);
  }
  uint4* o = (uint4*)(dst + b * 144);
#pragma unroll
  for (int k = 0; k < 9; ++k) o[k] = make_uint4(words[4 * k], words[4 * k + 1], words[4 * k + 2], words[4 * k + 3]);
}

// Q5_K blocks (176 B): d ~ |N(0, 2e-3)|, dmin ~ |N(0, 1e-3)| as f16, then
// 12 scale/min bytes, 32 high-bit bytes and 128 nibble bytes uniform.
__global__ __launch_bounds__(NT) void fill_q5k_kernel(uint8_t* dst, uint64_t nblocks, uint64_t seed) {
  const uint64_t b = (uint64_t)blockIdx.x * NT + threadIdx.x;
  if (b >= nblocks) return;
  uint64_t w[26];
#pragma unroll
  for (int i = 0; i < 26; ++i) w[i] = g4d::splitmix64(seed, 32 * b + (uint64_t)i);
  uint32_t words[44];
  const uint16_t d = g4d::f32_to_f16_bits((float)(fabs(normal_from(w[0], w[1])) * 2e-3));
  const uint16_t dm = g4d::f32_to_f16_bits((float)(fabs(normal_from(w[2], w[3])) * 1e-3));
  words[0] = (uint32_t)d | ((uint32_t)dm << 16);
  words[1] = (uint32_t)w[4];
  words[2] = (uint32_t)(w[4] >> 32);
  words[3] = (uint32_t)w[5];
#pragma unroll
  for (int k = 0; k < 20; ++k) {
    words[4 + 2 * k] = (uint32_t)w[6 + k];
    words[5 + 2 * k] = (uint32_t)(w[6 + k] >> 32);
  }
  uint4* o = (uint4*)(dst + b * 176);
#pragma unroll
  for (int k = 0; k < 11; ++k) o[k] = make_uint4(words[4 * k], words[4 * k + 1], words[4 * k + 2], words[4 * k + 3]);
}

__global__ __launch_bounds__(NT) void fill_q6k_kernel(uint8_t* dst, uint64_t nblocks, uint64_t seed) {
  const uint64_t b = (uint64_t)blockIdx.x * NT + threadIdx.x;
  if (b >= nblocks) return;
  uint8_t* o = dst + b * 210;  // 2-byte aligned
  uint16_t* o16 = (uint16_t*)o;
  for (int i = 0; i < 24; ++i) {
    const uint64_t w = g4d::splitmix64(seed, 32 * b + (uint64_t)i);
#pragma unroll
    for (int k = 0; k < 4; ++k) o16[4 * i + k] = (uint16_t)(w >> (16 * k));
  }
  for (int i = 0; i < 2; ++i) {
    const uint64_t w = g4d::splitmix64(seed, 32 * b + 24 + (uint64_t)i);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int lo = (int)((w >> (16 * k)) & 63u) - 32;
      const int hi = (int)((w >> (16 * k + 8)) & 63u) - 32;
      o16[96 + 4 * i + k] = (uint16_t)((uint8_t)(int8_t)lo | ((uint16_t)(uint8_t)(int8_t)hi << 8));
    }
  }
  const uint64_t w26 = g4d::splitmix64(seed, 32 * b + 26), w27 = g4d::splitmix64(seed, 32 * b + 27);
  o16[104] = g4d::f32_to_f16_bits((float)(fabs(normal_from(w26, w27)) * 2e-3));
}

__global__ __launch_bounds__(NT) void fill_normal_kernel(float* dst32, uint16_t* dst16, uint64_t n, uint64_t seed,
                                                         float mean, float std) {
  const uint64_t i = (uint64_t)blockIdx.x * NT + threadIdx.x;
  if (i >= n) return;
  const float v = (float)((double)mean + (double)std * normal_from(g4d::splitmix64(seed, 2 * i),
                                                                   g4d::splitmix64(seed, 2 * i + 1)));
  if (dst32) dst32[i] = v;
  else dst16[i] = g4d::f32_to_f16_bits(v);
}

// ---------------------------------------------------------------------------
// streaming-read probe (measurement export g4_streamRead): one pass over a
// buffer with 16-byte loads, four in flight per thread, under one cache
// policy; each workgroup writes the xor of what it read, so no load is dead.
// ---------------------------------------------------------------------------
typedef uint32_t sr_u4 __attribute__((ext_vector_type(4)));

template <int POL>
__global__ __launch_bounds__(NT) void stream_read_kernel(const uint8_t* src, uint32_t n16, uint32_t* sink) {
  __shared__ uint32_t red[NT / 64];
  const __amdgpu_buffer_rsrc_t rs =
      __builtin_amdgcn_make_buffer_rsrc((void*)src, (short)0, (int)(n16 * 16u), 0x00020000);
  const uint32_t stride = gridDim.x * NT;
  uint32_t acc = 0;
  uint32_t i = blockIdx.x * NT + threadIdx.x;
  for (; i + 3 * stride < n16; i += 4 * stride) {
    sr_u4 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = __builtin_amdgcn_raw_buffer_load_b128(rs, (i + u * stride) * 16u, 0, POL);
#pragma unroll
    for (int u = 0; u < 4; ++u) acc ^= v[u][0] ^ v[u][1] ^ v[u][2] ^ v[u][3];
  }
  for (; i < n16; i += stride) {
    const sr_u4 v = __builtin_amdgcn_raw_buffer_load_b128(rs, i * 16u, 0, POL);
    acc ^= v[0] ^ v[1] ^ v[2] ^ v[3];
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) acc ^= __shfl_xor(acc, o, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t a = 0;
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) a ^= red[w];
    sink[blockIdx.x] = a;
  }
}

}  // namespace

extern "C" {

int g4_rmsNorm(g4_ctx* ctx, const float* input, const uint16_t* weight, float* output, g4_rms_norm_params p) {
  G4_ENTER(ctx);
  G4_REQUIRE(input && weight && output, "g4_rmsNorm: null buffer");
  G4_REQUIRE(p.hidden_size > 0, "g4_rmsNorm: hidden_size 0");
  hipLaunchKernelGGL((rms_norm_kernel<false>), dim3(1), dim3(512), 0, ctx->stream, input, weight, nullptr, output,
                     p.hidden_size, p.eps);
  G4_LAUNCHED(ctx, "rms_norm");
  return G4_OK;
}

int g4_fusedNormAdd(g4_ctx* ctx, const float* input, const uint16_t* weight, const float* residual, float* output,
                    g4_norm_add_params p) {
  G4_ENTER(ctx);
  G4_REQUIRE(input && weight && residual && output, "g4_fusedNormAdd: null buffer");
  G4_REQUIRE(p.size > 0, "g4_fusedNormAdd: size 0");
  hipLaunchKernelGGL((rms_norm_kernel<true>), dim3(1), dim3(512), 0, ctx->stream, input, weight, residual, output,
                     p.size, p.eps);
  G4_LAUNCHED(ctx, "fused_norm_add");
  return G4_OK;
}

int g4_perHeadRmsNormNoWeight(g4_ctx* ctx, float* data, g4_per_head_norm_params p) {
  G4_ENTER(ctx);
  G4_REQUIRE(data, "g4_perHeadRmsNormNoWeight: null buffer");
  G4_REQUIRE(p.num_heads > 0 && p.head_dim > 0 && p.head_dim <= 512,
             "g4_perHeadRmsNormNoWeight: head_dim %u outside (0, 512]", p.head_dim);
  hipLaunchKernelGGL((head_norm_kernel<0>), dim3(p.num_heads), dim3(NT), 0, ctx->stream, data, nullptr, p.num_heads,
                     p.head_dim, p.eps, 0u, nullptr, 0.f, 0u, nullptr);
  G4_LAUNCHED(ctx, "per_head_rms_norm_no_weight");
  return G4_OK;
}

static int norm_rope(g4_ctx* ctx, float* data, const uint16_t* weight, g4_norm_rope_params p,
                     const uint16_t* rope_freqs, const uint32_t* position_dev) {
  G4_REQUIRE(data && weight, "g4_fusedPerHeadNormRope: null buffer");
  G4_REQUIRE(!p.apply_divisor || rope_freqs, "g4_fusedPerHeadNormRope: apply_divisor needs rope_freqs");
  G4_REQUIRE(p.num_heads > 0 && p.head_dim >= 2 && p.head_dim <= 512 && p.head_dim % 2 == 0,
             "g4_fusedPerHeadNormRope: head_dim %u must be even and <= 512", p.head_dim);
  hipLaunchKernelGGL((head_norm_kernel<1>), dim3(p.num_heads), dim3(NT), 0, ctx->stream, data, weight, p.num_heads,
                     p.head_dim, p.eps, p.position, position_dev, p.theta, p.apply_divisor, rope_freqs);
  G4_LAUNCHED(ctx, "fused_per_head_norm_rope");
  return G4_OK;
}

int g4_fusedPerHeadNormRope(g4_ctx* ctx, float* data, const uint16_t* weight, g4_norm_rope_params p,
                            const uint16_t* rope_freqs) {
  G4_ENTER(ctx);
  return norm_rope(ctx, data, weight, p, rope_freqs, nullptr);
}

int g4_fusedPerHeadNormRope_dev(g4_ctx* ctx, float* data, const uint16_t* weight, g4_norm_rope_params p,
                                const uint16_t* rope_freqs, const uint32_t* position_dev) {
  G4_ENTER(ctx);
  G4_REQUIRE(position_dev, "g4_fusedPerHeadNormRope_dev: null position");
  return norm_rope(ctx, data, weight, p, rope_freqs, position_dev);
}

int g4_geluMul(g4_ctx* ctx, const float* gate, const float* up, float* output, uint32_t size) {
  G4_ENTER(ctx);
  G4_REQUIRE(gate && up && output, "g4_geluMul: null buffer");
  if (!size) return G4_OK;
  hipLaunchKernelGGL(gelu_mul_kernel, dim3(ceil_div(size, NT)), dim3(NT), 0, ctx->stream, gate, up, output, size);
  G4_LAUNCHED(ctx, "gelu_mul");
  return G4_OK;
}

// shaders/embedding_lookup.wgsl:9-13: one thread per hidden element; the row is
// token * H, scaled by sqrt(H) in f32. The f16 row is read 8 halves (16 B) per
// thread when H is a multiple of 8 and the table 16-byte aligned, else one.
// blockIdx.y = output row: token_dev[y] (or `token` for the one-row host form).
__global__ __launch_bounds__(NT) void embedding_lookup_kernel(const uint16_t* __restrict__ emb, uint32_t rows,
                                                              float* __restrict__ out, uint32_t H, uint32_t token,
                                                              const uint32_t* __restrict__ token_dev, int vec8) {
  const uint32_t tok = token_dev ? token_dev[blockIdx.y] : token;
  out += (size_t)blockIdx.y * H;
  const float scale = sqrtf(static_cast<float>(H));
  const uint32_t t = blockIdx.x * NT + threadIdx.x;
  if (vec8) {
    const uint32_t i = t * 8;
    if (i >= H) return;
    float v[8];
    if (tok < rows) {
      const uint4 w = *reinterpret_cast<const uint4*>(emb + static_cast<size_t>(tok) * H + i);
      const uint32_t u[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v[2 * j] = g4d::f16_bits_to_f32(u[j] & 0xffffu) * scale;
        v[2 * j + 1] = g4d::f16_bits_to_f32(u[j] >> 16) * scale;
      }
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = 0.f;
    }
    *reinterpret_cast<float4*>(out + i) = make_float4(v[0], v[1], v[2], v[3]);
    *reinterpret_cast<float4*>(out + i + 4) = make_float4(v[4], v[5], v[6], v[7]);
  } else {
    if (t >= H) return;
    out[t] = tok < rows ? g4d::f16_bits_to_f32(emb[static_cast<size_t>(tok) * H + t]) * scale : 0.f;
  }
}

static int embedding_lookup(g4_ctx* ctx, const uint16_t* emb, uint32_t rows, float* out, g4_embedding_params p,
                            const uint32_t* token_dev, uint32_t count = 1) {
  G4_REQUIRE(emb && out, "g4_embeddingLookup: null buffer");
  if (!p.hidden_size || !count) return G4_OK;
  const int vec8 = p.hidden_size % 8 == 0 && reinterpret_cast<uintptr_t>(emb) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(out) % 16 == 0;
  const uint32_t threads = vec8 ? p.hidden_size / 8 : p.hidden_size;
  hipLaunchKernelGGL(embedding_lookup_kernel, dim3(ceil_div(threads, NT), count), dim3(NT), 0, ctx->stream, emb, rows,
                     out, p.hidden_size, p.token_id, token_dev, vec8);
  G4_LAUNCHED(ctx, "embedding_lookup");
  return G4_OK;
}

int g4_embeddingLookup(g4_ctx* ctx, const uint16_t* embedding, uint32_t num_rows, float* output,
                       g4_embedding_params p) {
  G4_ENTER(ctx);
  G4_REQUIRE(p.token_id < num_rows, "g4_embeddingLookup: token_id %u >= num_rows %u", p.token_id, num_rows);
  return embedding_lookup(ctx, embedding, num_rows, output, p, nullptr);
}

int g4_embeddingLookup_dev(g4_ctx* ctx, const uint16_t* embedding, uint32_t num_rows, float* output,
                           g4_embedding_params p, const uint32_t* token_dev) {
  G4_ENTER(ctx);
  G4_REQUIRE(token_dev, "g4_embeddingLookup_dev: null token");
  return embedding_lookup(ctx, embedding, num_rows, output, p, token_dev);
}

int g4_embeddingLookupBatch(g4_ctx* ctx, const uint16_t* embedding, uint32_t num_rows, float* output,
                            uint32_t hidden_size, const uint32_t* tokens_dev, uint32_t count) {
  G4_ENTER(ctx);
  G4_REQUIRE(tokens_dev, "g4_embeddingLookupBatch: null tokens");
  G4_REQUIRE(count <= 65535, "g4_embeddingLookupBatch: %u rows > 65535", count);
  return embedding_lookup(ctx, embedding, num_rows, output, g4_embedding_params{hidden_size, 0u}, tokens_dev, count);
}

int g4_repeatRow(g4_ctx* ctx, void* rows, uint32_t words, uint32_t src, uint32_t first, uint32_t count) {
  G4_ENTER(ctx);
  G4_REQUIRE(rows && ((uintptr_t)rows & 3) == 0, "g4_repeatRow: null or misaligned buffer");
  G4_REQUIRE((src < first || src - first >= count) && (uint64_t)first + count <= UINT32_MAX,
             "g4_repeatRow: row %u is one of the %u from %u", src, count, first);
  if (!words || !count) return G4_OK;
  hipLaunchKernelGGL(repeat_row_kernel, dim3(ceil_div(words, NT)), dim3(NT), 0, ctx->stream, (uint32_t*)rows, words,
                     src, first, count);
  G4_LAUNCHED(ctx, "repeat_row");
  return G4_OK;
}

int g4_logitSoftcap(g4_ctx* ctx, float* logits, g4_softcap_params p) {
  G4_ENTER(ctx);
  G4_REQUIRE(logits, "g4_logitSoftcap: null buffer");
  G4_REQUIRE(p.cap != 0.f, "g4_logitSoftcap: cap must be non-zero");
  if (!p.size) return G4_OK;
  hipLaunchKernelGGL(softcap_kernel, dim3(ceil_div(p.size, NT)), dim3(NT), 0, ctx->stream, logits, p.size, p.cap);
  G4_LAUNCHED(ctx, "logit_softcap");
  return G4_OK;
}

static int kv_store(g4_ctx* ctx, const float* k_in, const float* v_in, uint16_t* kc, uint16_t* vc,
                    g4_kv_store_params p, const uint32_t* position_dev) {
  G4_REQUIRE(k_in && v_in && kc && vc, "g4_kvCacheStore: null buffer");
  G4_REQUIRE(position_dev || p.position < p.max_seq_len, "g4_kvCacheStore: position %u >= max_seq_len %u",
             p.position, p.max_seq_len);
  const uint32_t total = p.num_kv_heads * p.head_dim;
  if (!total) return G4_OK;
  hipLaunchKernelGGL(kv_store_kernel, dim3(ceil_div(total, NT)), dim3(NT), 0, ctx->stream, k_in, v_in, kc, vc, total,
                     p.position, position_dev, p.max_seq_len);
  G4_LAUNCHED(ctx, "kv_cache_store");
  return G4_OK;
}

int g4_kvCacheStore(g4_ctx* ctx, const float* k_in, const float* v_in, uint16_t* k_cache, uint16_t* v_cache,
                    g4_kv_store_params p) {
  G4_ENTER(ctx);
  return kv_store(ctx, k_in, v_in, k_cache, v_cache, p, nullptr);
}

int g4_kvCacheStore_dev(g4_ctx* ctx, const float* k_in, const float* v_in, uint16_t* k_cache, uint16_t* v_cache,
                        g4_kv_store_params p, const uint32_t* position_dev) {
  G4_ENTER(ctx);
  G4_REQUIRE(position_dev, "g4_kvCacheStore_dev: null position");
  return kv_store(ctx, k_in, v_in, k_cache, v_cache, p, position_dev);
}

int g4_advancePosition(g4_ctx* ctx, uint32_t* position_dev, uint32_t delta) {
  G4_ENTER(ctx);
  G4_REQUIRE(position_dev, "g4_advancePosition: null position");
  hipLaunchKernelGGL(advance_kernel, dim3(1), dim3(64), 0, ctx->stream, position_dev, delta);
  G4_LAUNCHED(ctx, "advance_position");
  return G4_OK;
}

int g4_advanceSeqLens(g4_ctx* ctx, uint32_t* seq_lens, uint32_t num_seqs, uint32_t delta) {
  G4_ENTER(ctx);
  G4_REQUIRE(seq_lens, "g4_advanceSeqLens: null buffer");
  if (!num_seqs) return G4_OK;
  hipLaunchKernelGGL(advance_many_kernel, dim3(ceil_div(num_seqs, NT)), dim3(NT), 0, ctx->stream, seq_lens, num_seqs,
                     delta);
  G4_LAUNCHED(ctx, "advance_seq_lens");
  return G4_OK;
}

namespace {
int argmax_launch(g4_ctx* ctx, const char* fn, const float* logits, uint32_t* result, uint32_t size,
                  uint32_t batch, uint32_t* adv, uint32_t delta) {
  G4_REQUIRE(logits && result, "%s: null buffer", fn);
  G4_REQUIRE(batch >= 1 && batch <= 1024, "%s: batch %u not in 1..1024", fn, batch);
  // about 4096 workgroups in all, at most kArgmaxBlocks per row
  const unsigned want = ceil_div(size, 1024), cap = std::max(1u, 4096u / batch);
  const int nb = want == 0 ? 1 : (int)std::min({want, (unsigned)kArgmaxBlocks, cap});
  void* scratch = nullptr;
  int rc = g4_internal_scratch(ctx, (size_t)batch * nb * sizeof(Cand), &scratch);
  if (rc) return rc;
  hipLaunchKernelGGL(argmax_partial, dim3(nb, batch), dim3(NT), 0, ctx->stream, logits, size, (Cand*)scratch);
  G4_LAUNCHED(ctx, "argmax_partial");
  return g4_internal_argmax_final(ctx, scratch, nb, batch, result, adv, delta);
}
}  // namespace

int g4_argmaxBatch(g4_ctx* ctx, const float* logits, uint32_t* result, uint32_t size, uint32_t batch) {
  G4_ENTER(ctx);
  return argmax_launch(ctx, __func__, logits, result, size, batch, nullptr, 0);
}

int g4_argmaxAdvance(g4_ctx* ctx, const float* logits, uint32_t* result, uint32_t size, uint32_t batch,
                     uint32_t* positions, uint32_t delta) {
  G4_ENTER(ctx);
  G4_REQUIRE(positions, "g4_argmaxAdvance: null positions");
  return argmax_launch(ctx, __func__, logits, result, size, batch, positions, delta);
}

int g4_argmax(g4_ctx* ctx, const float* logits, uint32_t* result, uint32_t size) {
  return g4_argmaxBatch(ctx, logits, result, size, 1);
}

int g4_topk256Batch(g4_ctx* ctx, const float* logits, float* result, uint32_t size, uint32_t batch) {
  G4_ENTER(ctx);
  G4_REQUIRE(logits && result, "g4_topk256: null buffer");
  G4_REQUIRE(batch >= 1 && batch <= 1024, "g4_topk256Batch: batch %u not in 1..1024", batch);
  G4_REQUIRE(size > 0, "g4_topk256: empty logits");
  const uint32_t rows = (size + 255) / 256;
  const unsigned want = ceil_div(rows, 4), cap = std::max(1u, 1024u / batch);
  const int ns = (int)std::max(1u, std::min({want, (unsigned)kTopkSlabs, cap}));
  void* scratch = nullptr;
  int rc = g4_internal_scratch(ctx, (size_t)batch * ns * 256 * sizeof(Cand), &scratch);
  if (rc) return rc;
  hipLaunchKernelGGL(topk_partial, dim3(ns, batch), dim3(NT), 0, ctx->stream, logits, size, (Cand*)scratch);
  G4_LAUNCHED(ctx, "topk_partial");
  return g4_internal_topk_final(ctx, scratch, ns, batch, result);
}


int g4_topk256(g4_ctx* ctx, const float* logits, float* result, uint32_t size) {
  return g4_topk256Batch(ctx, logits, result, size, 1);
}

int g4_fill_q4k(g4_ctx* ctx, void* dst, uint64_t nblocks, uint64_t seed) {
  G4_ENTER(ctx);
  G4_REQUIRE(dst, "g4_fill_q4k: null buffer");
  G4_REQUIRE(((uintptr_t)dst & 15) == 0, "g4_fill_q4k: destination must be 16-byte aligned");
  if (!nblocks) return G4_OK;
  hipLaunchKernelGGL(fill_q4k_kernel, dim3(ceil_div(nblocks, NT)), dim3(NT), 0, ctx->stream, (uint8_t*)dst, nblocks,
                     seed);
  G4_LAUNCHED(ctx, "fill_q4k");
  return G4_OK;
}

int g4_fill_q5k(g4_ctx* ctx, void* dst, uint64_t nblocks, uint64_t seed) {
  G4_ENTER(ctx);
  G4_REQUIRE(dst, "g4_fill_q5k: null buffer");
  G4_REQUIRE(((uintptr_t)dst & 15) == 0, "g4_fill_q5k: destination must be 16-byte aligned");
  if (!nblocks) return G4_OK;
  hipLaunchKernelGGL(fill_q5k_kernel, dim3(ceil_div(nblocks, NT)), dim3(NT), 0, ctx->stream, (uint8_t*)dst, nblocks,
                     seed);
  G4_LAUNCHED(ctx, "fill_q5k");
  return G4_OK;
}

int g4_fill_q6k(g4_ctx* ctx, void* dst, uint64_t nblocks, uint64_t seed) {
  G4_ENTER(ctx);
  G4_REQUIRE(dst, "g4_fill_q6k: null buffer");
  G4_REQUIRE(((uintptr_t)dst & 1) == 0, "g4_fill_q6k: destination must be 2-byte aligned");
  if (!nblocks) return G4_OK;
  hipLaunchKernelGGL(fill_q6k_kernel, dim3(ceil_div(nblocks, NT)), dim3(NT), 0, ctx->stream, (uint8_t*)dst, nblocks,
                     seed);
  G4_LAUNCHED(ctx, "fill_q6k");
  return G4_OK;
}

int g4_fill_normal_f32(g4_ctx* ctx, float* dst, uint64_t n, uint64_t seed, float mean, float std) {
  G4_ENTER(ctx);
  G4_REQUIRE(dst, "g4_fill_normal_f32: null buffer");
  if (!n) return G4_OK;
  hipLaunchKernelGGL(fill_normal_kernel, dim3(ceil_div(n, NT)), dim3(NT), 0, ctx->stream, dst, (uint16_t*)nullptr, n,
                     seed, mean, std);
  G4_LAUNCHED(ctx, "fill_normal_f32");
  return G4_OK;
}

int g4_streamRead(g4_ctx* ctx, const void* src, uint64_t bytes, int policy, uint32_t nwgs, uint32_t* sink) {
  G4_ENTER(ctx);
  G4_REQUIRE(src && sink, "g4_streamRead: null buffer");
  G4_REQUIRE(((uintptr_t)src & 15) == 0 && bytes % 16 == 0 && bytes > 0 && bytes < (1ull << 32),
             "g4_streamRead: src 16-byte aligned, bytes a multiple of 16 below 4 GiB");
  G4_REQUIRE(nwgs >= 1 && nwgs <= 65535, "g4_streamRead: 1..65535 workgroups");
  G4_REQUIRE(policy >= 0 && policy <= 2, "g4_streamRead: policy 0 (plain), 1 (non-temporal) or 2 (device scope)");
  const uint32_t n16 = (uint32_t)(bytes / 16);
  if (policy == 0)
    hipLaunchKernelGGL(stream_read_kernel<0>, dim3(nwgs), dim3(NT), 0, ctx->stream, (const uint8_t*)src, n16, sink);
  else if (policy == 1)
    hipLaunchKernelGGL(stream_read_kernel<2>, dim3(nwgs), dim3(NT), 0, ctx->stream, (const uint8_t*)src, n16, sink);
  else
    hipLaunchKernelGGL(stream_read_kernel<16>, dim3(nwgs), dim3(NT), 0, ctx->stream, (const uint8_t*)src, n16, sink);
  G4_LAUNCHED(ctx, "stream_read");
  return G4_OK;
}

int g4_fill_normal_f16(g4_ctx* ctx, uint16_t* dst, uint64_t n, uint64_t seed, float mean, float std) {
  G4_ENTER(ctx);
  G4_REQUIRE(dst, "g4_fill_normal_f16: null buffer");
  if (!n) return G4_OK;
  hipLaunchKernelGGL(fill_normal_kernel, dim3(ceil_div(n, NT)), dim3(NT), 0, ctx->stream, (float*)nullptr, dst, n,
                     seed, mean, std);
  G4_LAUNCHED(ctx, "fill_normal_f16");
  return G4_OK;
}

}  // extern "C"

int g4_internal_topk_final(g4_ctx* ctx, const void* parts, int nparts, uint32_t batch, float* result) {
  hipLaunchKernelGGL(topk_final, dim3(256 / (NT / 16), batch), dim3(NT), 0, ctx->stream, (const Cand*)parts, nparts,
                     result);
  G4_LAUNCHED(ctx, "topk_final");
  return G4_OK;
}

int g4_internal_argmax_final(g4_ctx* ctx, const void* parts, int nparts, uint32_t batch, uint32_t* result,
                             uint32_t* adv, uint32_t delta) {
  hipLaunchKernelGGL(argmax_final, dim3(batch), dim3(64), 0, ctx->stream, (const Cand*)parts, nparts, result, adv,
                     delta);
  G4_LAUNCHED(ctx, "argmax_final");
  return G4_OK;
}
