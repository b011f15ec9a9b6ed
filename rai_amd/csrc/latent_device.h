// The rows of a single-row step's Linears behind a norm, wave by wave (latent_decode.hip, and beside a mixer: delta.hip).
#pragma once
#include "gemm.h"
#include "latent.h"

namespace rai {

typedef __attribute__((ext_vector_type(2))) __bf16 ld_bf16x2;
typedef __attribute__((ext_vector_type(4))) uint32_t ld_u32x4;
typedef __attribute__((ext_vector_type(4))) float ld_f32x4;

__device__ __forceinline__ float ld_dot8(ld_u32x4 a, ld_u32x4 b, float c) {
  // elements named one by one: see dot2_bf16 in gemm.hip
  auto dot2 = [](uint32_t x, uint32_t y, float z) {
    ld_bf16x2 p, q;
    __builtin_memcpy(&p, &x, 4);
    __builtin_memcpy(&q, &y, 4);
    return __builtin_amdgcn_fdot2_f32_bf16(p, q, z, false);
  };
  c = dot2(a.x, b.x, c);
  c = dot2(a.y, b.y, c);
  c = dot2(a.z, b.z, c);
  return dot2(a.w, b.w, c);
}
__device__ __forceinline__ float lo_f32(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float hi_f32(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
__device__ __forceinline__ float gated(int act, float g, float u) { return act_eval(act, g) * u; }
__device__ __forceinline__ float gated(const LatentInArgs &a, float g, float u) {
  return a.act == kActClampedGlu ? glu_clamped_bf16_out(g, u, a.act_limit, a.act_alpha) : gated(a.act, g, u);
}

// R rows of W in flight, rows n .. n + R - 1 clamped to n_last.  Every lane asks for something, those beyond K for the row's start
// (a load under a mask is waited for where the mask ends); piece() is what to multiply.
template <int KC, int R> struct RowSet {
  ld_u32x4 w[R][KC];
  __device__ __forceinline__ void load(const uint16_t *W, int64_t ldw, int n, int n_last, int K, int lane) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const uint16_t *p = W + (int64_t)(n + r < n_last ? n + r : n_last) * ldw;
#pragma unroll
      for (int u = 0; u < KC; ++u) w[r][u] = __builtin_nontemporal_load(reinterpret_cast<const ld_u32x4 *>(p + (lane * 8 + u * 512 < K ? lane * 8 + u * 512 : 0)));
    }
  }
  __device__ __forceinline__ ld_u32x4 piece(int r, int u, int K, int lane) const {
    return u * 512 + 512 <= K || lane * 8 + u * 512 < K ? w[r][u] : ld_u32x4{0u, 0u, 0u, 0u};
  }
};

// Rows [n0, n1) against the activation vector x, R at a time, the next set requested before the current one's sums are
// reduced; store(n, value of row n, value of row n + 1 or 0) runs on lane 0 for the first row of each pair (R == 2).
template <int KC, typename Store>
__device__ __forceinline__ void stream_rows(RowSet<KC, 2> &rs, const ld_u32x4 (&x)[KC], const uint16_t *W, int64_t ldw, int n0, int n1, int K,
                                            int lane, Store store) {
  for (int n = n0; n < n1; n += 2) {
    float a0 = 0.f, a1 = 0.f;
#pragma unroll
    for (int u = 0; u < KC; ++u) {
      a0 = ld_dot8(rs.piece(0, u, K, lane), x[u], a0);
      a1 = ld_dot8(rs.piece(1, u, K, lane), x[u], a1);
    }
    if (n + 2 < n1) rs.load(W, ldw, n + 2, n1 - 1, K, lane);
    a0 = wave_sum(a0);
    a1 = wave_sum(a1);
    if (lane == 0) store(n, a0, a1);
  }
}

// Block `block` of `blocks` (eight waves each) of a LatentInArgs' launch, meant to have a CU to itself.  The block forms the
// normalised vectors once, eight elements a thread, and its waves take them from LDS (2 K elements per product); a wave owns every
// (8 blocks)-th pair of rows, neighbouring blocks neighbouring pairs, and keeps one pair on its way, from the block's first instructions on,
// a row of the next asked for as soon as one of this is multiplied.  More on their way are slower: with two pairs, and neighbouring pairs to the waves of a
// block, width 2048, us, before / so: 6464 rows 8.3, 7.2; 16384 gated beside the delta step 14.7, 13.1; 24576, most of them gated, 18.5, 17.1; a
// head of 32768 22.7, 21.6; 2048 rows on f32 sums 5.5, 5.1.
constexpr int kRowWaves = 8, kRowThreads = 64 * kRowWaves, kRowGroups = 16;
inline size_t latent_in_lds(const LatentInArgs &a) { return ((size_t)a.K * ((a.N1 > 0) + (a.N2 > 0)) * 2 + 15) / 16 * 16 + (kRowWaves * (1 + kRowGroups)) * sizeof(float); }
// Whether the wave at pair `at` takes the second product's vector, which lies K elements behind the first one's if both are there.  A
// wave behind the last pair takes one as well, and only those that are there.
__host__ __device__ __forceinline__ bool latent_in_second(const LatentInArgs &a, int at) { return a.N2 > 0 && at >= (a.N1 + 1) / 2; }
template <int KC> __device__ __forceinline__ void latent_in_block(const LatentInArgs &a, int block, int blocks, char *lds) {
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int pairs1 = (a.N1 + 1) / 2, pairs = pairs1 + (a.N2 + 1) / 2, stride = blocks * kRowWaves;
  int at = wave * blocks + block;
  uint16_t *xs1 = reinterpret_cast<uint16_t *>(lds), *xs2 = xs1 + (a.N1 > 0 ? a.K : 0);
  float *part = reinterpret_cast<float *>(lds + ((size_t)a.K * ((a.N1 > 0) + (a.N2 > 0)) * 2 + 15) / 16 * 16), *gpart = part + kRowWaves;
  // the small, L2-resident vectors first (loads return in order), then the first weights
  const int k = tid * 8;
  const bool mine = k < a.H;   // (H is a multiple of 8)
  const int from = mine ? k : 0;
  ld_f32x4 x0, x1;
  ld_u32x4 raw, w1, w2;
  if (a.src_f32) {
    x0 = *reinterpret_cast<const ld_f32x4 *>((const float *)a.src + from);
    x1 = *reinterpret_cast<const ld_f32x4 *>((const float *)a.src + from + 4);
  } else {
    raw = *reinterpret_cast<const ld_u32x4 *>((const uint16_t *)a.src + from);
  }
  if (a.kind != kStreamCopy) {
    w1 = *reinterpret_cast<const ld_u32x4 *>((const uint16_t *)(a.N1 ? a.n1 : a.n2) + from);
    w2 = *reinterpret_cast<const ld_u32x4 *>((const uint16_t *)(a.N2 ? a.n2 : a.n1) + from);
  }
  RowSet<KC, 2> rs;
  // (behind the last pair: one line of the weights, again and again, so that the loads on their way can be counted)
  auto request = [&](int pair, int r) __attribute__((always_inline)) {
    const bool some = pair < pairs, second = some ? pair >= pairs1 : a.N1 == 0;
    const int n = !some ? 0 : 2 * (second ? pair - pairs1 : pair) + r, last = !some ? 0 : (second ? a.N2 : a.N1) - 1, K = some ? a.K : 0;
    const uint16_t *p = (const uint16_t *)(second ? a.W2 : a.W1) + (int64_t)(n < last ? n : last) * a.ldw;
#pragma unroll
    for (int u = 0; u < KC; ++u) rs.w[r][u] = __builtin_nontemporal_load(reinterpret_cast<const ld_u32x4 *>(p + (lane * 8 + u * 512 < K ? lane * 8 + u * 512 : 0)));
  };
  request(at, 0);
  request(at, 1);
  float x[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = a.src_f32 ? (e < 4 ? x0[e & 3] : x1[e & 3]) : e & 1 ? hi_f32(raw[e >> 1]) : lo_f32(raw[e >> 1]);
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = mine ? x[e] : 0.f;
  if (a.src_scale != 0.f) {
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] *= a.src_scale;
  }
  if (a.kind == kStreamLayerNorm) {
    float s = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) s += x[e];
    s = wave_sum(s);
    if (lane == 0) part[wave] = s;
    __syncthreads();
    s = 0.f;
#pragma unroll
    for (int w = 0; w < kRowWaves; ++w) s += part[w];
    const float mean = s / (float)a.H;
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = mine ? x[e] - mean : 0.f;
  }
  float sc = a.h_scale != 0.f ? a.h_scale : 1.0f;
  if (a.kind != kStreamCopy) {
    const int gsize = a.groups == 1 ? a.H : a.H / a.groups, grp = a.groups == 1 ? (k < a.H ? 0 : 1) : k / gsize;
    float q = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) q = fmaf(x[e], x[e], q);
    for (int g = 0; g < a.groups; ++g) {
      const float s = wave_sum(grp == g ? q : 0.f);
      if (lane == 0) gpart[g * kRowWaves + wave] = s;
    }
    __syncthreads();
    float s = 0.f;
#pragma unroll
    for (int w = 0; w < kRowWaves; ++w) s += gpart[(grp < a.groups ? grp : 0) * kRowWaves + w];
    sc /= sqrtf(s / (float)gsize + a.eps);
  }
  if (k < a.K) {
    const ld_u32x4 ones = {0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};
    auto put = [&](uint16_t *xs, const ld_u32x4 &w) {
      ld_u32x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = mine ? pack_bf16x2(x[2 * e] * sc * lo_f32(w[e]), x[2 * e + 1] * sc * hi_f32(w[e])) : 0u;
      *reinterpret_cast<ld_u32x4 *>(xs + k) = v;
      return v;
    };
    if (a.N1) put(xs1, a.kind == kStreamCopy ? ones : w1);
    if (a.N2) {
      const ld_u32x4 v = put(xs2, a.kind == kStreamCopy ? ones : w2);
      if (a.h2 && block == 0) *reinterpret_cast<ld_u32x4 *>((uint16_t *)a.h2 + k) = v;
    }
  }
  __syncthreads();
  ld_u32x4 xv[KC];
  auto take = [&](bool second) {
#pragma unroll
    for (int u = 0; u < KC; ++u)
      xv[u] = lane * 8 + u * 512 < a.K ? *reinterpret_cast<const ld_u32x4 *>((second ? xs2 : xs1) + lane * 8 + u * 512) : ld_u32x4{0u, 0u, 0u, 0u};
  };
  bool second = latent_in_second(a, at);
  take(second);
  auto finish = [&]() {
    if (!second && latent_in_second(a, at)) take(second = true);
    float v0 = 0.f, v1 = 0.f;
#pragma unroll
    for (int u = 0; u < KC; ++u) v0 = ld_dot8(rs.piece(0, u, a.K, lane), xv[u], v0);
    __builtin_amdgcn_sched_barrier(0);
    request(at + stride, 0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < KC; ++u) v1 = ld_dot8(rs.piece(1, u, a.K, lane), xv[u], v1);
    __builtin_amdgcn_sched_barrier(0);
    request(at + stride, 1);
    __builtin_amdgcn_sched_barrier(0);
    v0 = wave_sum(v0);
    v1 = wave_sum(v1);
    if (lane != 0) return;
    const int n = 2 * (second ? at - pairs1 : at), N = second ? a.N2 : a.N1;
    if (!second) {
      uint16_t *o = (uint16_t *)a.out1 + n;
      o[0] = f32_to_bf16_bits(v0);
      if (n + 1 < N) o[1] = f32_to_bf16_bits(v1);
    } else if (a.gated2) {
      ((uint16_t *)a.out2)[n >> 1] = f32_to_bf16_bits(gated(a, v0, v1));
    } else {
      float *o = (float *)a.out2 + n;
      if (a.add2) { v0 += a.add2[n]; if (n + 1 < N) v1 += a.add2[n + 1]; }
      if (a.bias2) { v0 += bf16_bits_to_f32(((const uint16_t *)a.bias2)[n]); if (n + 1 < N) v1 += bf16_bits_to_f32(((const uint16_t *)a.bias2)[n + 1]); }
      o[0] = v0;
      if (n + 1 < N) o[1] = v1;
    }
  };
  for (; at < pairs; at += stride) finish();
}

}  // namespace rai
