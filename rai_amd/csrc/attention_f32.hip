// Prefill attention in f32 on the f32 matrix instructions (scores, probabilities and sums all in f32).
//
// Reference semantics: rai-models/src/llm/phi2.rs:244-262, qwen2.rs:205-221, gemma.rs:238-254 (see attention.hip).
#include <cstdlib>

#include "attention.h"

namespace rai {

typedef __attribute__((ext_vector_type(4))) float af_f32x4;
typedef __attribute__((ext_vector_type(16))) float af_f32x16;

__device__ __forceinline__ float af_gate(float z) { return 1.0f / (1.0f + expf(-z)); }

// A wave owns 32 query rows of one head and walks key tiles of 32, both products on v_mfma_f32_32x32x2_f32 in the
// transposed orientation S^T = K Q^T, O^T = V^T P^T.  Lane (r, h) then owns query r: register e of its scores is key
// 8 (e / 4) + 4 h + e % 4, and that register is, as it stands, the operand of the e-th MFMA of the second product, whose other
// operand is feature r of that key.  Tiles go straight from memory into LDS (K with its 16-byte chunks swizzled by row, so
// that the 16-byte reads of 32 rows spread over the banks; V as it lies); the registers hold the queries, the output and
// one tile's sums.  (A form without LDS, both operands loaded into registers a tile ahead, was as fast and ran out of those.)
//   One wave is one SIMD's 150 GFLOP/s, so where there are few query groups KSP waves share one, each with every KSP-th
// key tile, and are merged through LDS.  DB: two LDS stages, the next round's tiles requested before this one's are
// multiplied; otherwise several waves share the work of a group and cover each other's waits.
//   Sums of products are kept in short chains, two side by side (16 features of a score, 8 keys of an output; twice that
// beyond 128 features): less rounding, and no MFMA waits for the one before it.  That takes 512 registers, one block to a CU.
//   A masked probability is zero and must not meet an infinity or a NaN of V in the product (0 x inf): in tiles with masks
// those are left out, and afterwards added for the queries that see them.
//   Head sizes of 128 and more; smaller ones take the form for 16 rows below.  Measured (us; one block per query row on the vector
// units in brackets): 16 x 12 x 1024 x 128 on 2 key heads 993 (3900), 2 x 8 x 512 x 256 130 (178).  Off by 1.28e-7 (1.36e-7),
// 1.43e-7 (1.47e-7).  Two stages also with two waves at 128 features: 16 heads x 1024 112 -> 109.5.
template <int D> struct F32Attn {
  static_assert(D >= 128 && D % 64 == 0, "whole 32-feature tiles, a row of K over all banks, as many pieces for every wave");
  static constexpr int CPR = D / 4, DT = D / 32, TILE = 32 * D, LOADS = D / 8;   // 1 KB pieces of a tile
  static __device__ __forceinline__ int swizzle(int row) { return row & 15; }
};

template <int D, int KSP, bool DB>
__global__ void __launch_bounds__(256, 1) k_flash_prefill_f32(AttnArgs a) {
  typedef F32Attn<D> F;
  constexpr int NG = 4 / KSP, KC = D / 8, CG = D <= 128 ? 2 : 4, DT = F::DT, STAGE = KSP * 2 * F::TILE, LW = F::LOADS / 4;
  extern __shared__ __attribute__((aligned(16))) float af_lds[];
  typedef __attribute__((address_space(3))) void *lds_ptr;
  const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), kh = wave % KSP;
  const int head = blockIdx.x, b = blockIdx.z, hk = head / (a.Hq / a.Hkv);
  // The last query groups see the most keys under a causal mask: those of all heads go first.  Heads next to each other
  // land on different XCDs, whose L2s then hold the keys of few heads each.
  const int block_q0 = (int)(gridDim.y - 1 - blockIdx.y) * NG * 32, q0 = block_q0 + wave / KSP * 32;
  const int off = a.T - a.S;
  const float *Kg = (const float *)a.k + b * a.ks[0] + hk * a.ks[1];
  const float *Vg = (const float *)a.v + b * a.vs[0] + hk * a.vs[1];
  const int qrow = q0 + r, q_abs = off + qrow;
  const float *qp = (const float *)a.q + b * a.qs[0] + head * a.qs[1] + (int64_t)min(qrow, a.S - 1) * a.qs[2] + 4 * h;
  af_f32x4 qf[KC];
#pragma unroll
  for (int c = 0; c < KC; ++c) qf[c] = *reinterpret_cast<const af_f32x4 *>(qp + 8 * c);
  af_f32x16 o[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[t][e] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;
  bool left_out = false;   // some infinity or NaN of V in a tile with masks
  const int last_key = a.causal ? min(q_abs, a.T - 1) : a.T - 1;              // newest and oldest key this lane's query sees
  const int first_key = a.window > 0 ? q_abs - a.window + 1 : 0;
  auto end_of = [&](int q, int n) { return q >= a.S ? 0 : a.causal ? min(off + min(q + n, a.S), a.T) : a.T; };
  const int kv_end = end_of(q0, 32), block_end = end_of(block_q0, 32 * NG);  // of any query of the group, of the block
  const int oldest = a.window > 0 ? max(off + q0 - a.window + 1, 0) : 0;
  const int begin = a.window > 0 ? max(off + block_q0 - a.window + 1, 0) & ~31 : 0;

  // this thread's 16 bytes of the wave's LW loads of a tile
  uint32_t k_off[LW], v_off[LW];
#pragma unroll
  for (int j = 0; j < LW; ++j) {
    const int i = (wave + 4 * j) * 64 + lane, row = i / F::CPR, c = i % F::CPR;
    k_off[j] = (uint32_t)(row * (int)a.ks[2] + 4 * (c ^ F::swizzle(row)));
    v_off[j] = (uint32_t)(row * (int)a.vs[2] + 4 * c);
  }
  // where this lane's chunks of a row of K lie: the swizzle stays within PAT chunks, what is beyond goes into the instruction
  constexpr int PAT = 16;
  int k_lane[PAT / 2];
#pragma unroll
  for (int c = 0; c < PAT / 2; ++c) k_lane[c] = r * D + 4 * ((2 * c + h) ^ F::swizzle(r));
  // a tile past the end of the keys starts early: what lies before its own first key is masked
  auto fetch = [&](int base, int stage) {
#pragma unroll
    for (int i = 0; i < KSP; ++i) {
      const int kt = min(base + 32 * i, a.T - 32);
      const float *kp = Kg + (int64_t)kt * a.ks[2], *vp = Vg + (int64_t)kt * a.vs[2];
      float *kd = af_lds + stage * STAGE + i * 2 * F::TILE, *vd = kd + F::TILE;
#pragma unroll
      for (int j = 0; j < LW; ++j) {
        __builtin_amdgcn_global_load_lds((const void *)(kp + k_off[j]), (lds_ptr)(kd + (wave + 4 * j) * 256), 16, 0, 0);
        __builtin_amdgcn_global_load_lds((const void *)(vp + v_off[j]), (lds_ptr)(vd + (wave + 4 * j) * 256), 16, 0, 0);
      }
    }
  };
  auto landed = [&]() {   // every wave's loads, for every wave
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  };
  if (DB && begin < block_end) fetch(begin, 0);
  int stage = 0;
  for (int base = begin; base < block_end; base += 32 * KSP) {
    if (DB) {
      landed();   // and everybody is done with the other stage
      if (base + 32 * KSP < block_end) fetch(base + 32 * KSP, stage ^ 1);
    } else {
      if (base > begin) __syncthreads();   // everybody is done with the last round's tiles
      fetch(base, 0);
      landed();
    }
    const float *Kt = af_lds + stage * STAGE + kh * 2 * F::TILE, *Vt = Kt + F::TILE;
    if (DB) stage ^= 1;
    const int k0 = base + 32 * kh, kt = min(k0, a.T - 32);
    if (k0 >= kv_end || k0 + 31 < oldest) continue;   // nothing this wave's queries see
    // (the fences keep the compiler from starting several steps' sums at once, which takes more registers than there are)
    af_f32x16 s;
#pragma unroll
    for (int c0 = 0; c0 < KC; c0 += CG) {
      af_f32x16 sg[2];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) sg[i][e] = 0.f;
#pragma unroll
      for (int c = c0; c < c0 + CG; ++c) {
        const af_f32x4 kf = *reinterpret_cast<const af_f32x4 *>(Kt + k_lane[c % (PAT / 2)] + 4 * (2 * c & ~(PAT - 1)));
#pragma unroll
        for (int j = 0; j < 4; ++j) sg[j & 1] = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[j], qf[c][j], sg[j & 1], 0, 0, 0);
      }
#pragma unroll
      for (int e = 0; e < 16; ++e) s[e] = (c0 ? s[e] : 0.f) + (sg[0][e] + sg[1][e]);
      __builtin_amdgcn_sched_barrier(0);
    }
    // ---- scale, cap, mask (the scale, where nothing follows it, goes into the exponent's subtraction: one rounding less)
    const bool masked = k0 != kt || (a.causal && k0 + 31 > off + q0) || (a.window > 0 && k0 <= off + q0 + 31 - a.window);
    float mx = -INFINITY;
    const float now = a.softcap > 0.f || !(a.scale > 0.f) ? a.scale : 1.f, later = now == 1.f ? a.scale : 1.f;
#pragma unroll
    for (int e = 0; e < 16; ++e) s[e] *= now;
    if (a.softcap > 0.f) {
#pragma unroll
      for (int e = 0; e < 16; ++e) s[e] = a.softcap * tanhf(s[e] / a.softcap);
    }
    if (masked) {
      const int from = max(first_key, k0);
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int key = kt + 8 * (e >> 2) + 4 * h + (e & 3);
        s[e] = key > last_key || key < from ? -INFINITY : s[e];
      }
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) mx = fmaxf(mx, s[e] * later);
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float m_new = fmaxf(m_run, mx), m_safe = m_new == -INFINITY ? 0.f : m_new;
    const float alpha = expf(m_run - m_safe);
    float sum[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      s[e] = expf(fmaf(s[e], later, -m_safe));
      sum[e & 3] += s[e];
    }
    m_run = m_new;
    l_run = l_run * alpha + ((sum[0] + sum[1]) + (sum[2] + sum[3]));
    // ---- O^T <- alpha O^T + V^T P^T, the products of sixteen keys in a chain
#pragma unroll
    for (int t = 0; t < DT; ++t) {
      const float *vp = Vt + 4 * h * D + 32 * t + r;
      float v[16];
#pragma unroll
      for (int e = 0; e < 16; ++e) v[e] = vp[(8 * (e >> 2) + (e & 3)) * D];
      if (masked) {
#pragma unroll
        for (int e = 0; e < 16; ++e)
          if (!(fabsf(v[e]) < INFINITY)) { v[e] = 0.f; left_out = true; }
      }
      af_f32x16 p0, p1;
#pragma unroll
      for (int e = 0; e < 16; ++e) p0[e] = p1[e] = 0.f;
      if constexpr (D <= 128) {   // four chains
        af_f32x16 q;
#pragma unroll
        for (int half = 0; half < 2; ++half) {
          if (half) {
#pragma unroll
            for (int e = 0; e < 16; ++e) { q[e] = p0[e] + p1[e]; p0[e] = p1[e] = 0.f; }
            __builtin_amdgcn_sched_barrier(0);
          }
#pragma unroll
          for (int e = 8 * half; e < 8 * half + 4; ++e) {
            p0 = __builtin_amdgcn_mfma_f32_32x32x2f32(v[e], s[e], p0, 0, 0, 0);
            p1 = __builtin_amdgcn_mfma_f32_32x32x2f32(v[e + 4], s[e + 4], p1, 0, 0, 0);
          }
        }
#pragma unroll
        for (int e = 0; e < 16; ++e) p0[e] += q[e];
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          p0 = __builtin_amdgcn_mfma_f32_32x32x2f32(v[e], s[e], p0, 0, 0, 0);
          p1 = __builtin_amdgcn_mfma_f32_32x32x2f32(v[e + 8], s[e + 8], p1, 0, 0, 0);
        }
      }
#pragma unroll
      for (int e = 0; e < 16; ++e) o[t][e] = fmaf(o[t][e], alpha, p0[e] + p1[e]);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  if (__builtin_amdgcn_ballot_w64(left_out)) {
    // What was left out goes to the queries that see it: the tiles with masks once more, key by key.
#pragma unroll 1
    for (int k1 = begin + 32 * kh; k1 < kv_end; k1 += 32 * KSP) {
      if (k1 + 31 < oldest) continue;
      const int kt = min(k1, a.T - 32), from = max(first_key, k1);
      if (!(k1 != kt || (a.causal && k1 + 31 > off + q0) || (a.window > 0 && k1 <= off + q0 + 31 - a.window))) continue;
#pragma unroll 1
      for (int key = kt; key < kt + 32; ++key) {
        const float *kp = Kg + (int64_t)key * a.ks[2] + 4 * h, *vp = Vg + (int64_t)key * a.vs[2] + 4 * h;
        float dot = 0.f;
#pragma unroll
        for (int c = 0; c < KC; ++c)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            dot = fmaf(kp[8 * c + j], qf[c][j], dot);
            if (c % 4 == 3 && j == 3) __builtin_amdgcn_sched_barrier(0);
          }
        dot = (dot + __shfl_xor(dot, 32, 64)) * a.scale;
        if (a.softcap > 0.f) dot = a.softcap * tanhf(dot / a.softcap);
        if (key > last_key || key < from) continue;
        const float p = expf(dot - m_run);
#pragma unroll
        for (int t = 0; t < DT; ++t) {
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            const float x = vp[32 * t + 8 * (e >> 2) + (e & 3)];
            o[t][e] = fabsf(x) < INFINITY ? o[t][e] : fmaf(p, x, o[t][e]);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
  }
  float l_tot = l_run + __shfl_xor(l_run, 32, 64);
  if constexpr (KSP > 1) {
    constexpr int MS = (2 + DT * 16) * 64;   // floats a wave hands over: value by value, lane by lane
    __syncthreads();                         // the tiles are no longer read
    if (kh > 0) {
      float *mine = af_lds + (wave / KSP * (KSP - 1) + kh - 1) * MS + lane;
      mine[0] = m_run;
      mine[64] = l_tot;
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) mine[(2 + t * 16 + e) * 64] = o[t][e];
    }
    __syncthreads();
    if (kh > 0) return;
    const float *theirs = af_lds + wave / KSP * (KSP - 1) * MS + lane;
    float m = m_run;
#pragma unroll
    for (int j = 0; j < KSP - 1; ++j) m = fmaxf(m, theirs[j * MS]);
    const float ms = m == -INFINITY ? 0.f : m, w0 = expf(m_run - ms);
    l_tot *= w0;
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int e = 0; e < 16; ++e) o[t][e] *= w0;
#pragma unroll 1
    for (int j = 0; j < KSP - 1; ++j) {
      const float *p = theirs + j * MS, w = expf(p[0] - ms);
      l_tot = fmaf(p[64], w, l_tot);
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[t][e] = fmaf(p[(2 + t * 16 + e) * 64], w, o[t][e]);
    }
    m_run = m;
  }
  if (qrow >= a.S) return;
  float scale = 1.0f;
  if (a.sink) {   // relative to the larger of the two exponents
    const float sink = ((const float *)a.sink)[head], m = fmaxf(m_run, sink);
    scale = expf(m_run - m);
    l_tot = l_tot * scale + expf(sink - m);
  }
  const float inv = scale / l_tot;
  const int64_t row = (int64_t)b * a.S + qrow;
  float *op = (float *)a.out + row * a.out_row_stride + (int64_t)head * D;
  const float *gp = a.gate ? (const float *)a.gate + row * a.gate_row_stride + (int64_t)head * D : nullptr;
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int e = 0; e < 16; e += 4) {
      const int d = 32 * t + 2 * e + 4 * h;   // 8 (e / 4)
      af_f32x4 w = {o[t][e] * inv, o[t][e + 1] * inv, o[t][e + 2] * inv, o[t][e + 3] * inv};
      if (gp) {
#pragma unroll
        for (int j = 0; j < 4; ++j) w[j] *= af_gate(gp[d + j]);
      }
      *reinterpret_cast<af_f32x4 *>(op + d) = w;
    }
}

// The same for 16 query rows to a wave, on v_mfma_f32_16x16x4_f32: half the registers, so that two blocks share a CU and a wave's
// exponentials and sums run beside another's products (32 rows to a wave: one wave a SIMD, MFMAs a fifth of the time).  Lane
// (r, g) = (l % 16, l / 16) owns query r: register 4 hh + e of its scores is key 16 hh + g + 4 e of the tile, and the operand of an MFMA
// of the second product as it stands; row a of the first product's other operand is therefore key (a / 4) + 4 (a % 4).  A wave's
// key tiles are its own, K and V in one buffer each: the next K is asked for when the scores are formed, the next V behind the
// products with this one, and nothing waits for another wave until the merge.  V's 16-feature blocks are swapped by row where a row
// is a multiple of 64 floats (vswizzle), so that the four keys of a read are on different banks.
//   Chains of sums as above: 8 features of a score (two side by side), 8 keys of an output.
//   Measured against 32 rows to a wave (us): 32 heads x 128 x 80 10.1 -> 6.6, 32 x 333 x 80 24.5 -> 18.4, 32 x 700 x 80 54.4 -> 41.0,
// 8 x 32 x 200 x 80 70.7 -> 45.3, 32 x 1024 x 64 74.1 -> 64.2, 4 x 32 x 500 x 64 on 900 keys 175 -> 145, 32 x 1024 x 32 47.3 -> 36.4; off by
// 1.22e-7 (1.23e-7), 1.26e-7 (1.27e-7) at 512 x 80, 1.23e-7 (1.25e-7) at 500 x 64.  At 128 features the tiles are 128 KB and the
// registers spill: 132 instead of 110 at 16 x 1024.  What bounds it: the MFMAs are 1.07 us of a tile's two or so at 80 features,
// and each block reads its own keys from L2 (79 MB at 32 x 333, some 7 us of it).
template <int D> struct F32Attn16 {
  static constexpr int CPR = D / 4, TILE = 32 * D, LOADS = D / 8, KC = D / 16;   // 1 KB pieces of a tile; 16-feature blocks
  static __device__ __forceinline__ int kswizzle(int row) { return D == 80 ? (row >> 2) & 3 : D == 32 ? (row >> 1) & 7 : row & 15; }
  static __device__ __forceinline__ int vswizzle(int row) { return D == 80 ? 0 : D == 32 ? (row >> 1 & 1) << 2 : (row & 3) << 2; }   // of 16-byte chunks
};
__device__ __forceinline__ float af_quarter_fold_max(float v) {   // over the four lanes of a query
  typedef __attribute__((ext_vector_type(2))) unsigned pair;
  pair p = __builtin_bit_cast(pair, __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false));
  v = fmaxf(__uint_as_float(p.x), __uint_as_float(p.y));
  p = __builtin_bit_cast(pair, __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false));
  return fmaxf(__uint_as_float(p.x), __uint_as_float(p.y));
}
__device__ __forceinline__ float af_quarter_sum(float v) {
  typedef __attribute__((ext_vector_type(2))) unsigned pair;
  pair p = __builtin_bit_cast(pair, __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false));
  v = __uint_as_float(p.x) + __uint_as_float(p.y);
  p = __builtin_bit_cast(pair, __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false));
  return __uint_as_float(p.x) + __uint_as_float(p.y);
}

template <int D, int KSP>
__global__ void __launch_bounds__(256, 2) k_flash_prefill_f32_q16(AttnArgs a) {
  typedef F32Attn16<D> F;
  constexpr int NG = 4 / KSP, KC = F::KC;
  extern __shared__ __attribute__((aligned(16))) float af_lds[];
  typedef __attribute__((address_space(3))) void *lds_ptr;
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), kh = wave % KSP;
  const int head = blockIdx.x, b = blockIdx.z, hk = head / (a.Hq / a.Hkv);
  const int q0 = (int)(gridDim.y - 1 - blockIdx.y) * NG * 16 + wave / KSP * 16;   // the groups that see the most keys first
  const int off = a.T - a.S;
  const float *Kg = (const float *)a.k + b * a.ks[0] + hk * a.ks[1];
  const float *Vg = (const float *)a.v + b * a.vs[0] + hk * a.vs[1];
  float *Kt = af_lds + wave * 2 * F::TILE, *Vt = Kt + F::TILE;
  const int qrow = q0 + r, q_abs = off + qrow;
  const int last_key = a.causal ? min(q_abs, a.T - 1) : a.T - 1;              // newest and oldest key this lane's query sees
  const int first_key = a.window > 0 ? q_abs - a.window + 1 : 0;
  const int kv_end = q0 >= a.S ? 0 : a.causal ? min(off + min(q0 + 16, a.S), a.T) : a.T;   // of any query of the group
  const int oldest = a.window > 0 ? max(off + q0 - a.window + 1, 0) : 0;
  uint32_t k_off[F::LOADS], v_off[F::LOADS];
#pragma unroll
  for (int j = 0; j < F::LOADS; ++j) {
    const int i = j * 64 + lane, row = i / F::CPR, c = i % F::CPR;
    k_off[j] = (uint32_t)(row * (int)a.ks[2] + 4 * (c ^ F::kswizzle(row)));
    v_off[j] = (uint32_t)(row * (int)a.vs[2] + 4 * (c ^ F::vswizzle(row)));
  }
  // a tile past the end of the keys starts early: what lies before its own first key is masked
  auto fetch_k = [&](int base) __attribute__((always_inline)) {
    const float *p = Kg + (int64_t)min(base, a.T - 32) * a.ks[2];
#pragma unroll
    for (int j = 0; j < F::LOADS; ++j) __builtin_amdgcn_global_load_lds((const void *)(p + k_off[j]), (lds_ptr)(Kt + j * 256), 16, 0, 0);
  };
  auto fetch_v = [&](int base) __attribute__((always_inline)) {
    const float *p = Vg + (int64_t)min(base, a.T - 32) * a.vs[2];
#pragma unroll
    for (int j = 0; j < F::LOADS; ++j) __builtin_amdgcn_global_load_lds((const void *)(p + v_off[j]), (lds_ptr)(Vt + j * 256), 16, 0, 0);
  };
  const int begin = (oldest & ~31) + 32 * kh;
  const float *qp = (const float *)a.q + b * a.qs[0] + head * a.qs[1] + (int64_t)min(qrow, a.S - 1) * a.qs[2] + 4 * g;
  af_f32x4 qf[KC];
#pragma unroll
  for (int c = 0; c < KC; ++c) qf[c] = *reinterpret_cast<const af_f32x4 *>(qp + 16 * c);
  if (begin < kv_end) {
    fetch_k(begin);
    fetch_v(begin);
  }
  af_f32x4 o[KC];
#pragma unroll
  for (int t = 0; t < KC; ++t) o[t] = af_f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_run = 0.f;
  bool left_out = false;   // some infinity or NaN of V in a tile with masks
  const int arow = (r >> 2) + 4 * (r & 3);   // the key of this lane's row of the first product
  for (int k0 = begin; k0 < kv_end; k0 += 32 * KSP) {
    const bool more = k0 + 32 * KSP < kv_end;
    const int kt = min(k0, a.T - 32);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(F::LOADS) : "memory");   // K is here, V on its way
    af_f32x4 s[2];
#pragma unroll
    for (int c = 0; c < KC; ++c) {
      af_f32x4 sg[2][2], kf[2];
#pragma unroll
      for (int i = 0; i < 4; ++i) sg[i >> 1][i & 1] = af_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) {
        const int row = 16 * hh + arow;
        kf[hh] = *reinterpret_cast<const af_f32x4 *>(Kt + row * D + 4 * ((4 * c + g) ^ F::kswizzle(row)));
      }
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) sg[hh][j & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[hh][j], qf[c][j], sg[hh][j & 1], 0, 0, 0);
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) s[hh] = c ? s[hh] + (sg[hh][0] + sg[hh][1]) : sg[hh][0] + sg[hh][1];
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (more) fetch_k(k0 + 32 * KSP);
    // ---- scale, cap, mask (the scale, where nothing follows it, goes into the exponent's subtraction: one rounding less)
    const bool masked = k0 != kt || (a.causal && k0 + 31 > off + q0) || (a.window > 0 && k0 <= off + q0 + 15 - a.window);
    const float now = a.softcap > 0.f || !(a.scale > 0.f) ? a.scale : 1.f, later = now == 1.f ? a.scale : 1.f;
    float mx = -INFINITY;
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) s[hh] *= now;
    if (a.softcap > 0.f) {
#pragma unroll
      for (int e = 0; e < 8; ++e) s[e >> 2][e & 3] = a.softcap * tanhf(s[e >> 2][e & 3] / a.softcap);
    }
    if (masked) {
      const int from = max(first_key, k0);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int key = kt + 16 * (e >> 2) + g + 4 * (e & 3);
        s[e >> 2][e & 3] = key > last_key || key < from ? -INFINITY : s[e >> 2][e & 3];
      }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) mx = fmaxf(mx, s[e >> 2][e & 3] * later);
    mx = af_quarter_fold_max(mx);
    const float m_new = fmaxf(m_run, mx), m_safe = m_new == -INFINITY ? 0.f : m_new;
    const float alpha = expf(m_run - m_safe);
    float sum[2] = {0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      s[e >> 2][e & 3] = expf(fmaf(s[e >> 2][e & 3], later, -m_safe));
      sum[e & 1] += s[e >> 2][e & 3];
    }
    m_run = m_new;
    l_run = l_run * alpha + (sum[0] + sum[1]);
    if (more) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(F::LOADS) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    // ---- O^T <- alpha O^T + V^T P^T, the products of eight keys in a chain
#pragma unroll
    for (int t = 0; t < KC; ++t) {
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int row = 16 * (e >> 2) + g + 4 * (e & 3);
        v[e] = Vt[row * D + 4 * ((4 * t) ^ F::vswizzle(row)) + r];
      }
      if (masked) {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (!(fabsf(v[e]) < INFINITY)) { v[e] = 0.f; left_out = true; }
      }
      af_f32x4 p[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) p[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[2 * i], s[i >> 1][2 * i & 3], af_f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; ++i) p[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[2 * i + 1], s[i >> 1][(2 * i & 3) + 1], p[i], 0, 0, 0);
#pragma unroll
      for (int e = 0; e < 4; ++e) o[t][e] = fmaf(o[t][e], alpha, (p[0][e] + p[1][e]) + (p[2][e] + p[3][e]));
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (more) fetch_v(k0 + 32 * KSP);
  }
  if (__builtin_amdgcn_ballot_w64(left_out)) {
    // What was left out goes to the queries that see it: the tiles with masks once more, key by key.
#pragma unroll 1
    for (int k1 = begin; k1 < kv_end; k1 += 32 * KSP) {
      const int kt = min(k1, a.T - 32), from = max(first_key, k1);
      if (!(k1 != kt || (a.causal && k1 + 31 > off + q0) || (a.window > 0 && k1 <= off + q0 + 15 - a.window))) continue;
#pragma unroll 1
      for (int key = kt; key < kt + 32; ++key) {
        const float *kp = Kg + (int64_t)key * a.ks[2] + 4 * g, *vp = Vg + (int64_t)key * a.vs[2] + 4 * g;
        float dot = 0.f;
#pragma unroll
        for (int c = 0; c < KC; ++c)
#pragma unroll
          for (int j = 0; j < 4; ++j) dot = fmaf(kp[16 * c + j], qf[c][j], dot);
        dot = af_quarter_sum(dot) * a.scale;
        if (a.softcap > 0.f) dot = a.softcap * tanhf(dot / a.softcap);
        if (key > last_key || key < from) continue;
        const float p = expf(dot - m_run);
#pragma unroll
        for (int t = 0; t < KC; ++t)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float x = vp[16 * t + e];
            o[t][e] = fabsf(x) < INFINITY ? o[t][e] : fmaf(p, x, o[t][e]);
          }
      }
    }
  }
  float l_tot = af_quarter_sum(l_run);
  if constexpr (KSP > 1) {
    constexpr int MS = (2 + KC * 4) * 64;   // floats a wave hands over: value by value, lane by lane
    __syncthreads();                        // the tiles are no longer read
    if (kh > 0) {
      float *mine = af_lds + (wave / KSP * (KSP - 1) + kh - 1) * MS + lane;
      mine[0] = m_run;
      mine[64] = l_tot;
#pragma unroll
      for (int t = 0; t < KC; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) mine[(2 + t * 4 + e) * 64] = o[t][e];
    }
    __syncthreads();
    if (kh > 0) return;
    const float *theirs = af_lds + wave / KSP * (KSP - 1) * MS + lane;
    float m = m_run;
#pragma unroll
    for (int j = 0; j < KSP - 1; ++j) m = fmaxf(m, theirs[j * MS]);
    const float ms = m == -INFINITY ? 0.f : m, w0 = expf(m_run - ms);
    l_tot *= w0;
#pragma unroll
    for (int t = 0; t < KC; ++t) o[t] *= w0;
#pragma unroll
    for (int j = 0; j < KSP - 1; ++j) {
      const float *p = theirs + j * MS, w = expf(p[0] - ms);
      l_tot = fmaf(p[64], w, l_tot);
#pragma unroll
      for (int t = 0; t < KC; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) o[t][e] = fmaf(p[(2 + t * 4 + e) * 64], w, o[t][e]);
    }
    m_run = m;
  }
  if (qrow >= a.S) return;
  float scale = 1.0f;
  if (a.sink) {   // relative to the larger of the two exponents
    const float sink = ((const float *)a.sink)[head], m = fmaxf(m_run, sink);
    scale = expf(m_run - m);
    l_tot = l_tot * scale + expf(sink - m);
  }
  const float inv = scale / l_tot;
  const int64_t row = (int64_t)b * a.S + qrow;
  float *op = (float *)a.out + row * a.out_row_stride + (int64_t)head * D + 4 * g;
  const float *gp = a.gate ? (const float *)a.gate + row * a.gate_row_stride + (int64_t)head * D + 4 * g : nullptr;
#pragma unroll
  for (int t = 0; t < KC; ++t) {
    af_f32x4 w = o[t] * inv;
    if (gp) {
#pragma unroll
      for (int j = 0; j < 4; ++j) w[j] *= af_gate(gp[16 * t + j]);
    }
    *reinterpret_cast<af_f32x4 *>(op + 16 * t) = w;
  }
}

// (see launch_f32_split for KSP)
template <int D, int KSP> static int launch_f32_q16(hipStream_t st, const AttnArgs &a) {
  constexpr int NG = 4 / KSP;
  constexpr size_t lds = (size_t)4 * 2 * F32Attn16<D>::TILE * sizeof(float);
  static_assert((size_t)NG * (KSP - 1) * (2 + D / 4) * 64 * sizeof(float) <= lds, "the merge fits the tiles");
  static bool attr_set = false;
  if (lds > 64 * 1024 && !attr_set) {
    RAI_HIP_TRY(hipFuncSetAttribute((const void *)k_flash_prefill_f32_q16<D, KSP>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    attr_set = true;
  }
  hipLaunchKernelGGL((k_flash_prefill_f32_q16<D, KSP>), dim3(a.Hq, (a.S + 16 * NG - 1) / (16 * NG), a.B), dim3(256), lds, st, a);
  return launch_check("flash_prefill_f32_q16");
}

template <int D, int KSP> static int launch_f32(hipStream_t st, const AttnArgs &a) {
  constexpr int NG = 4 / KSP;
  constexpr bool DB = D <= 128 && KSP <= 2;
  constexpr size_t tiles = (size_t)(DB ? 2 : 1) * KSP * 2 * F32Attn<D>::TILE * sizeof(float);
  constexpr size_t merge = (size_t)NG * (KSP - 1) * (2 + F32Attn<D>::DT * 16) * 64 * sizeof(float), lds = tiles > merge ? tiles : merge;
  static_assert(lds <= 160 * 1024, "LDS of a block");
  static bool attr_set = false;
  if (lds > 64 * 1024 && !attr_set) {
    RAI_HIP_TRY(hipFuncSetAttribute((const void *)k_flash_prefill_f32<D, KSP, DB>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    attr_set = true;
  }
  hipLaunchKernelGGL((k_flash_prefill_f32<D, KSP, DB>), dim3(a.Hq, (a.S + 32 * NG - 1) / (32 * NG), a.B), dim3(256), lds, st, a);
  return launch_check("flash_prefill_f32");
}

// RAI_HIP_ATTN_F32 = 1, 2 or 4 (read per call) forces this kernel with so many waves to a group; 0: not set.
static int forced_waves() {
  const char *e = getenv("RAI_HIP_ATTN_F32");
  return e ? atoi(e) : 0;
}

// Waves to a query group.  More of them make its chain of key tiles shorter and the blocks more.
//   Up to 80 features (16 rows), measured (us, with four, two, one; S = T, causal): 32 heads x 333 x 80 (672 groups) 18.5, 19.7, 28.2;
// 400 x 80 (800) 22.7, 22.6, 32.1; 700 x 80 (1408) 42.9, 41.0, 59.8; 1024 x 64 (2048) 63.6, 64.2, 77.1; 1400 x 80 132, 127, 136; short
// ones 4 x 32 x 128 x 80 (1024) 15.3, 13.1, 13.2, 16 x 32 x 64 x 80 (2048) 27.7, 16.5, 13.9, 8 x 32 x 128 x 80 28.5, 23.8, 21.5.
//   Beyond (32 rows): 16 x 1024 x 128 (512 groups) two 110, four 148.
template <int D> static int launch_f32_split(hipStream_t st, const AttnArgs &a) {
  constexpr int ROWS = D <= 80 ? 16 : 32;
  int waves = forced_waves();
  RAI_REQUIRE(waves == 0 || waves == 1 || waves == 2 || (waves == 4 && D <= 128), RAI_ERR_UNSUPPORTED, "attention: RAI_HIP_ATTN_F32=%d, head size %d", waves, D);
  if (!waves) {
    const int64_t groups = (int64_t)((a.S + ROWS - 1) / ROWS) * a.Hq * a.B;
    const int seen = a.window > 0 && a.window + 31 < a.T ? a.window + 31 : a.T, tiles = (seen + 31) / 32;
    if constexpr (D <= 80) waves = tiles >= 3 && groups <= 3 * kNumCU ? 4 : tiles >= 2 && (tiles > 4 || groups < 4 * kNumCU) ? 2 : 1;
    else waves = D == 128 && groups <= kNumCU && tiles >= 3 ? 4 : groups * 2 <= (D == 128 ? 8 : 4) * kNumCU && tiles >= 2 ? 2 : 1;
  }
  if constexpr (D <= 80) {
    return waves == 4 ? launch_f32_q16<D, 4>(st, a) : waves == 2 ? launch_f32_q16<D, 2>(st, a) : launch_f32_q16<D, 1>(st, a);
  } else {
    if constexpr (D == 128) {
      if (waves == 4) return launch_f32<D, 4>(st, a);
    }
    return waves == 2 ? launch_f32<D, 2>(st, a) : launch_f32<D, 1>(st, a);
  }
}

// What the kernel is written for, whatever it costs.
static bool takes(const AttnArgs &a) {
  if (a.S < 16 || a.T < 32 || a.t_dev) return false;
  if (a.D != 32 && a.D != 64 && a.D != 80 && a.D != 128 && a.D != 192 && a.D != 256) return false;
  auto al = [](const void *p, const int64_t *s) { return (uintptr_t)p % 16 == 0 && s[0] % 4 == 0 && s[1] % 4 == 0 && s[2] % 4 == 0 && s[2] < (1 << 24); };
  return al(a.q, a.qs) && al(a.k, a.ks) && al(a.v, a.vs) && (uintptr_t)a.out % 16 == 0 && a.out_row_stride % 4 == 0 && (a.S + 31) / 32 <= 65535 && a.B <= 65535;
}

// A block per query row (attention.hip) is done sooner where there are few rows.  Up to 80 features it is up to 512 rows, as long as an XCD's L2
// holds all keys and values, and up to 1024 rows on few keys: measured (us; block per row, here) 16 rows x 80 on 256 keys 7.4, 8.0, on 2000
// 31.5, 38.8; 8 heads x 64 x 80 on 700 (3.6 MB) 15.4, 17.5, on 1000 (5.1 MB) 23.8, 21.9; 32 x 16 x 80 on 160 7.2, 8.5, on 256 10.7, 8.6; 32 x 33 x 64
// on 64 5.9, 5.7, on 256 10.9, 7.7.  But its sums over the keys are longer chains: off by 1.88e-7 where the tiles are by 1.59e-7 (8 x 64 x 64 on 700),
// 2.06e-7 and 1.64e-7 (8 x 64 x 80 on 700), 2.84e-7 and 1.91e-7 (16 x 80 on 2000).  So it has only what is short, fewer than 64 keys, where it
// is ahead by a sixth (32 x 18 x 64 on 50 5.3, 5.9).
//   Beyond, a tile is a chain of up to 8 us (256), which takes enough rows or keys to be worth it: 8 x 64 on 300 x 128 20.0, 29.3, 32 x 64 on
// 300 38.1, 29.6; 32 x 64 on 300 x 256 66, 86, 2 x 8 x 512 x 256 174, 129.  The sums of a score are then longer chains than a row's
// lanes make of them, and less exact than those until there are a few hundred keys (1.17e-7 and 1.11e-7 at 100 x 128, 1.67e-7 and
// 1.86e-7 on 300).
bool attention_f32_serves(const AttnArgs &a) {
  if (a.dtype != RAI_F32) return false;
  if (forced_waves()) return true;
  const int64_t rows = (int64_t)a.B * a.Hq * a.S;
  // (few rows of more keys than a row's block can hold stay with it: refused, unless a window makes them fewer)
  if (a.D <= 80 ? rows < 2048 && (a.T > 32768 || (a.T < 64 && rows <= 1024)) : rows < (a.D <= 128 ? 2048 : 8192) || a.T < (a.D <= 128 ? 256 : 512)) return false;
  return takes(a);
}

int launch_attention_f32(hipStream_t st, const AttnArgs &a) {
  RAI_REQUIRE(takes(a), RAI_ERR_UNSUPPORTED, "attention: RAI_HIP_ATTN_F32 does not apply to %d x %d x %d on %d keys", a.B, a.Hq, a.S, a.T);
  switch (a.D) {
    case 32: return launch_f32_split<32>(st, a);
    case 64: return launch_f32_split<64>(st, a);
    case 80: return launch_f32_split<80>(st, a);
    case 128: return launch_f32_split<128>(st, a);
    case 192: return launch_f32_split<192>(st, a);
    default: return launch_f32_split<256>(st, a);
  }
}

}  // namespace rai
