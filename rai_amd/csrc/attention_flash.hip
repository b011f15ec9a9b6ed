// Prefill attention in bf16 on the matrix instructions: the score matrix never exists in memory (the reference
// materialises [B, H, S, T]).
//
// Reference semantics: rai-models/src/llm/phi2.rs:244-262 (f32 scores and softmax, P cast to V's dtype), qwen2.rs:205-221 and
// gemma.rs:238-254 (scores and scale rounded to the model dtype), repeat_kv gemma.rs:191-201.
#include <cstdlib>

#include "attention.h"

namespace rai {

typedef __attribute__((ext_vector_type(8))) __bf16 fa_bf16x8;
typedef __attribute__((ext_vector_type(16))) float fa_f32x16;
typedef __attribute__((ext_vector_type(4))) uint32_t fa_u32x4;
typedef __attribute__((ext_vector_type(2))) uint32_t fa_u32x2;
typedef __attribute__((ext_vector_type(4))) short fa_s16x4;

// How rows of D features lie in LDS: unpadded, as the direct loads leave them, with the 16-byte chunk c of row r in place
// c ^ k_place(r) (K: a fragment read takes one chunk of 32 rows) or c ^ v_place(r) (V: a transposing read takes 64 bytes of each of
// four consecutive rows), so that a read's addresses spread over all banks.  KPAT, VPAT: the chunks and the 32-feature tiles
// after which the pattern repeats.
template <int D> struct FlashRows {
  static constexpr int CPR = D / 8, DT = (D + 31) / 32;
  static constexpr int KPAT = D % 128 == 0 ? 16 : D % 64 == 0 ? 8 : D == 32 ? 4 : 2, VPAT = D % 128 == 0 ? 4 : D % 64 == 0 ? 2 : 1;
  static __device__ __forceinline__ int k_place(int r) { return D % 128 == 0 ? r & 15 : D % 64 == 0 ? (r >> 1) & 7 : D == 32 ? (r >> 2) & 3 : (r >> 3) & 1; }
  static __device__ __forceinline__ int v_place(int r) { return D % 128 == 0 ? (r & 3) << 2 : D % 64 == 0 ? ((r >> 1) & 1) << 2 : 0; }
};

__device__ __forceinline__ float fa_round(float x) { return bf16_bits_to_f32(f32_to_bf16_bits(x)); }

// Block = NW * KSP waves, each owning 32 query rows; key tiles of TK keys pass through LDS and are shared by the waves.  Both
// products run on v_mfma_f32_32x32x16_bf16 in the transposed orientation
//     S^T = K . Q^T        (rows = keys, columns = queries)
//     O^T = V^T . P^T      (rows = head features, columns = queries)
// so every lane owns one query column: the online softmax's statistics are per-lane scalars, and the accumulator registers of S^T
// are, in order, the B-operand fragments of the second product.  K and V go to LDS by direct loads as they lie; V^T's
// fragments come out of the transposing LDS read.
//
// Two buffers each of K and V, one barrier a tile; the next tile's loads go out between this one's score products, the exponentials of
// sixteen keys beside the value products of the sixteen before.  Two waves to a SIMD (at 128 features), so that one's softmax also runs
// beside the other's products.  16 x 12 heads x 1024 x 128, causal: 81 us with rounded scores, 68 with f32 ones (149 and 136 with
// tiles through registers, V transposed on the way, two barriers a tile).  Of the clocks the matrix cores take 31 %, the vector
// units 35 %, the LDS less; what is left is waves waiting for one another's turn and the first and last rounds of a block.  A pipeline over
// tiles of 32 keys (scores of the next and values of the last tile beside one softmax) took 108 us: twice the barriers.
// KSP > 1: every 32-query group is worked on by KSP waves, which take every KSP-th key tile with a running maximum, sum and output of
// their own; merged through LDS at the end.  For few query rows, where a wave's chain of key tiles is what the launch takes.
// MODE: 0 scores rounded to bf16, 1 scores in f32, 2 scores in f32 with the cap and the sink of AttnArgs.
template <int NW, int D, int MODE, int KSP, int TK>
__global__ void __launch_bounds__(NW * KSP * 64, D <= 128 ? 2 : 1) k_flash_prefill_bf16(AttnArgs a) {
  typedef FlashRows<D> F;
  constexpr int KS = D / 16, DT = F::DT, CPR = F::CPR, U = TK / 32, NT = NW * KSP * 64;
  constexpr int TILE = TK * D;                   // elements of one K or V tile
  constexpr int CHUNKS = KSP * TK * CPR;         // 16-byte chunks of a round's K (or V) tiles
  constexpr int CH = (CHUNKS + NT - 1) / NT;
  extern __shared__ __attribute__((aligned(16))) uint16_t fa_smem[];
  uint16_t *const Kb = fa_smem, *const Vb = fa_smem + 2 * KSP * TILE;   // two buffers each
  typedef __attribute__((address_space(3))) void *lds_ptr;
  typedef __attribute__((address_space(3))) fa_s16x4 *tr_ptr;

  const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5, l32 = lane & 31;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wave = w / KSP, kh = w % KSP;   // query group of the block, key tiles kh, kh + KSP, ...
  // Under a causal mask the last query tiles see the most keys: those of all heads go first, so that the short ones fill the
  // tail.  Blocks go to the XCDs in turn, so an XCD takes a run of heads, whose keys then are in its L2 alone.
  const int heads = a.Hq * a.B, tiles = (a.S + NW * 32 - 1) / (NW * 32), id = (int)(blockIdx.y * gridDim.x + blockIdx.x);
  if (id >= tiles * heads) return;
  int hb, qt;
  if (heads % 8 == 0) {
    const int per = heads / 8, slot = id / 8;
    hb = id % 8 * per + slot % per;
    qt = tiles - 1 - slot / per;
  } else {
    hb = id % heads;
    qt = tiles - 1 - id / heads;
  }
  const int h = hb % a.Hq, b = hb / a.Hq, hk = h / (a.Hq / a.Hkv);
  const int q0 = qt * (NW * 32), qw = q0 + wave * 32;
  const int off = a.T - a.S;  // absolute position of query row 0
  const uint16_t *Kg = (const uint16_t *)a.k + b * a.ks[0] + hk * a.ks[1];
  const uint16_t *Vg = (const uint16_t *)a.v + b * a.vs[0] + hk * a.vs[1];

  int kv_end = a.T;
  if (a.causal) kv_end = min(off + min(q0 + NW * 32, a.S), a.T);
  // sliding window: the block's first query sets the oldest key tile any of its queries may see
  const int first_key = a.window > 0 ? off + q0 - a.window + 1 : 0;
  const int kv_begin = first_key > 0 ? first_key & ~63 : 0;
  const int wave_end = min(kv_end, a.causal ? off + qw + 32 : a.T);          // past the newest key any row of this wave may see
  const int wave_old = a.window > 0 ? off + qw - a.window + 1 : 0;           // the oldest
  const int rounds = kv_end > kv_begin ? (kv_end - kv_begin + KSP * TK - 1) / (KSP * TK) : 0;

  // This thread's chunks of a round's tiles.  Where a load instruction of the block moves whole periods of the placement, they differ
  // by a multiple of the row stride alone and one pointer serves them all.
  constexpr bool EVEN = NT % CPR == 0 && NT / CPR % 16 == 0;
  constexpr int NP = EVEN ? 1 : CH;
  const uint16_t *kp[NP], *vp[NP];
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int c = tid + i * NT, row = c / CPR, place = c % CPR;
    kp[i] = Kg + (int64_t)(kv_begin + row) * a.ks[2] + 8 * (place ^ F::k_place(row));
    vp[i] = Vg + (int64_t)(kv_begin + row) * a.vs[2] + 8 * (place ^ F::v_place(row));
  }
  // Load j of 2 CH of a round: K's, then V's.  `end`: rows past the context re-read its last row (masked below).
  auto load = [&](int j, int round, bool end, uint16_t *k_dst, uint16_t *v_dst) __attribute__((always_inline)) {
    const int i = j % CH;
    if (CHUNKS % NT != 0 && i * NT + w * 64 >= CHUNKS) return;
    const int64_t stride = j < CH ? a.ks[2] : a.vs[2];
    const uint16_t *base = j < CH ? kp[EVEN ? 0 : i] : vp[EVEN ? 0 : i], *src = EVEN ? base + i * (NT / CPR) * stride : base;
    if (end) src -= (int64_t)max(kv_begin + round * KSP * TK + (tid + i * NT) / CPR - (a.T - 1), 0) * stride;
    __builtin_amdgcn_global_load_lds((const void *)src, (lds_ptr)((j < CH ? k_dst : v_dst) + (i * NT + w * 64) * 8), 16, 0, 0);
  };
  auto advance = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      kp[i] += a.ks[2] * (KSP * TK);
      vp[i] += a.vs[2] * (KSP * TK);
    }
  };
  auto past_end = [&](int round) { return kv_begin + (round + 1) * KSP * TK > a.T; };
  auto landed = [&]() {   // every wave's loads, for every wave
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
  };
  if (rounds > 0) {
#pragma unroll
    for (int j = 0; j < 2 * CH; ++j) load(j, 0, past_end(0), Kb, Vb);
    advance();
  }

  const int qrow = qw + l32, q_abs = off + qrow;
  const uint16_t *qp = (const uint16_t *)a.q + b * a.qs[0] + h * a.qs[1] + (int64_t)min(qrow, a.S - 1) * a.qs[2] + half * 8;
  fa_bf16x8 qf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) qf[ks] = *reinterpret_cast<const fa_bf16x8 *>(qp + ks * 16);
  fa_f32x16 o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[dt][r] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;
  // Scaling keeps the order of scores (a negative scale's sign goes to the queries, and a scale of zero: a score of 0 x infinity or NaN
  // stays NaN), so the maximum is taken of the products as they are, and scaled alone.
  float scale = MODE == 0 ? fa_round(a.scale) : a.scale;
  if (scale <= 0.f) {
    const bool zero = scale == 0.f;
    scale = zero ? 1.f : -scale;
    auto turned = [&](uint32_t x) { return zero ? ((x & 0x7f80u) == 0x7f80u ? 0x7fc0u : 0u) : x ^ 0x8000u; };   // of one bf16
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      fa_u32x4 v = __builtin_bit_cast(fa_u32x4, qf[ks]);
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = turned(v[j] & 0xffffu) | turned(v[j] >> 16) << 16;
      qf[ks] = __builtin_bit_cast(fa_bf16x8, v);
    }
  }
  constexpr float kLog2e = 1.4426950408889634f;
  const bool capped = MODE == 2 && a.softcap > 0.f;
  const float cap_exp = capped ? 2.0f * kLog2e / a.softcap * scale : 0.f;
  const float to_exp = MODE == 0 || capped ? kLog2e : scale * kLog2e, to_score = MODE == 0 || capped ? 1.f : scale;
  auto score = [&](float x) {   // of a product
    if constexpr (MODE == 0) return fa_round(fa_round(x) * scale);   // the product and its scaling are each rounded to bf16
    else return x * to_score;
  };

  // this lane's place in a K tile by chunk pair and in a V tile by feature tile, the pattern's period only
  int k_lane[F::KPAT / 2], v_lane[F::VPAT];
#pragma unroll
  for (int j = 0; j < F::KPAT / 2; ++j) k_lane[j] = l32 * D + 8 * ((2 * j + half) ^ F::k_place(l32)) + kh * TILE;
  {
    // lanes a = 0..15 of a transposing read point at row a / 4, features 4 (a % 4) .. + 3 and receive feature a of the four rows
    const int i = lane & 15, row = 4 * half + (i >> 2);
#pragma unroll
    for (int j = 0; j < F::VPAT; ++j)
      v_lane[j] = row * D + 8 * ((4 * j + 2 * ((lane >> 4) & 1) + ((i & 3) >> 1)) ^ F::v_place(i >> 2)) + 4 * (i & 1) + kh * TILE;
  }

  struct Scores { fa_f32x16 u[U]; };
  // S^T tile: TK keys x 32 queries; register r of sub-tile u is key 32 u + 8 (r / 4) + 4 half + r % 4.  Fragments are read two steps
  // ahead; beside(ks) goes with a step's products.  (The fences keep the compiler from reading all fragments first, which takes more
  // registers than there are.)
  auto multiply = [&](const uint16_t *Kt, auto &&beside) __attribute__((always_inline)) {
    Scores s;
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int r = 0; r < 16; ++r) s.u[u][r] = 0.f;
    fa_bf16x8 kf[3][U];
    auto read = [&](int ks) {
#pragma unroll
      for (int u = 0; u < U; ++u)
        kf[ks % 3][u] = *reinterpret_cast<const fa_bf16x8 *>(Kt + k_lane[ks % (F::KPAT / 2)] + 8 * (2 * ks / F::KPAT * F::KPAT) + u * 32 * D);
    };
    read(0);
    read(1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      if (ks + 2 < KS) read(ks + 2);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < U; ++u) s.u[u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[ks % 3][u], qf[ks], s.u[u], 0, 0, 0);
      beside(ks);
      __builtin_amdgcn_sched_barrier(0);
    }
    return s;
  };
  auto mask = [&](Scores &s, int k0) {
    const int last_key = a.causal && q_abs < a.T - 1 ? q_abs : a.T - 1;   // newest key this lane's query may see
    const int rel = last_key - k0 - 4 * half;
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int r = 0; r < 16; ++r) s.u[u][r] = u * 32 + 8 * (r >> 2) + (r & 3) > rel ? -INFINITY : s.u[u][r];
    if (a.window > 0) {
      const int rel_lo = q_abs - a.window - k0 - 4 * half;   // newest key before this lane's window
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int r = 0; r < 16; ++r) s.u[u][r] = u * 32 + 8 * (r >> 2) + (r & 3) <= rel_lo ? -INFINITY : s.u[u][r];
    }
  };
  // m_run is the exponent every p, the running sum and the output are relative to; it need not be the maximum.  It is moved (and sum
  // and output rescaled) only when some query of the wave has met a score more than kLazy above its own: after the first tiles that
  // is rare, and the rescaling multiplies are skipped.  A p may then reach e^kLazy instead of 1: nothing to bf16 or f32.
  auto move_to = [&](const Scores &s) {
    constexpr float kLazy = 6.0f;
    float m[4 * U];   // short chains
#pragma unroll
    for (int c = 0; c < 4 * U; ++c) {
      const fa_f32x16 &x = s.u[c / 4];
      m[c] = fmaxf(x[4 * (c % 4)], x[4 * (c % 4) + 1]);
      asm("v_max3_f32 %0, %0, %1, %2" : "+v"(m[c]) : "v"(x[4 * (c % 4) + 2]), "v"(x[4 * (c % 4) + 3]));
    }
#pragma unroll
    for (int c = 0; c < 2 * U; c += 2) asm("v_max3_f32 %0, %0, %1, %2" : "+v"(m[c]) : "v"(m[c + 1]), "v"(m[2 * U + c]));
    float mx = m[0];
#pragma unroll
    for (int c = 2; c < 2 * U; c += 2) mx = fmaxf(mx, m[c]);
#pragma unroll
    for (int c = 1; c < 2 * U; c += 2) mx = fmaxf(mx, m[2 * U + c]);
    {
      typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;
      const u32x2 both = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
      mx = score(fmaxf(__uint_as_float(both[0]), __uint_as_float(both[1])));
    }
    if (__builtin_amdgcn_ballot_w64(mx > m_run + kLazy) == 0) return;   // (-inf + kLazy = -inf: the first tile moves)
    const float m_new = fmaxf(m_run, mx), m_safe = m_new == -INFINITY ? 0.f : m_new;
    const float alpha = __builtin_amdgcn_exp2f((m_run - m_safe) * kLog2e);
    l_run *= alpha;
    m_run = m_new;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[dt][r] *= alpha;
  };
  // p = exp(s - m_run), and O^T += V^T . P^T, sixteen keys at a time: the next sixteen's exponentials beside one's products
  auto weigh = [&](const Scores &s, const uint16_t *Vt) __attribute__((always_inline)) {
    fa_bf16x8 vf[2][DT];
    fa_u32x4 pw[2];
    auto read = [&](int g) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const uint16_t *at = Vt + v_lane[dt % F::VPAT] + 32 * (dt / F::VPAT * F::VPAT) + g * 16 * D;
        const fa_s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr)at);
        const fa_s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr)(at + 8 * D));
        const __attribute__((ext_vector_type(8))) short f = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        vf[g & 1][dt] = __builtin_bit_cast(fa_bf16x8, f);
      }
    };
    read(0);
    move_to(s);
    const float ml2 = (m_run == -INFINITY ? 0.f : m_run) * kLog2e;   // fully masked so far: every p is exp(-inf) = 0
    float sum = 0.f;
    auto pair = [&](int g, int j) {
      float x = s.u[g / 2][8 * (g % 2) + 2 * j], y = s.u[g / 2][8 * (g % 2) + 2 * j + 1];
      if constexpr (MODE == 0) {   // two scores per conversion
        uint32_t pk = pack_bf16x2(x, y);
        pk = pack_bf16x2(__uint_as_float(pk << 16) * scale, __uint_as_float(pk & 0xffff0000u) * scale);
        x = __uint_as_float(pk << 16);
        y = __uint_as_float(pk & 0xffff0000u);
      }
      const float p0 = __builtin_amdgcn_exp2f(fmaf(x, to_exp, -ml2)), p1 = __builtin_amdgcn_exp2f(fmaf(y, to_exp, -ml2));
      sum += p0 + p1;
      asm volatile("" : "+v"(sum));   // here, and not behind the products
      pw[g & 1][j] = pack_bf16x2(p0, p1);
    };
#pragma unroll
    for (int j = 0; j < 4; ++j) pair(0, j);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = 0; g < 2 * U; ++g) {
      if (g + 1 < 2 * U) read(g + 1);
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[g & 1][dt], __builtin_bit_cast(fa_bf16x8, pw[g & 1]), o[dt], 0, 0, 0);
        if (g + 1 < 2 * U) {
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (j * DT / 4 == dt) pair(g + 1, j);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    l_run += sum;
  };

  // some query of this wave sees a key of the tile at k0; some does not see all of it
  auto seen = [&](int k0) { return k0 < wave_end && k0 + TK > wave_old; };
  auto masked = [&](int k0) {
    return k0 + TK > a.T || (a.causal && k0 + TK - 1 > off + qw) || (a.window > 0 && k0 <= off + qw + 31 - a.window);
  };
  // One round: the next one's loads, then this one's products.  (The pointers do not alias: without being told so, the compiler waits for
  // the loads before it reads the tiles that are there.)
  auto step = [&](int round, uint16_t *__restrict__ next_k, uint16_t *__restrict__ next_v, const uint16_t *__restrict__ kt,
                  const uint16_t *__restrict__ vt) __attribute__((always_inline)) {
    // The loads go between the products one by one: all at once, the four waves' stand in each other's way (600 clocks of a tile's 3700)
    // and the wave with them.
    const int k0 = kv_begin + round * KSP * TK + kh * TK;
    const bool more = round + 1 < rounds, here = seen(k0);
    Scores s;
    if (more && here && !past_end(round + 1)) {
      s = multiply(kt, [&](int ks) {
#pragma unroll
        for (int j = 0; j < 2 * CH; ++j)
          if (j * KS / (2 * CH) == ks) load(j, round + 1, false, next_k, next_v);
      });
      advance();
    } else {
      if (more) {
#pragma unroll
        for (int j = 0; j < 2 * CH; ++j) load(j, round + 1, past_end(round + 1), next_k, next_v);
        advance();
      }
      if (!here) return;
      s = multiply(kt, [](int) {});
    }
    if (capped) {   // cap * tanh(s / cap) = cap - 2 cap / (exp(2 s / cap) + 1)
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          s.u[u][r] = fmaf(-2.0f * a.softcap, __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(s.u[u][r] * cap_exp)), a.softcap);
    }
    if (masked(k0)) mask(s, k0);
    weigh(s, vt);
  };
  for (int i = 0; i < rounds; ++i) {
    landed();   // this round's tiles, and everybody is done with the last one's
    const int cur = (i & 1) * KSP * TILE, next = ((i + 1) & 1) * KSP * TILE;
    step(i, Kb + next, Vb + next, Kb + cur, Vb + cur);
  }

  if constexpr (KSP > 1) {
    // the waves of key tiles 1 .. KSP-1 (mod KSP) hand their maximum, sum and output over; the wave of tiles 0 merges
    // and goes on alone
    __syncthreads();   // the tiles are no longer read
    constexpr int MS = (2 + DT * 16) * 64;   // floats a wave hands over: value by value, lane by lane
    float *mb = reinterpret_cast<float *>(fa_smem) + (size_t)wave * (KSP - 1) * MS + lane;
    if (kh > 0) {
      float *mine = mb + (kh - 1) * MS;
      mine[0] = m_run;
      mine[64] = l_run;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) mine[(2 + dt * 16 + r) * 64] = o[dt][r];
    }
    __syncthreads();
    if (kh > 0) return;
    float m = m_run;
#pragma unroll
    for (int j = 0; j < KSP - 1; ++j) m = fmaxf(m, mb[j * MS]);
    const float ms = m == -INFINITY ? 0.f : m;   // nothing seen by any of them: every weight is exp(-inf) = 0
    const float w0 = __builtin_amdgcn_exp2f((m_run - ms) * kLog2e);
    l_run *= w0;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[dt][r] *= w0;
#pragma unroll
    for (int j = 0; j < KSP - 1; ++j) {
      const float wj = __builtin_amdgcn_exp2f((mb[j * MS] - ms) * kLog2e);
      l_run += mb[j * MS + 64] * wj;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[dt][r] += mb[j * MS + (2 + dt * 16 + r) * 64] * wj;
    }
    m_run = ms;
  }
  float l_tot = l_run + __shfl_xor(l_run, 32, 64);
  if constexpr (MODE == 2) {
    if (a.sink) {   // relative to the running exponent, moved up to the sink's where that is larger by much
      const float sink = bf16_bits_to_f32(((const uint16_t *)a.sink)[h]), m = fmaxf(m_run, sink);
      const float ws = expf(m_run - m);
      l_tot = l_tot * ws + expf(sink - m);
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[dt][r] *= ws;
    }
  }
  if (qrow < a.S) {
    const float inv = l_tot > 0.f ? 1.0f / l_tot : 0.f;
    uint16_t *op = (uint16_t *)a.out + ((int64_t)b * a.S + qrow) * a.out_row_stride + (int64_t)h * D;
    const uint16_t *gp = a.gate ? (const uint16_t *)a.gate + ((int64_t)b * a.S + qrow) * a.gate_row_stride + (int64_t)h * D : nullptr;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int d = dt * 32 + 8 * g + 4 * half;
        if (d < D) {
          if (gp) {
            const fa_u32x2 gv = *reinterpret_cast<const fa_u32x2 *>(gp + d);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const uint32_t wd = e < 2 ? gv.x : gv.y;
              o[dt][4 * g + e] *= 1.0f / (1.0f + expf(-__uint_as_float(e & 1 ? wd & 0xffff0000u : wd << 16)));
            }
          }
          fa_u32x2 pk;
          pk.x = pack_bf16x2(o[dt][4 * g] * inv, o[dt][4 * g + 1] * inv);
          pk.y = pack_bf16x2(o[dt][4 * g + 2] * inv, o[dt][4 * g + 3] * inv);
          *reinterpret_cast<fa_u32x2 *>(op + d) = pk;
        }
      }
  }
}

template <int NW, int D, int MODE, int KSP, int TK> static int launch_flash_cfg(hipStream_t st, const AttnArgs &a) {
  // (64 elements more: the last feature tile of 80 reads past a tile's last row)
  constexpr size_t tiles = ((size_t)4 * KSP * TK * D + 64) * sizeof(uint16_t);
  constexpr size_t merge = (size_t)NW * (KSP - 1) * (2 + FlashRows<D>::DT * 16) * 64 * sizeof(float), lds = tiles > merge ? tiles : merge;
  static_assert(lds <= 160 * 1024, "LDS of a block");
  static bool attr_set = false;
  if (lds > 64 * 1024 && !attr_set) {
    RAI_HIP_TRY(hipFuncSetAttribute((const void *)k_flash_prefill_bf16<NW, D, MODE, KSP, TK>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    attr_set = true;
  }
  const int64_t blocks = (int64_t)((a.S + 32 * NW - 1) / (32 * NW)) * a.Hq * a.B;
  RAI_REQUIRE(blocks < 1 << 30, RAI_ERR_UNSUPPORTED, "attention: grid too large");   // (the output alone would be a terabyte)
  dim3 grid;
  RAI_TRY(grid_of_blocks(blocks, NW * KSP * 64, &grid));
  hipLaunchKernelGGL((k_flash_prefill_bf16<NW, D, MODE, KSP, TK>), grid, dim3(NW * KSP * 64), lds, st, a);
  return launch_check("flash_prefill");
}

// Waves to a query group and keys to a tile, by the groups there are.  More waves shorten a group's chain of key tiles while the CUs hold
// all blocks at once; tiles of 64 keys have half the barriers of tiles of 32, whose blocks fit a CU two or three times.  Measured,
// us, one wave and 64 keys / two and 32 / two and 64 / four and 32: 128 features, 512 x 512, 256 groups 15.3 / 12.7 / 11.4 / -, 512 groups
// 15.6 / 13.1 / 11.8, 1024 groups 16.3 / 14.3 / 18.0, 2048 groups 20.6 / 24.6 / 36; 80 features, 256 groups 12.6 / 10.5 / 9.0 / 8.3, 512
// groups 12.8 / 10.8 / 9.4 / 12.4, 1408 groups (333 x 333) 12.0 / 11.7 / 18.7, 2048 groups 15.7 / 18.2; 64 features, 512 groups 11.2 / 9.5 /
// 8.5 / 7.9, 1024 groups 11.6 / 9.8 / 9.4 / 13.1, 1600 groups (777 x 777) 15.9 / 14.5 / 17.1; 256 features, 512 groups 23.8 / 20.2, 1024
// groups 25.8 / 29.6.  A single tile of keys has nothing to share out.
// Beyond 128 features one wave with tiles of 32 keys (no register is left beside tiles of 64, one block to a CU) serves a
// single tile (256 features, 16 x 16: 6.8 for 8.1) and many groups of 192 (2816 groups, 333 x 333: 40 for 45).
template <int D, int MODE> static int launch_flash_mode(hipStream_t st, const AttnArgs &a) {
  const int64_t groups = (int64_t)((a.S + 31) / 32) * a.Hq * a.B;
  const int seen = a.window > 0 && a.window + 31 < a.T ? a.window + 31 : a.T;   // keys a group sees
  const char *no_split = getenv("RAI_HIP_FLASH_NO_KEY_SPLIT");   // read per call: tests compare both forms
  const bool split = seen > 64 && !(no_split && *no_split && *no_split != '0');
  if constexpr (D <= 128) {
    if constexpr (D <= 80) {
      if (split && groups <= (D <= 64 ? 2 : 1) * kNumCU) return launch_flash_cfg<1, D, MODE, 4, 32>(st, a);
    }
    if (split && groups <= (D <= 64 ? 4 : 2) * kNumCU) return launch_flash_cfg<2, D, MODE, 2, 64>(st, a);
    if (split && groups <= (D <= 80 ? 6 : 4) * kNumCU) return launch_flash_cfg<2, D, MODE, 2, 32>(st, a);
  } else {
    if (split && groups <= 2 * kNumCU) return launch_flash_cfg<2, D, MODE, 2, 32>(st, a);
    if (seen <= 64 || (D == 192 && groups >= 7 * kNumCU)) return launch_flash_cfg<4, D, MODE, 1, 32>(st, a);
  }
  return launch_flash_cfg<4, D, MODE, 1, 64>(st, a);
}
template <int D> static int launch_flash(hipStream_t st, const AttnArgs &a) {
  if (!a.f32_scores) return launch_flash_mode<D, 0>(st, a);
  return a.softcap > 0.f || a.sink ? launch_flash_mode<D, 2>(st, a) : launch_flash_mode<D, 1>(st, a);
}

bool flash_serves(const AttnArgs &a) {
  if (a.dtype != RAI_BF16 || a.S < 16 || a.t_dev) return false;
  if (a.D != 32 && a.D != 64 && a.D != 80 && a.D != 128 && a.D != 192 && a.D != 256) return false;
  if (a.gate && ((uintptr_t)a.gate % 8 || a.gate_row_stride % 4)) return false;
  auto al = [](const void *p, const int64_t *s) {
    return (uintptr_t)p % 16 == 0 && s[0] % 8 == 0 && s[1] % 8 == 0 && s[2] % 8 == 0;
  };
  return al(a.q, a.qs) && al(a.k, a.ks) && al(a.v, a.vs) && (uintptr_t)a.out % 8 == 0 && a.out_row_stride % 4 == 0 &&
         a.Hq <= 65535 && a.B <= 65535;
}

int launch_flash_prefill(hipStream_t st, const AttnArgs &a) {
  switch (a.D) {
    case 32: return launch_flash<32>(st, a);
    case 64: return launch_flash<64>(st, a);
    case 80: return launch_flash<80>(st, a);
    case 128: return launch_flash<128>(st, a);
    case 192: return launch_flash<192>(st, a);
    default: return launch_flash<256>(st, a);
  }
}

}  // namespace rai
