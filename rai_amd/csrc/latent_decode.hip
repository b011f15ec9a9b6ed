// The single-row step of a latent-attention decoder in bf16: the Linears of a layer in three launches around the
// absorbed attention (latent_attention.hip), each with what precedes it folded in.
//   k_latent_in    both norms of the f32 stream + [query latent | latent | gate] from the first, and from the second the
//                  gated MLP or the router; also the final norm + head
//   k_latent_mid   norm of the query latent + queries; norm of the latent + cache append; choice of the experts + the
//                  chosen experts' gated products on the scaled input
//   k_latent_down  o and down (or the chosen experts' downs) as one contraction per stream element, residual added in f32
// A wave streams R weight rows at a time with the activation vector in registers (as k_gemv_bf16_reg does), lane l
// holding positions l * 8 + 512 u.  k_latent_in's blocks (a CU each) prepare that vector once for their eight waves while the
// first weights fly, k_latent_mid's waves each by themselves.
// Bound by the weights' stream behind a start of some 3 us (launch, activations, norm).  Width 2048, us, with a block of four waves that
// each formed the norm and waited for the weights first (loads under masks are waited for where the mask ends), 6464 rows 9.9; 16384 gated
// 15.1; a head of 32768 24.0; [o | down] of 2048 x 10240 11.1; now 7.2, 13.1 (beside the delta step), 21.6, 8.7.
#include <cstdlib>

#include "latent_device.h"
#include "moe.h"

namespace rai {

template <int KC>
__global__ void __launch_bounds__(kRowThreads) k_latent_in(LatentInArgs a) {
  extern __shared__ __attribute__((aligned(16))) char in_lds[];
  latent_in_block<KC>(a, blockIdx.x, gridDim.x, in_lds);
}

// The expert of rank j among the logits, and its score (the choice of k_moe_route_ranked).
template <int N> __device__ __forceinline__ int nth_of(const float *z, int experts, int j, int lane, float *score) {
  float v[N];
  int rank[N], e = 0;
  float zj = 0.f;
  rank_experts<N>(z, experts, lane, v, rank);
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const unsigned long long hit = __ballot(rank[i] == j);
    if (hit) {   // exactly one lane of one i
      const int l = __ffsll(hit) - 1;
      e = 64 * i + l;
      zj = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v[i]), l));
    }
  }
  *score = router_score(zj);
  return __builtin_amdgcn_readfirstlane(e);
}
__device__ __forceinline__ int nth_expert(const float *z, int experts, int j, int lane, float *score) {
  if (experts <= 64) return nth_of<1>(z, experts, j, lane, score);
  if (experts <= 128) return nth_of<2>(z, experts, j, lane, score);
  return nth_of<4>(z, experts, j, lane, score);
}

// Gated rows [n0, n1) of one expert on score * h, to out[n / 2].
template <int KC>
__device__ __forceinline__ void expert_rows(const uint16_t *h, const uint16_t *W, int K, int n0, int n1, float score, int act, uint16_t *out, int lane) {
  ld_u32x4 xv[KC];
#pragma unroll
  for (int u = 0; u < KC; ++u)
    xv[u] = lane * 8 + u * 512 < K ? *reinterpret_cast<const ld_u32x4 *>(h + lane * 8 + u * 512) : ld_u32x4{0u, 0u, 0u, 0u};
  RowSet<KC, 2> rs;
  rs.load(W, K, n0, n1 - 1, K, lane);
#pragma unroll
  for (int u = 0; u < KC; ++u)
#pragma unroll
    for (int i = 0; i < 4; ++i) xv[u][i] = pack_bf16x2(score * lo_f32(xv[u][i]), score * hi_f32(xv[u][i]));
  stream_rows<KC>(rs, xv, W, K, n0, n1, K, lane, [&](int n, float v0, float v1) { out[n >> 1] = f32_to_bf16_bits(gated(act, v0, v1)); });
}

// Few rows: every (token, choice) slot is a product of its own, the expert's weights shared through the caches where two
// tokens chose it.
template <int KC>
__global__ void __launch_bounds__(256) k_moe_slots(MoeSlotsArgs a) {
  const int lane = threadIdx.x & 63;
  const int gw = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
  const int slot = gw / a.waves_e, n0 = (gw - slot * a.waves_e) * a.rows_per_wave, N = 2 * a.EFp;
  if (slot >= a.slots) return;
  const int n1 = n0 + a.rows_per_wave < N ? n0 + a.rows_per_wave : N;
  expert_rows<KC>((const uint16_t *)a.h + (int64_t)(slot / a.top) * a.ld, (const uint16_t *)a.We_gu + (int64_t)a.choice[slot] * a.gu_stride, a.Hp, n0, n1,
                  a.weight[slot], a.act, (uint16_t *)a.eact + (int64_t)slot * a.EFp, lane);
}

template <int KC>
__global__ void __launch_bounds__(256) k_latent_mid(LatentMidArgs a) {
  const int lane = threadIdx.x & 63;
  int gw = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
  const int total = a.waves_q + a.top * a.waves_e;
  if (gw > total) return;
  ld_u32x4 xv[KC];
  if (gw == total || gw < a.waves_q) {
    // one of the two latents, normalised: the last wave appends the cached one, the others take the query's
    const bool append = gw == total;
    const int n = append ? a.kv_rank : a.q_rank;
    const uint16_t *src = (const uint16_t *)a.dn + (append ? a.Qp : 0), *w = (const uint16_t *)(append ? a.c_w : a.q_w);
    ld_u32x4 wn[KC];
#pragma unroll
    for (int u = 0; u < KC; ++u) {
      const int k = lane * 8 + u * 512;
      xv[u] = wn[u] = ld_u32x4{0u, 0u, 0u, 0u};
      if (k < n) {   // ranks that are not multiples of 8 end inside a pack: the padding of dn is zero, the norm's guarded
        xv[u] = *reinterpret_cast<const ld_u32x4 *>(src + k);
        if (k + 8 <= n) wn[u] = *reinterpret_cast<const ld_u32x4 *>(w + k);
        else {
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (k + e < n) wn[u][e >> 1] |= (uint32_t)w[k + e] << (16 * (e & 1));
        }
      }
    }
    RowSet<KC, 2> rs;
    const int n0 = gw * a.rows_per_wave, n1 = n0 + a.rows_per_wave < a.Nq ? n0 + a.rows_per_wave : a.Nq;
    if (!append) rs.load((const uint16_t *)a.Wuq, a.Qp, n0, n1 - 1, a.Qp, lane);
    float q = 0.f;
#pragma unroll
    for (int u = 0; u < KC; ++u) q = ld_dot8(xv[u], xv[u], q);
    const float sc = 1.0f / sqrtf(wave_sum(q) / (float)n + a.eps);
#pragma unroll
    for (int u = 0; u < KC; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        xv[u][e] = pack_bf16x2(lo_f32(xv[u][e]) * sc * lo_f32(wn[u][e]), hi_f32(xv[u][e]) * sc * hi_f32(wn[u][e]));
    if (append) {
      uint16_t *dst = (uint16_t *)a.cache + (int64_t)a.state->pos * a.Rp;
#pragma unroll
      for (int u = 0; u < KC; ++u)
        if (lane * 8 + u * 512 < a.Rp) *reinterpret_cast<ld_u32x4 *>(dst + lane * 8 + u * 512) = xv[u];
      return;
    }
    stream_rows<KC>(rs, xv, (const uint16_t *)a.Wuq, a.Qp, n0, n1, a.Qp, lane, [&](int nn, float v0, float v1) {
      uint16_t *o = (uint16_t *)a.q + nn;
      o[0] = f32_to_bf16_bits(v0);
      if (nn + 1 < n1) o[1] = f32_to_bf16_bits(v1);
    });
    return;
  }
  gw -= a.waves_q;
  const int slot = gw / a.waves_e, n0 = (gw - slot * a.waves_e) * a.rows_per_wave, N = 2 * a.EFp;
  const int n1 = n0 + a.rows_per_wave < N ? n0 + a.rows_per_wave : N;
  float score;
  const int e = nth_expert(a.rlogits, a.experts, slot, lane, &score);
  if (n0 == 0 && lane == 0) a.choice[slot] = e;
  expert_rows<KC>((const uint16_t *)a.h2, (const uint16_t *)a.We_gu + (int64_t)e * a.gu_stride, a.Hp, n0, n1, score, a.act,
                  (uint16_t *)a.eact + (int64_t)slot * a.EFp, lane);
}

// Chunks of up to 512 columns of the concatenated contraction: where the weights of row 0 are, the row stride, where the
// activations sit in LDS and how many columns there are.
struct DownChunk {
  const uint16_t *w;
  int ld;
  int meta;   // LDS offset | columns << 20
};

// A block of eight waves shares one copy of the activations; a wave owns one output row and has Q chunks in flight, each
// replaced by the chunk Q places on as soon as it has been multiplied.  Without experts (EX false) a row is one run of K0 columns and
// needs no table.  Every lane and every place in flight asks for something, where there is nothing for the row's first piece: a load
// under a mask is waited for where the mask ends, and loads that may not have been made cannot be counted.
constexpr int kDownWaves = 8, kDownThreads = kDownWaves * 64;
template <int Q, bool EX>
__global__ void __launch_bounds__(kDownThreads) k_latent_down(LatentDownArgs a) {
  extern __shared__ __attribute__((aligned(16))) char dn_lds[];
  typedef const __attribute__((address_space(1))) ld_u32x4 *weights;   // (a pointer out of LDS would be a flat one)
  const int tid = threadIdx.x, lane = tid & 63;
  {   // this block's row
    const int64_t m = blockIdx.y;
    a.x0 = (const uint16_t *)a.x0 + m * a.K0;
    a.x1 = (const uint16_t *)a.x1 + m * a.top * a.K1;
    if (EX) a.choice += m * a.top;
    a.res = a.res_f32 ? (const void *)((const float *)a.res + m * a.N) : (const void *)((const uint16_t *)a.res + m * a.H);
    a.out += m * a.N;
  }
  const int c0 = (a.K0 + 511) / 512, c1 = EX ? (a.K1 + 511) / 512 : 0, chunks = EX ? c0 + a.top * c1 : c0;
  const int Kt = EX ? a.K0 + a.top * a.K1 : a.K0;
  DownChunk *table = reinterpret_cast<DownChunk *>(dn_lds);
  uint16_t *xs = reinterpret_cast<uint16_t *>(table + (EX ? chunks : 0));
  const int n = __builtin_amdgcn_readfirstlane(blockIdx.x * kDownWaves + (tid >> 6));
  const int64_t row = n < a.N ? n : a.N - 1;
  if constexpr (EX) {
    for (int c = tid; c < chunks; c += kDownThreads) {
      DownChunk d;
      if (c < c0) {
        d.w = (const uint16_t *)a.W0 + c * 512;
        d.ld = a.K0;
        d.meta = (c * 512) | ((a.K0 - c * 512 < 512 ? a.K0 - c * 512 : 512) << 20);
      } else {
        const int j = (c - c0) / c1, i = (c - c0) - j * c1;
        d.w = (const uint16_t *)a.W1 + (int64_t)a.choice[j] * a.stride1 + i * 512;
        d.ld = a.K1;
        d.meta = (a.K0 + j * a.K1 + i * 512) | ((a.K1 - i * 512 < 512 ? a.K1 - i * 512 : 512) << 20);
      }
      table[c] = d;
    }
    __syncthreads();
  }
  // rows start where chunks do: each wave begins its own at another, so that together they ask all of the HBM's channels
  const int turn = n % chunks;
  auto place = [&](int c) { return (c + turn < chunks ? c + turn : c + turn - chunks) * 512; };
  ld_u32x4 w[Q];
  auto request = [&](ld_u32x4 &dst, int c) {
    if constexpr (EX) {
      const DownChunk d = table[c < chunks ? c : 0];
      dst = __builtin_nontemporal_load((weights)(d.w + row * d.ld + (c < chunks && lane * 8 < (d.meta >> 20) ? lane * 8 : 0)));
    } else {
      const int at = place(c);
      dst = __builtin_nontemporal_load((weights)((const uint16_t *)a.W0 + row * a.K0 + (c < chunks && at + lane * 8 < a.K0 ? at + lane * 8 : 0)));
    }
  };
  // the residual and the activations come from the L2 and are asked for first; the latter reach LDS while the weights are on their way
  const int64_t rat = n < a.H ? n : 0;
  uint32_t rraw;
  if (a.res_f32) rraw = ((const uint32_t *)a.res)[rat];
  else rraw = ((const uint16_t *)a.res)[rat];
  constexpr int XP = 3;
  ld_u32x4 xp[XP];
  auto x_at = [&](int k) { return *reinterpret_cast<const ld_u32x4 *>(!EX || k < a.K0 ? (const uint16_t *)a.x0 + k : (const uint16_t *)a.x1 + (k - a.K0)); };
#pragma unroll
  for (int i = 0; i < XP; ++i) xp[i] = x_at((tid + i * kDownThreads) * 8 < Kt ? (tid + i * kDownThreads) * 8 : 0);
#pragma unroll
  for (int u = 0; u < Q; ++u) {
    request(w[u], u);
    if (EX && u % 4 == 3) __builtin_amdgcn_sched_barrier(0);   // (with everything at hand at once registers run out)
  }
#pragma unroll
  for (int i = 0; i < XP; ++i)
    if ((tid + i * kDownThreads) * 8 < Kt) *reinterpret_cast<ld_u32x4 *>(xs + (tid + i * kDownThreads) * 8) = xp[i];
  for (int k = (tid + XP * kDownThreads) * 8; k < Kt; k += kDownThreads * 8) *reinterpret_cast<ld_u32x4 *>(xs + k) = x_at(k);
  __syncthreads();
  float acc = 0.f;
  auto multiply = [&](const ld_u32x4 &w, int c) {   // (a chunk's last lanes may have nothing)
    int at = place(c), cols = a.K0 - at;
    if constexpr (EX) {
      const int meta = table[c < chunks ? c : 0].meta;
      at = meta & 0xfffff;
      cols = meta >> 20;
    }
    const bool some = c < chunks && lane * 8 < cols;
    const ld_u32x4 x = *reinterpret_cast<const ld_u32x4 *>(xs + (some ? at + lane * 8 : 0)), zero = {0u, 0u, 0u, 0u};
    acc = ld_dot8(some ? w : zero, some ? x : zero, acc);
  };
  int first = 0;
  for (; first + Q < chunks; first += Q) {
#pragma unroll
    for (int u = 0; u < Q; ++u) {
      multiply(w[u], first + u);
      request(w[u], first + Q + u);
      if (u % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int u = 0; u < Q; ++u) {
    multiply(w[u], first + u);
    if (u % 4 == 3) __builtin_amdgcn_sched_barrier(0);
  }
  acc = wave_sum(acc);
  float res = a.res_f32 ? __uint_as_float(rraw) : __uint_as_float(rraw << 16);
  if (a.res_scale != 0.f) res *= a.res_scale;
  if (lane == 0 && n < a.N) a.out[n] = n < a.H ? fmaf(a.mult, acc, res) : 0.f;
}

// ---------------------------------------------------------------- launchers
bool latent_single_row_serves(int width, int groups, int max_rank, int max_experts, int64_t down_columns) {
  const char *off = getenv("RAI_HIP_NO_LATENT_FUSED");   // read per call: the tests compare both forms in one process
  if (off && *off && *off != '0') return false;
  return width % 8 == 0 && width <= 4096 && groups <= 16 && (width / groups) % 8 == 0 && max_rank <= 4096 && max_experts <= kRankedExperts && down_columns * 2 + 16 * 1024 <= 150 * 1024;
}

int latent_in_blocks(const LatentInArgs &a, int cus) {
  const int pairs = (a.N1 + 1) / 2 + (a.N2 + 1) / 2, blocks = (pairs + kRowWaves - 1) / kRowWaves;
  return blocks < cus ? blocks : cus;
}
int launch_latent_in(hipStream_t st, const LatentInArgs &a) {
  RAI_REQUIRE(a.groups <= kRowGroups && a.K <= 8 * kRowThreads, RAI_ERR_UNSUPPORTED, "latent in: %d groups, %d columns", a.groups, a.K);
  const dim3 grid(latent_in_blocks(a, kNumCU)), block(kRowThreads);
  const size_t lds = latent_in_lds(a);
  if (a.K <= 512) hipLaunchKernelGGL(k_latent_in<1>, grid, block, lds, st, a);
  else if (a.K <= 1024) hipLaunchKernelGGL(k_latent_in<2>, grid, block, lds, st, a);
  else if (a.K <= 2048) hipLaunchKernelGGL(k_latent_in<4>, grid, block, lds, st, a);
  else if (a.K <= 2560) hipLaunchKernelGGL(k_latent_in<5>, grid, block, lds, st, a);
  else hipLaunchKernelGGL(k_latent_in<8>, grid, block, lds, st, a);
  return launch_check("latent_in");
}

int launch_latent_mid(hipStream_t st, LatentMidArgs a) {
  const int rows = a.Nq + a.top * 2 * a.EFp;
  int rpw = (rows + kNumCU * 16 - 1) / (kNumCU * 16);
  a.rows_per_wave = rpw < 2 ? 2 : (rpw + 1) / 2 * 2;
  a.waves_q = (a.Nq + a.rows_per_wave - 1) / a.rows_per_wave;
  a.waves_e = a.top ? (2 * a.EFp + a.rows_per_wave - 1) / a.rows_per_wave : 1;
  const int waves = a.waves_q + a.top * a.waves_e + 1;
  int K = a.Qp > a.Rp ? a.Qp : a.Rp;
  if (a.top && a.Hp > K) K = a.Hp;
  const dim3 grid((waves + 3) / 4), block(256);
  if (K <= 512) hipLaunchKernelGGL(k_latent_mid<1>, grid, block, 0, st, a);
  else if (K <= 1024) hipLaunchKernelGGL(k_latent_mid<2>, grid, block, 0, st, a);
  else if (K <= 2048) hipLaunchKernelGGL(k_latent_mid<4>, grid, block, 0, st, a);
  else if (K <= 2560) hipLaunchKernelGGL(k_latent_mid<5>, grid, block, 0, st, a);
  else hipLaunchKernelGGL(k_latent_mid<8>, grid, block, 0, st, a);
  return launch_check("latent_mid");
}

bool moe_slots_serves(int64_t slots, int experts, int Hp, int top, int EFp) {
  const char *off = getenv("RAI_HIP_NO_LATENT_FUSED");   // read per call: the tests compare both forms in one process
  if (off && *off && *off != '0') return false;
  // more slots than experts: several tokens share an expert, whose weights the grouped tiles read once
  return slots <= 64 && slots <= experts && Hp <= 4096 && (int64_t)top * EFp * 2 + 16 * 1024 <= 150 * 1024;
}
int launch_moe_slots(hipStream_t st, MoeSlotsArgs a) {
  int rpw = (a.slots * 2 * a.EFp + kNumCU * 16 - 1) / (kNumCU * 16);
  a.rows_per_wave = rpw < 2 ? 2 : (rpw + 1) / 2 * 2;
  a.waves_e = (2 * a.EFp + a.rows_per_wave - 1) / a.rows_per_wave;
  const dim3 grid((a.slots * a.waves_e + 3) / 4), block(256);
  if (a.Hp <= 512) hipLaunchKernelGGL(k_moe_slots<1>, grid, block, 0, st, a);
  else if (a.Hp <= 1024) hipLaunchKernelGGL(k_moe_slots<2>, grid, block, 0, st, a);
  else if (a.Hp <= 2048) hipLaunchKernelGGL(k_moe_slots<4>, grid, block, 0, st, a);
  else if (a.Hp <= 2560) hipLaunchKernelGGL(k_moe_slots<5>, grid, block, 0, st, a);
  else hipLaunchKernelGGL(k_moe_slots<8>, grid, block, 0, st, a);
  return launch_check("moe_slots");
}

template <int Q, bool EX> static int launch_latent_down_q(hipStream_t st, const LatentDownArgs &a, size_t lds) {
  static bool attr_set = false;
  if (!attr_set) {
    RAI_HIP_TRY(hipFuncSetAttribute((const void *)k_latent_down<Q, EX>, hipFuncAttributeMaxDynamicSharedMemorySize, 150 * 1024));
    attr_set = true;
  }
  hipLaunchKernelGGL((k_latent_down<Q, EX>), dim3((a.N + kDownWaves - 1) / kDownWaves, a.rows), dim3(kDownThreads), lds, st, a);
  return launch_check("latent_down");
}
template <bool EX> static int launch_latent_down_e(hipStream_t st, const LatentDownArgs &a, int chunks, size_t lds) {
  if (chunks <= 8) return launch_latent_down_q<8, EX>(st, a, lds);
  // (chunks on their way at 2048 x 10240, us: 20 9.9, 16 10.6, 12 9.5, 10 8.8, 7 8.8, 5 8.7, 4 8.8)
  return launch_latent_down_q<EX ? 16 : 5, EX>(st, a, lds);
}
int launch_latent_down(hipStream_t st, const LatentDownArgs &a) {
  const int chunks = (a.K0 + 511) / 512 + a.top * ((a.K1 + 511) / 512);
  const size_t lds = (size_t)chunks * sizeof(DownChunk) + ((size_t)a.K0 + (size_t)a.top * a.K1) * 2;
  RAI_REQUIRE(lds <= 150 * 1024 && a.K0 % 8 == 0 && a.K1 % 8 == 0, RAI_ERR_UNSUPPORTED, "latent down: %d + %d x %d columns", a.K0, a.top, a.K1);
  return a.top ? launch_latent_down_e<true>(st, a, chunks, lds) : launch_latent_down_e<false>(st, a, chunks, lds);
}

}  // namespace rai
