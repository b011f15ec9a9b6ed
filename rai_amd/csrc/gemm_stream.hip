// bf16 Linears of 5 to 32 rows (a batched decode step; one of 9 and more for weights in fragment order) by v_mfma_f32_16x16x32_bf16, on weights in fragment order or in rows as they lie.
#include "gemm_device.h"

namespace rai {

typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;

constexpr int kPastL2 = 17;   // cache policy bits sc0 and sc1: past the (per-XCD, mutually incoherent) L2s

// A block's eight waves take the K steps of 32 in turn (step 8 i + wave, i = 0 .. KS - 1; of rows as they lie, pairs of steps: whole lines) with the
// activations of theirs in registers for the whole launch; it walks over groups of G tiles of 16 weight rows, RT tiles on their way, and the eight partial sums of an output meet in LDS.
// K in parts (SPLIT): part s of n takes the eights of steps s, s + n, ...; a block has one group then, its tiles a grid apart, and two
// blocks share a CU.
// Bound by the stream of W behind a start (launch, activations, norm) and an end (the sums' way through LDS, with parts through memory) of some
// 5 us together.  The compiler's wait for a load that may not have been made counts none that follow: a residual asked for under a condition
// drained the ring at every group's start.  So nothing is loaded under a condition; rows beyond M and steps beyond K are those at the
// end once more.  Measured on weights from HBM, 24 rows, in a graph, against the kernel in gemm_mfma.hip, which is also bigger by its outputs of any
// alignment (us, it, this): 32768 x 2048 normed and gated 28.9, 24.8 (134 MB: 5.4 TB/s; a kernel that only reads them takes 21 to 23), plain 25.4,
// 23.5; 2560 x 2048 normed 9.9, 7.9; 2048 x 2048 with residual 6.6, 6.3; 2048 x 16384 in eight parts 19.5, 16.3; 17920 x 1536 normed and gated 21.1, 13.6;
// 1536 x 8960 in five parts 14.1, 10.2; 2048 x 1536 normed 9.1, 6.2.
// How the blocks' reads lie to each other counts as much: 2048 x 16384 took 21.4 with four neighbouring tiles to a block (each 512 KB), 17.2
// with two, 16.3 with four a grid apart, but 32768 x 2048 (tiles of 64 KB) 24.8 with two neighbours, 26.5 with two a grid apart, 29 with four neighbours; eights
// of steps of all tiles side by side 27.1.  A wave's steps in one piece instead of in turn: no difference.  Rows as they lie take some 13 %
// more than fragments.
// Registers: 128 at two blocks to a CU hold the activations, a tile and the sums of four, if nothing else is live then: uniform addresses, a load
// behind the multiply whose operand it replaces, first sums on a zero that takes none (with spills 2048 x 16384 took 20.2 us).
template <int MT, int KS, int G, bool FRAG, bool NORM, bool GLU, bool SPLIT, bool F32O>
__global__ void __launch_bounds__(512, SPLIT ? 4 : 2) k_linear_bf16_stream(LinearArgs a, int tiles, float *partial, int *tickets) {
  constexpr int NW = 8, RT = G < 2 || SPLIT ? 1 : 2, PCH = 4 * G + 1, ITEMS = MT * G * 64;
  static_assert(ITEMS <= 512 && !(F32O && (NORM || GLU)) && !(SPLIT && (NORM || GLU)), "a thread finishes one piece of a group");
  extern __shared__ __attribute__((aligned(16))) char stream_lds[];
  f32x4 *red = reinterpret_cast<f32x4 *>(stream_lds);                     // [NW][MT * 16 rows][PCH]
  float *squares = reinterpret_cast<float *>(red + NW * MT * 16 * PCH);   // [NW][MT * 16 rows]
  __shared__ int s_ticket;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lrow = lane & 15, lq = lane >> 4;
  const int parts = SPLIT ? gridDim.y : 1, part = SPLIT ? blockIdx.y : 0, ksteps = a.K / 32;
  constexpr int RUN = FRAG ? 1 : 2;   // neighbouring steps to a wave; all but the last run are within K
  static_assert(KS % RUN == 0, "whole runs");
  auto place = [&](int ks) { return ((ks / RUN * parts + part) * NW + wave) * RUN + ks % RUN; };
  auto beyond = [&](int ks) { return ks >= KS - RUN && place(ks) >= ksteps; };
  auto step_at = [&](int ks) { return beyond(ks) ? 0 : place(ks); };

  bf16x8 xf[MT][KS], wv[KS], w[RT][KS];
  const uint32_t lane_at = lane * 16;
  auto load = [&](bf16x8 &dst, int tile, int ks) __attribute__((always_inline)) {
    tile = tile < tiles ? tile : tiles - 1;
    if constexpr (FRAG) {   // one instruction reads 1 KB of consecutive memory
      const char *p = (const char *)a.Wfrag + ((int64_t)tile * ksteps + step_at(ks)) * 1024;
      dst = __builtin_nontemporal_load(reinterpret_cast<const bf16x8 *>(p + lane_at));
    } else {                // 64 bytes of sixteen rows, the second half of their lines with the next step: through the caches
      const char *p = (const char *)a.W + ((int64_t)tile * 16 * a.ldw + step_at(ks) * 32) * 2;
      const int rows = a.N - tile * 16;   // (addresses as a uniform part and 32 bits of a lane's own: no registers for pairs)
      dst = *reinterpret_cast<const bf16x8 *>(p + (uint32_t)((lrow < rows ? lrow : rows - 1) * (int)a.ldw + lq * 8) * 2u);
    }
  };
  const int stride = gridDim.x * G;
  auto tile_at = [&](int g0, int pos) { return SPLIT ? g0 + pos * (int)gridDim.x : pos < G ? g0 + pos : g0 + stride + pos - G; };
  int g0 = SPLIT ? blockIdx.x : blockIdx.x * G;
  // The activations first, which come from the L2 and are needed first (loads return in order), then the first tiles.
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int m = mt * 16 + lrow;
    const uint32_t row = (uint32_t)((m < a.M ? m : a.M - 1) * (int)a.lda + lq * 8) * 2u;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) xf[mt][ks] = *reinterpret_cast<const bf16x8 *>((const char *)a.A + step_at(ks) * 64 + row);
  }
  if constexpr (NORM) {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) wv[ks] = *reinterpret_cast<const bf16x8 *>((const char *)a.ln_w + step_at(ks) * 64 + lq * 16u);
  }
#pragma unroll
  for (int pos = 0; pos < RT; ++pos)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) load(w[pos][ks], tile_at(g0, pos), ks);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int ks = KS - RUN; ks < KS; ++ks)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
      if (beyond(ks)) xf[mt][ks] = bf16x8{};
  if constexpr (NORM) {
    // RMSNorm of the rows (ln_kind 1: x * w / rms, 2: x * (1 + w) / rms).  The fragments take the weight, in f32 and rounded once; the factor
    // 1 / rms is the finished sums', so that no wave waits for another's squares before it multiplies.  Every block norms all rows, so vector
    // instructions count: the squares are the diagonal of X X^T (lane (row, quarter) holds row 4 quarter + r of column `row`).
#pragma unroll
    for (int ks = KS - RUN; ks < KS; ++ks)
      if (beyond(ks)) wv[ks] = bf16x8{};   // an infinite weight would make the zeros NaN
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      f32x4 xx = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) xx = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf[mt][ks], xf[mt][ks], xx, 0, 0, 0);
      const float lo = lrow & 1 ? xx.y : xx.x, hi = lrow & 1 ? xx.w : xx.z;
      if (lq == lrow >> 2) squares[wave * (MT * 16) + mt * 16 + lrow] = lrow & 2 ? hi : lo;
    }
    const float one = a.ln_kind == 2 ? 1.f : 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float wf = (float)wv[ks][j] + one;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) xf[mt][ks][j] = (__bf16)((float)xf[mt][ks][j] * wf);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // what a thread finishes: four columns of row m, at column n of a group (ITEMS <= 512)
  const int lds_item = tid < ITEMS ? tid : 0;
  float scale = 1.f;
  // columns n .. n + 3 (N is a multiple of 4) and what is added to them
  auto word = [&](const void *p, int64_t at) { return *reinterpret_cast<const u32x2 *>(p ? (const char *)p + at * 2 : (const char *)a.A); };
  auto value = [&](const u32x2 &v, int e) { return bf16_bits_to_f32((uint16_t)((e < 2 ? v.x : v.y) >> (16 * (e & 1)))); };
  typedef std::conditional_t<F32O, f32x4, u32x2> Residual;
  auto residual = [&](int64_t at) {
    if constexpr (F32O) return *reinterpret_cast<const f32x4 *>(a.residual ? (const float *)a.residual + at : (const float *)a.A);
    else return word(a.residual, at);
  };
  auto finish = [&](int m, int n, f32x4 s, const u32x2 &bv, const u32x2 &bv2, const Residual &rv) __attribute__((always_inline)) {
    float x[4] = {s.x, s.y, s.z, s.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] += (a.bias ? value(bv, e) : 0.f) + (a.bias2 ? value(bv2, e) : 0.f);
    if constexpr (GLU) {   // (gate, up) pairs; gate, act(gate) and up each rounded, as glu_bf16
      float o[2];
      if (a.act == kActClampedGlu) {
#pragma unroll
        for (int e = 0; e < 2; ++e) o[e] = glu_clamped_bf16_out(x[2 * e], x[2 * e + 1], a.act_limit, a.act_alpha);
      } else {
        float g[2] = {bf16_bits_to_f32(f32_to_bf16_bits(x[0])), bf16_bits_to_f32(f32_to_bf16_bits(x[2]))};
        act_exact<2>(a.act, g, 0, 0);
#pragma unroll
        for (int e = 0; e < 2; ++e) o[e] = bf16_bits_to_f32(f32_to_bf16_bits(g[e])) * bf16_bits_to_f32(f32_to_bf16_bits(x[2 * e + 1]));
      }
      *reinterpret_cast<uint32_t *>((uint16_t *)a.out1 + (int64_t)m * a.ld1 + (n >> 1)) = pack_bf16x2(o[0], o[1]);
    } else {
      if (a.act >= 0) act_exact<4>(a.act, x, n, a.act_from);
      if constexpr (F32O) {
        f32x4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = fmaf(a.out_scale, x[e], a.residual ? rv[e] : 0.f);
        *reinterpret_cast<f32x4 *>((float *)a.out1 + (int64_t)m * a.ld1 + n) = o;
        return;
      } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (a.residual) x[e] += value(rv, e);
      uint16_t *dst = n < a.n_split ? (uint16_t *)a.out1 + (int64_t)m * a.ld1 + n : (uint16_t *)a.out2 + (int64_t)m * a.ld2 + (n - a.n_split);
      *reinterpret_cast<u32x2 *>(dst) = u32x2{pack_bf16x2(x[0], x[1]), pack_bf16x2(x[2], x[3])};
      }
    }
  };
  auto group = [&](auto last, const int g0, const bool first) __attribute__((always_inline)) {
    constexpr bool LAST = decltype(last)::value;   // nothing follows: no more loads
    f32x4 acc[G][MT];
    int item, m, c, n, n_in, m_in;
    auto whose = [&](int t) {
      item = t; m = t / (G * 4); c = t % (G * 4);
      n = (tile_at(g0, c >> 2) * 4 + (c & 3)) * 4;
      n_in = n < a.N ? n : 0;
      m_in = m < a.M ? m : 0;
    };
    u32x2 bv, bv2;
    Residual rv;
    if constexpr (!SPLIT) {   // on their way while the weights are
      whose(lds_item);
      bv = word(a.bias, n_in);
      bv2 = word(a.bias2, n_in);
      if (!GLU) rv = residual((int64_t)m_in * a.ldr + n_in);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < G; ++j)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[j][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[j % RT][ks], xf[mt][ks], ks ? acc[j][mt] : f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        if (!LAST || j + RT < G) load(w[j % RT][ks], tile_at(g0, j + RT), ks);   // (left alone, it would sink to just before its use)
        __builtin_amdgcn_sched_barrier(0);
      }
    if constexpr (SPLIT) {   // (not before: every register is taken)
      int t = lds_item;
      asm volatile("" : "+v"(t));
      whose(t);
    }
    // Parked as [row m][G tiles x 4 column quads], a pitch of an odd number of 16-byte chunks: the 16 lanes of a quad, a row each, hit
    // distinct banks; a thread then owns four consecutive columns of one row.
    if (!first) __syncthreads();   // the previous group's sums have been read
#pragma unroll
    for (int j = 0; j < G; ++j)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) red[(wave * MT * 16 + mt * 16 + lrow) * PCH + j * 4 + lq] = acc[j][mt];
    __syncthreads();
    f32x4 s4 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NW; ++w) s4 += red[(w * MT * 16 + m) * PCH + c];
    if constexpr (NORM) {
      if (first) {
        float tot = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) tot += squares[w * (MT * 16) + m];
        scale = 1.0f / sqrtf(tot / (float)a.K + a.ln_eps);
      }
      s4 *= scale;
    }
    const bool on = tid < ITEMS && m < a.M && n < a.N;
    if constexpr (!SPLIT) {
      if (on) finish(m, n, s4, bv, bv2, rv);
    } else {
      // A block counts itself in once its partial sums have reached memory (past the L2s), and the block that counts last, whichever it is,
      // adds all of them in the order of the parts and finishes.  Nobody waits.
      const int each = gridDim.x * ITEMS * 16;   // bytes of a part: [group][item]
      const auto ws = __builtin_amdgcn_make_buffer_rsrc(partial, 0, parts * each, 0x00020000);
      const int at = (blockIdx.x * ITEMS + item) * 16;
      if (on) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, s4), ws, at + part * each, 0, kPastL2);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (tid == 0) s_ticket = __hip_atomic_fetch_add(tickets + blockIdx.x, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __syncthreads();
      if (s_ticket != parts - 1) return;
      if (tid == 0) __hip_atomic_store(tickets + blockIdx.x, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // for the next launch
      if (!on) return;
      bv = word(a.bias, n_in);
      bv2 = word(a.bias2, n_in);
      rv = residual((int64_t)m_in * a.ldr + n_in);
      s4 = f32x4{0.f, 0.f, 0.f, 0.f};
      for (int sp = 0; sp < parts; sp += 8) {   // eight by one trip to memory
        f32x4 t[8];
#pragma unroll
        for (int i = 0; i < 8; ++i)
          t[i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(ws, at + (sp + i < parts ? sp + i : parts - 1) * each, 0, kPastL2));
#pragma unroll
        for (int i = 0; i < 8; ++i)
          if (sp + i < parts) s4 += t[i];
      }
      finish(m, n, s4, bv, bv2, rv);
    }
  };
  if constexpr (SPLIT) {
    group(std::integral_constant<bool, true>{}, g0, true);
  } else {
    bool first = true;
    for (; g0 + stride < tiles; g0 += stride, first = false) group(std::integral_constant<bool, false>{}, g0, first);
    group(std::integral_constant<bool, true>{}, g0, first);
  }
}

template <int MT, int KS, int G, bool FRAG, bool NORM, bool GLU, bool SPLIT, bool F32O>
static int launch_stream(hipStream_t st, const LinearArgs &a, int parts, int *tickets) {
  const int tiles = (a.N + 15) / 16, groups = (tiles + G - 1) / G;
  const size_t lds = (size_t)8 * MT * 16 * ((4 * G + 1) * sizeof(f32x4) + sizeof(float));
  static bool attr_set = false;
  if (lds > 64 * 1024 && !attr_set) {
    RAI_HIP_TRY(hipFuncSetAttribute((const void *)k_linear_bf16_stream<MT, KS, G, FRAG, NORM, GLU, SPLIT, F32O>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    attr_set = true;
  }
  hipLaunchKernelGGL((k_linear_bf16_stream<MT, KS, G, FRAG, NORM, GLU, SPLIT, F32O>), dim3(SPLIT || groups < kNumCU ? groups : kNumCU, parts), dim3(512), lds, st, a,
                     tiles, (float *)a.splitk_ws, tickets);
  return launch_check("linear_bf16_stream");
}
template <int MT, int KS, bool FRAG, bool F32O> static int launch_stream_form(hipStream_t st, const LinearArgs &a, int parts, int *tickets) {
  const int tiles = (a.N + 15) / 16;
  if constexpr (KS >= 6 && KS <= 8) {
    if (parts > 1) {   // one group to a block: as few tiles as two blocks to a CU allow
      if (tiles * parts <= kNumCU) return launch_stream<MT, KS, 1, FRAG, false, false, true, F32O>(st, a, parts, tickets);
      if (tiles * parts <= 2 * kNumCU) return launch_stream<MT, KS, 2, FRAG, false, false, true, F32O>(st, a, parts, tickets);
      return launch_stream<MT, KS, 4, FRAG, false, false, true, F32O>(st, a, parts, tickets);
    }
  }
  auto with = [&](auto g) -> int {
    constexpr int G = decltype(g)::value;
    if constexpr (!F32O) {
      if constexpr (FRAG && KS <= 8) {
        if (a.ln_kind > 0)
          return a.glu ? launch_stream<MT, KS, G, FRAG, true, true, false, false>(st, a, 1, nullptr) : launch_stream<MT, KS, G, FRAG, true, false, false, false>(st, a, 1, nullptr);
      }
      if (a.glu) return launch_stream<MT, KS, G, FRAG, false, true, false, false>(st, a, 1, nullptr);
    }
    return launch_stream<MT, KS, G, FRAG, false, false, false, F32O>(st, a, 1, nullptr);
  };
  return tiles <= kNumCU ? with(std::integral_constant<int, 1>{}) : with(std::integral_constant<int, 2>{});
}

// K steps to a wave: ten at most with K whole (eight with a norm, whose weight takes registers too), eight with K in parts, as few parts as that
// gives and the steps dealt out evenly (K = 1536 in six, 8960 in five parts of seven).
static int stream_parts(const LinearArgs &a) { return a.K <= (a.ln_kind > 0 ? 2048 : 2560) ? 1 : (a.K / 32 + 63) / 64; }
static size_t stream_parts_bytes(const LinearArgs &a) { return (size_t)stream_parts(a) * ((a.N + 63) / 64 * 64) * ((a.M + 15) / 16 * 16) * sizeof(float); }
// What it takes: whole pieces of four columns everywhere, K long enough for four steps a wave and, where K is cut, room for the parts; weights in rows as they lie without
// a norm or an f32 output, and not where the caller keeps to the other kernels' sums.
bool linear_stream_serves(const LinearArgs &a) {
  const int parts = stream_parts(a), piece = a.f32_out ? 16 : 8;
  auto whole = [](const void *p, int n) { return ((uintptr_t)p & (n - 1)) == 0; };
  if (a.M < 2 || a.M > 32 || a.K % 32 || a.K <= 24 * 32 || a.N % 4 || a.n_split % 4 || a.ln_kind == 0 || a.K2 || a.force_splits > 0) return false;
  if (a.Wfrag ? a.M <= 8 : a.fixed_sums || a.ln_kind > 0 || a.f32_out) return false;
  if ((a.ln_kind > 0 || a.glu) && (parts > 1 || a.f32_out)) return false;
  if (!a.Wfrag && (a.ldw % 8 || a.ldw >= 1 << 26 || !whole(a.W, 16))) return false;
  if (a.lda % 8 || a.lda >= 1 << 25 || !whole(a.A, 16) || (a.ln_kind > 0 && !whole(a.ln_w, 16))) return false;
  if (a.glu ? a.ld1 % 2 || !whole(a.out1, 4) : a.ld1 % 4 || !whole(a.out1, piece)) return false;
  if (a.n_split != a.N && (a.ld2 % 4 || !whole(a.out2, 8))) return false;
  if (!whole(a.bias, 8) || !whole(a.bias2, 8) || (a.residual && (a.ldr % 4 || !whole(a.residual, piece)))) return false;
  return parts == 1 || (a.splitk_ws && whole(a.splitk_ws, 16) && stream_parts_bytes(a) <= a.splitk_ws_bytes && stream_parts_bytes(a) < (1u << 31) &&
                        (a.N + 15) / 16 <= kSplitTickets);
}
// Where it is the fastest form.  On fragments it always is.  On rows as they lie, weights from HBM and, in brackets, from the caches
// where the two disagree: two to four rows are k_linear_bf16_rows's (4 x 8960 x 1536 8.3, 10.1; 4 x 4096 x 4096 9.5, 9.6), which at five to eight
// loses but for small matrices (8 x 2560 x 2048 7.9, 5.6; 8 x 16384 x 2048 21.0, 14.7; 8 x 1536 x 8960 12.2, 9.6; 8 x 512 x 1536 4.4, 4.5; 8 x
// 1024 x 4096 6.4, 6.7); 9 to 32 rows, against tiles and the kernel in gemm_mfma.hip: 16 x 2048 x 2048 7.1, 5.9; 16 x 4096 x 1024 7.0, 4.2; 32 x 8960 x
// 1536 14.6, 11.6; 24 x 2048 x 16384 22.7, 17.6; 24 x 16384 x 2048 19.0, 15.9 (12.5, 14.1); tiles keep wide matrices of ten steps a wave (24 x 10240 x
// 2560 19.5, 17.3 (12.9, 15.2)) and, beyond 16 rows, large ones in parts (32 x 8192 x 8192 36.4, 38.0 (25.7, 28.5)).
bool linear_stream_pays(const LinearArgs &a) {
  const char *off = getenv("RAI_HIP_NO_MFMA_STREAM"), *off2 = getenv("RAI_HIP_NO_MFMA_SKINNY");   // read per call: tests force the other kernels
  if (off || off2) return false;
  if (a.Wfrag) return true;
  const int64_t size = (int64_t)a.N * a.K;
  const bool parts = stream_parts(a) > 1;
  if (a.M <= 4) return false;
  if (a.M <= 8) return size >= (parts ? 8 << 20 : 3 << 19);
  return !(a.M > 16 && parts && size >= 48 << 20) && !(!parts && a.K > 2048 && a.N >= 9000);
}
size_t linear_stream_workspace_bytes(const LinearArgs &a) {
  return a.M > 4 && a.M <= 32 && a.K % 32 == 0 && stream_parts(a) > 1 && linear_stream_pays(a) ? stream_parts_bytes(a) : 0;
}
int launch_linear_bf16_stream(hipStream_t st, const LinearArgs &a) {
  const int parts = stream_parts(a), ks = (a.K / 32 + 8 * parts - 1) / (8 * parts);
  int *tickets = nullptr;
  if (parts > 1) {
    tickets = splitk_tickets(a);
    RAI_REQUIRE(tickets, RAI_ERR_HIP, "linear: the device's split counters were not found");
  }
  auto steps = [&](auto mt, auto f32o) -> int {
    constexpr int MT = decltype(mt)::value;
    constexpr bool F = decltype(f32o)::value;
    if (!a.Wfrag) {   // rows as they lie: pairs of steps
      if (ks > 8) return launch_stream_form<MT, 10, false, false>(st, a, parts, tickets);
      if (ks > 6) return launch_stream_form<MT, 8, false, false>(st, a, parts, tickets);
      return ks > 4 ? launch_stream_form<MT, 6, false, false>(st, a, parts, tickets) : launch_stream_form<MT, 4, false, false>(st, a, parts, tickets);
    }
    switch (ks) {
      case 10: return launch_stream_form<MT, 10, true, F>(st, a, parts, tickets);
      case 9: return launch_stream_form<MT, 9, true, F>(st, a, parts, tickets);
      case 8: return launch_stream_form<MT, 8, true, F>(st, a, parts, tickets);
      case 7: return launch_stream_form<MT, 7, true, F>(st, a, parts, tickets);
      case 6: return launch_stream_form<MT, 6, true, F>(st, a, parts, tickets);
      case 5: return launch_stream_form<MT, 5, true, F>(st, a, parts, tickets);
      default: return launch_stream_form<MT, 4, true, F>(st, a, parts, tickets);
    }
  };
  auto rows = [&](auto mt) -> int { return a.f32_out ? steps(mt, std::integral_constant<bool, true>{}) : steps(mt, std::integral_constant<bool, false>{}); };
  return a.M <= 16 ? rows(std::integral_constant<int, 1>{}) : rows(std::integral_constant<int, 2>{});
}

}  // namespace rai
