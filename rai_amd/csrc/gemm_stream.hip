// bf16 Linears of a batched decode step by v_mfma_f32_16x16x32_bf16: 9 to 32 rows on weights in fragment order, 5 to 32 on rows as they lie.
#include "gemm_device.h"

namespace rai {

typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;

constexpr int kPastL2 = 17;   // cache policy bits sc0 and sc1: past the (per-XCD, mutually incoherent) L2s

// A wave takes eight K steps of 32 with their activations in registers for the whole launch: NW waves to a block, as many as K has eights.  The block walks over
// groups of G tiles of 16 weight rows, RT tiles on their way, and the waves' partial sums of an output meet in LDS.  K beyond 2560 in parts of 64
// steps (SPLIT): a block has one group of one part then, its tiles a grid apart, and two blocks share a CU.
// On fragments a wave's steps are neighbours.  The order of every f32 sum and the one rounding of a normed activation are then those of
// k_linear_bf16_mfma_stream (gemm_mfma.hip), bit for bit, which a decoder's results rest on (LinearArgs::fixed_sums): steps dealt out otherwise, and the norm's
// factor on the finished sums, saved 0.3 to 1.5 us a launch and moved the logits of four layers of Gemma by 1 %, none of them nearer to the exact ones.
// On rows as they lie the waves take pairs of steps (whole lines) in turn: 8 rows x 16384 x 2048 14.3 us, in pieces 17.6.
// Bound by the stream of W behind a start (launch, activations, norm) and an end (the sums' way through LDS, with parts through memory) of some
// 5 us together.  The compiler's wait for a load that may not have been made counts none that follow: a residual asked for under a condition
// drained the ring at every group's start.  So nothing is loaded under a condition; rows beyond M are the last once more, steps beyond K are zeros.
// Measured on fragments from HBM, 24 rows, against the kernel in gemm_mfma.hip, which is also bigger by its outputs of any alignment (us, it, this):
// 32768 x 2048 normed and gated 28.9, 26.1 (134 MB: 5.1 TB/s; a kernel that only reads them takes 21 to 23); 2560 x 2048 normed 9.9, 9.0; 2048 x 2048
// with residual 6.6, 6.6; 2048 x 16384 in eight parts 19.5, 16.0; 17920 x 1536 normed and gated 21.1, 15.2; 1536 x 8960 in five parts 14.1, 10.4; 2048 x 1536
// normed 9.1, 7.9; Phi-2's 12800 x 2560 and 2560 x 12800 29.7 in the mean, 20.7 and 21.0.
// How the blocks' reads lie to each other counts as much: 2048 x 16384 took 21.4 with four neighbouring tiles to a block (each 512 KB), 17.2
// with two, 16.3 with four a grid apart, but 32768 x 2048 (tiles of 64 KB) 24.8 with two neighbours, 26.5 with two a grid apart, 29 with four neighbours.
// Registers: 128 at two blocks to a CU hold the activations, a tile and the sums of four, if nothing else is live then: uniform addresses, a load
// behind the multiply whose operand it replaces, first sums on a zero that takes none (with spills 2048 x 16384 took 20.2 us).  Beyond eight waves and 16
// rows one tile is on its way: of two, the second spills.
static __device__ u32x4 g_stream_zeros[64];   // never written

template <int MT, int NW, int G, bool FRAG, bool NORM, bool GLU, bool SPLIT, bool F32O>
__global__ void __launch_bounds__(64 * NW, SPLIT ? 4 : (NW + 3) / 4) k_linear_bf16_stream(LinearArgs a, int tiles, float *partial, int *tickets) {
  constexpr int KS = 8, RT = G < 2 || SPLIT || (NW > 8 && MT > 1) ? 1 : 2, PCH = 4 * G + 1, ITEMS = MT * G * 64;
  static_assert(ITEMS <= 64 * NW && !(F32O && (NORM || GLU)) && !(SPLIT && (NORM || GLU || NW != 8)), "a thread finishes one piece of a group");
  extern __shared__ __attribute__((aligned(16))) char stream_lds[];
  f32x4 *red = reinterpret_cast<f32x4 *>(stream_lds);                     // [NW][MT * 16 rows][PCH]
  float *squares = reinterpret_cast<float *>(red + NW * MT * 16 * PCH);   // [NW][MT * 16 rows]
  __shared__ int s_ticket;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lrow = lane & 15, lq = lane >> 4;
  const int parts = SPLIT ? gridDim.y : 1, part = SPLIT ? blockIdx.y : 0, ksteps = a.K / 32;
  auto place = [&](int ks) { return FRAG ? (part * NW + wave) * KS + ks : ((ks / 2 * parts + part) * NW + wave) * 2 + ks % 2; };
  constexpr int SURE = FRAG ? 0 : SPLIT ? 4 : 6;   // as many are within K wherever it ends
  auto within = [&](int ks) { return ks < SURE || place(ks) < ksteps; };
  auto step_at = [&](int ks) { return within(ks) ? place(ks) : 0; };
  // Beyond K both operands are zeros, or an infinity in one would make the other's NaN: activations by a mask, fragments from a page of them (for
  // nothing; a branch around the products cost 0.2 to 0.6 us a launch), rows as they lie, where only the last steps can be beyond, by a mask as well.
  bf16x8 xf[MT][KS], wv[KS], w[RT][KS];
  uint32_t kept[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) kept[ks] = within(ks) ? ~0u : 0u;
  auto keep = [&](bf16x8 v, int ks) { return ks < SURE ? v : __builtin_bit_cast(bf16x8, __builtin_bit_cast(u32x4, v) & kept[ks]); };
  const uint32_t lane_at = lane * 16;
  auto load = [&](bf16x8 &dst, int tile, int ks) __attribute__((always_inline)) {
    tile = tile < tiles ? tile : tiles - 1;
    if constexpr (FRAG) {   // one instruction reads 1 KB of consecutive memory
      const char *p = within(ks) ? (const char *)a.Wfrag + ((int64_t)tile * ksteps + place(ks)) * 1024 : (const char *)g_stream_zeros;
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
  for (int ks = SURE; ks < KS; ++ks) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) xf[mt][ks] = keep(xf[mt][ks], ks);
    if constexpr (NORM) wv[ks] = keep(wv[ks], ks);
  }
  if constexpr (NORM) {
    // RMSNorm of the rows (ln_kind 1: x * w / rms, 2: x * (1 + w) / rms): the sum of squares of a row is gathered from the waves that hold its pieces,
    // then every fragment is scaled and rounded once, as the stand-alone kernel does.  Every block norms all rows, so vector
    // instructions count: the squares are the diagonal of X X^T (lane (row, quarter) holds row 4 quarter + r of column `row`), and the weight is widened
    // ahead of the barrier that they wait for.
    f32x4 xx[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) xx[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) xx[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf[mt][ks], xf[mt][ks], xx[mt], 0, 0, 0);
    float wf[KS][8];
    const float one = a.ln_kind == 2 ? 1.f : 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        wf[ks][j] = (float)wv[ks][j] + one;
        asm volatile("" : "+v"(wf[ks][j]));
      }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const float lo = lrow & 1 ? xx[mt].y : xx[mt].x, hi = lrow & 1 ? xx[mt].w : xx[mt].z;
      if (lq == lrow >> 2) squares[wave * (MT * 16) + mt * 16 + lrow] = lrow & 2 ? hi : lo;
    }
    __syncthreads();
    float scale[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      float tot = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) tot += squares[w * (MT * 16) + mt * 16 + lrow];
      scale[mt] = 1.0f / sqrtf(tot / (float)a.K + a.ln_eps);
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
      for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) xf[mt][ks][j] = (__bf16)((float)xf[mt][ks][j] * scale[mt] * wf[ks][j]);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // what a thread finishes: four columns of row m, at column n of a group (ITEMS <= 512)
  const int lds_item = tid < ITEMS ? tid : 0;
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
        const bf16x8 wk = FRAG ? w[j % RT][ks] : keep(w[j % RT][ks], ks);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[j][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wk, xf[mt][ks], ks ? acc[j][mt] : f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
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
    for (int w = 0; w < 8 && w < NW; ++w) s4 += red[(w * MT * 16 + m) * PCH + c];
    if constexpr (NW > 8) {   // what a second part would hold
      f32x4 second = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 8; w < NW; ++w) second += red[(w * MT * 16 + m) * PCH + c];
      s4 += second;
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

template <int MT, int NW, int G, bool FRAG, bool NORM, bool GLU, bool SPLIT, bool F32O>
static int launch_stream(hipStream_t st, const LinearArgs &a, int parts, int *tickets) {
  const int tiles = (a.N + 15) / 16, groups = (tiles + G - 1) / G;
  const size_t lds = (size_t)NW * MT * 16 * ((4 * G + 1) * sizeof(f32x4) + sizeof(float));
  static bool attr_set = false;
  if (lds > 64 * 1024 && !attr_set) {
    RAI_HIP_TRY(hipFuncSetAttribute((const void *)k_linear_bf16_stream<MT, NW, G, FRAG, NORM, GLU, SPLIT, F32O>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    attr_set = true;
  }
  hipLaunchKernelGGL((k_linear_bf16_stream<MT, NW, G, FRAG, NORM, GLU, SPLIT, F32O>), dim3(SPLIT || groups < kNumCU ? groups : kNumCU, parts), dim3(64 * NW), lds, st, a,
                     tiles, (float *)a.splitk_ws, tickets);
  return launch_check("linear_bf16_stream");
}
template <int MT, bool FRAG, bool F32O> static int launch_stream_parts(hipStream_t st, const LinearArgs &a, int parts, int *tickets) {
  const int tiles = (a.N + 15) / 16;   // one group to a block: as few tiles as two blocks to a CU allow
  if (tiles * parts <= kNumCU) return launch_stream<MT, 8, 1, FRAG, false, false, true, F32O>(st, a, parts, tickets);
  if (tiles * parts <= 2 * kNumCU) return launch_stream<MT, 8, 2, FRAG, false, false, true, F32O>(st, a, parts, tickets);
  return launch_stream<MT, 8, 4, FRAG, false, false, true, F32O>(st, a, parts, tickets);
}
template <int MT, int NW, bool FRAG, bool F32O> static int launch_stream_whole(hipStream_t st, const LinearArgs &a) {
  auto with = [&](auto g) -> int {
    constexpr int G = decltype(g)::value;
    if constexpr (!F32O) {
      if constexpr (FRAG && NW <= 8) {
        if (a.ln_kind > 0) return a.glu ? launch_stream<MT, NW, G, true, true, true, false, false>(st, a, 1, nullptr) : launch_stream<MT, NW, G, true, true, false, false, false>(st, a, 1, nullptr);
      }
      if (a.glu) return launch_stream<MT, NW, G, FRAG, false, true, false, false>(st, a, 1, nullptr);
    }
    return launch_stream<MT, NW, G, FRAG, false, false, false, F32O>(st, a, 1, nullptr);
  };
  return (a.N + 15) / 16 <= kNumCU ? with(std::integral_constant<int, 1>{}) : with(std::integral_constant<int, 2>{});
}

// K whole up to ten eights of steps (eight with a norm, whose weight takes registers too), beyond that in parts of eight.
static int stream_parts(const LinearArgs &a) { return a.K <= 2560 ? 1 : (a.K + 2047) / 2048; }
static size_t stream_parts_bytes(const LinearArgs &a) { return (size_t)stream_parts(a) * ((a.N + 63) / 64 * 64) * ((a.M + 15) / 16 * 16) * sizeof(float); }
// What it takes: whole pieces of four columns everywhere, K of four eights of steps and more and, where K is cut, room for the parts; weights in rows as they lie without
// a norm or an f32 output, and not where the caller keeps to the other kernels' sums.
bool linear_stream_serves(const LinearArgs &a) {
  const int parts = stream_parts(a), piece = a.f32_out ? 16 : 8;
  auto whole = [](const void *p, int n) { return ((uintptr_t)p & (n - 1)) == 0; };
  if (a.M < 2 || a.M > 32 || a.K % 32 || a.K <= 3 * 256 || a.N % 4 || a.n_split % 4 || a.ln_kind == 0 || a.K2 || a.force_splits > 0) return false;
  // what the other kernels refuse is theirs to refuse
  if (a.N <= 0 || !a.A || !a.W || !a.out1 || a.n_split < 0 || a.n_split > a.N || (a.n_split != a.N && (!a.out2 || a.f32_out))) return false;
  if (a.glu && (a.act < 0 || a.residual || a.n_split != a.N || (a.M > 8 && a.N % 8))) return false;
  if (a.Wfrag ? a.M <= 8 : a.fixed_sums || a.ln_kind > 0 || a.f32_out) return false;
  if (a.ln_kind > 0 && (a.K > 2048 || a.f32_out)) return false;
  if (a.glu && (parts > 1 || a.f32_out)) return false;
  // fragments and a K that k_linear_bf16_mfma_stream cuts: without the scratch that it takes, k_linear_bf16_mfma_skinny has been the one to serve it
  if (a.Wfrag && a.K > 2048 && (!a.splitk_ws || (size_t)((a.K + 2047) / 2048) * a.M * a.N * sizeof(float) > a.splitk_ws_bytes)) return false;
  if (!a.Wfrag && (a.ldw % 8 || a.ldw >= 1 << 26 || !whole(a.W, 16))) return false;
  if (a.lda % 8 || a.lda >= 1 << 25 || !whole(a.A, 16) || (a.ln_kind > 0 && !whole(a.ln_w, 16))) return false;
  if (a.glu ? a.ld1 % 2 || !whole(a.out1, 4) : a.ld1 % 4 || !whole(a.out1, piece)) return false;
  if (a.n_split != a.N && (a.ld2 % 4 || !whole(a.out2, 8))) return false;
  if (!whole(a.bias, 8) || !whole(a.bias2, 8) || (a.residual && (a.ldr % 4 || !whole(a.residual, piece)))) return false;
  return parts == 1 || (a.splitk_ws && whole(a.splitk_ws, 16) && stream_parts_bytes(a) <= a.splitk_ws_bytes && stream_parts_bytes(a) < (1u << 31) &&
                        (a.N + 15) / 16 <= kSplitTickets);
}
// Where it is the fastest form.  On fragments it always is.  On rows as they lie, weights from HBM and, in brackets, from the caches
// where the two disagree (us): two to four rows are k_linear_bf16_rows's (4 x 8960 x 1536 8.3, 10.1; 4 x 4096 x 4096 9.5, 9.6), which at five to eight
// loses but for small matrices (8 x 2560 x 2048 8.1, 5.1; 8 x 16384 x 2048 21.1, 14.3; 8 x 1536 x 8960 12.2, 9.5; 8 x 512 x 1536 4.4, 4.5; 8 x
// 1024 x 4096 6.3, 6.7); 9 to 32 rows, against tiles and the kernel in gemm_mfma.hip: 16 x 2048 x 2048 6.9, 5.5; 16 x 4096 x 1024 7.0, 3.7; 32 x 8960 x
// 1536 14.2, 11.5; 24 x 2048 x 16384 22.7, 16.7; 24 x 16384 x 2048 18.1, 15.5 (12.4, 13.4); tiles keep wide matrices of more than eight waves (24 x 10240 x
// 2560 19.5, 17.3 (12.9, 15.2)) and, beyond 16 rows, large ones in parts (32 x 8192 x 8192 36.1, 38.0 (25.4, 28.5)).
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
  const int parts = stream_parts(a), waves = (a.K + 255) / 256;
  int *tickets = nullptr;
  if (parts > 1) {
    tickets = splitk_tickets(a);
    RAI_REQUIRE(tickets, RAI_ERR_HIP, "linear: the device's split counters were not found");
  }
  auto go = [&](auto mt, auto frag, auto f32o) -> int {
    constexpr int MT = decltype(mt)::value;
    constexpr bool FRAG = decltype(frag)::value, F = decltype(f32o)::value;
    if (parts > 1) return launch_stream_parts<MT, FRAG, F>(st, a, parts, tickets);
    switch (waves) {
      case 10: return launch_stream_whole<MT, 10, FRAG, F>(st, a);
      case 9: return launch_stream_whole<MT, 9, FRAG, F>(st, a);
      case 8: return launch_stream_whole<MT, 8, FRAG, F>(st, a);
      case 7: return launch_stream_whole<MT, 7, FRAG, F>(st, a);
      case 6: return launch_stream_whole<MT, 6, FRAG, F>(st, a);
      case 5: return launch_stream_whole<MT, 5, FRAG, F>(st, a);
      default: return launch_stream_whole<MT, 4, FRAG, F>(st, a);
    }
  };
  const std::integral_constant<bool, true> yes;
  const std::integral_constant<bool, false> no;
  auto rows = [&](auto mt) -> int { return !a.Wfrag ? go(mt, no, no) : a.f32_out ? go(mt, yes, yes) : go(mt, yes, no); };
  return a.M <= 16 ? rows(std::integral_constant<int, 1>{}) : rows(std::integral_constant<int, 2>{});
}

}  // namespace rai
