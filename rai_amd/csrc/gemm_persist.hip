// The 256 x 256 tiles of a bf16 Linear by one block per CU that goes from tile to tile without letting its pipeline run
// empty.
//
// A block's work is one sequence of K stages of 64 across all of its tiles: a buffer that is let go is filled with the stage
// after the next, whichever tile that is in.  So the first stages of a tile arrive while the one before is multiplied and
// written, where a block per tile starts each with a trip to memory, and the outputs leave through LDS of their own (4 KB a
// wave behind the two 64 KB stages, all of the CU's 160 KB) beside those loads.
//
// What bounds it: with operands as they come (normal, not zero) the chip's power, 1.8 GHz of 2.4 at 16384 x 16384 x 1536, and LDS
// bandwidth: a stage's fragment reads and incoming tiles take the 2048 clocks that its multiplies take.  16 x 16 x 32 MFMAs
// instead of 32 x 32 x 16 move a fifth fewer bits per flop through the registers (registers alone, random operands:
// 2021, 1797 TFLOP/s; here 656 us, 684).  Measured, with a block per tile / so: 16384 x 16384 x 1536 757, 654 us; x 256 268, 194;
// 16384 x 17920 x 1536 gated silu 850, 733; 4096 x 16384 x 2560 new_gelu 313, 273.
// Not taken: four waves of 128 x 128 (two thirds of the LDS reads, but one wave a SIMD stalls on its own loads: 788 us), one
// barrier a stage with reads, loads and multiplies mixed in each wave (32 x 32 x 16: 684, 16 x 16 x 32: 668 to 690).
#include "gemm_device.h"

namespace rai {
namespace {

constexpr int kTileDim = 256, kStageK = 64, kWaves = 8, kThreads = 64 * kWaves;
constexpr int kWM = 128, kWN = kPersistColumns, kMT = kWM / 16, kNT = kWN / 16;   // a wave's part of the tile, waves 2 x 4, in 16 x 16 pieces
constexpr int kLoads = kTileDim / (8 * kWaves);                     // per wave, stage and operand: 8 rows of 128 bytes each
constexpr int kStageElems = 2 * kTileDim * kStageK;
constexpr int kStagingFloats = 16 * kWN;                            // a wave's 16 rows of outputs
constexpr size_t kLdsBytes = 2 * kStageElems * sizeof(uint16_t) + kWaves * kStagingFloats * sizeof(float);
typedef f32x4 (&Acc)[kMT][kNT];
typedef __attribute__((address_space(3))) void *lds_ptr;

// The lane, worked out anew wherever a tile begins or ends: what is derived from it there, held through the multiplies, spills.
__device__ __forceinline__ int lane_again() {
  int lane;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(lane));
  return lane;
}

// What a block does next: K stages k0 .. k0 + n - 1 of a tile.  Shares of the stream-K tiles first, then its whole tiles.
struct Segment { int tile, k0, n; };
struct Walk {
  int u, u_end, whole, whole_end, step, stages;
  __device__ __forceinline__ bool next(Segment &s) {
    if (u < u_end) {
      s.tile = u / stages;
      s.k0 = u - s.tile * stages;
      s.n = s.k0 + (u_end - u) < stages ? u_end - u : stages - s.k0;
      u += s.n;
      return true;
    }
    if (whole >= whole_end) return false;
    s = {whole, 0, stages};
    whole += step;
    return true;
  }
};

// ---- outputs
// The weights are the A operand, so accumulator register r of lane l is out[l % 16][4 (l / 16) + r] of its 16 x 16 piece:
// four neighbouring columns of a row in four registers.  Bias and activation are applied there, the rounded results are
// put into the wave's own LDS eight bytes at a time and leave it as 16 bytes of a row.
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;

// The fast forms, where gemm_persist_plain() holds; the rest goes row by row through store_row8.
enum { kRows, kPlain, kPlainResidual };

// The wave's 64 biases, or the first 32 rows of its residual, go to its staging area a stage before the outputs are written:
// ahead of the loads of the next tile, behind which they would wait.
__device__ __forceinline__ const uint16_t *residual_piece(const LinearArgs &a, int m, int n) {
  m = m < a.M ? m : a.M - 1;
  n = n < a.N ? n : 0;
  return (const uint16_t *)a.residual + (int64_t)m * a.ldr + n;
}
__device__ __forceinline__ void ask_for(const LinearArgs &a, char *staging, int m0, int n0) {
  const int lane = lane_again();
  if (a.bias) {
    const int n = n0 + 2 * (lane & 31);
    __builtin_amdgcn_global_load_lds((const void *)((const uint16_t *)a.bias + (n < a.N ? n : 0)), (lds_ptr)staging, 4, 0, 0);
  } else if (a.residual) {
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const int r = p * 8 + (lane >> 3);
      __builtin_amdgcn_global_load_lds((const void *)residual_piece(a, m0 + r, n0 + ((lane & 7) ^ ((r >> 1) & 7)) * 8), (lds_ptr)(staging + p * 1024), 16, 0, 0);
    }
  }
}

// 32 rows at a time: 128 bytes a row in LDS (64 with a gated activation), 16-byte chunk c of row r at c ^ ((r >> 1) & 7)
// (c ^ ((r >> 2) & 3)): the writes, a column of 16 rows, and the 16-byte reads, whole rows, each spread over all banks.
// Stores past the caches (nontemporal) where rows begin on 64-byte boundaries: outputs that stay in the L2s push the operand
// panels out that their tiles share there (16384 x 16384 x 1536: 727 us, so 685).  Elsewhere the L2 puts the pieces of a line
// together first (13563 x 9224 x 192: past it 136 us, 88 through it).
__device__ __forceinline__ bool whole_pieces(const void *out, int64_t ld) { return ((uintptr_t)out & 63) == 0 && ld % 32 == 0; }
__device__ __forceinline__ void store_rows(uint16_t *p, u32x4 x, bool past) {
  if (past) __builtin_nontemporal_store(x, reinterpret_cast<u32x4 *>(p));
  else *reinterpret_cast<u32x4 *>(p) = x;
}

__device__ __forceinline__ void write_plain(const LinearArgs &a, Acc acc, char *staging, int m0, int n0) {
  const int lane = lane_again();
  const bool second = n0 >= a.n_split;
  const int act = a.glu || n0 >= a.act_from ? a.act : -1;
  const int64_t ld = second ? a.ld2 : a.ld1;
  uint16_t *out = second ? (uint16_t *)a.out2 + (n0 - a.n_split) : (uint16_t *)a.out1 + (a.glu ? n0 / 2 : n0);
  out += m0 * ld;
  const bool past = whole_pieces(out, ld);
  float bv[4 * kNT];
#pragma unroll
  for (int j = 0; j < kNT; ++j) {
    const u32x2 b = *reinterpret_cast<const u32x2 *>(staging + j * 32 + 8 * (lane >> 4));
#pragma unroll
    for (int e = 0; e < 4; ++e) bv[4 * j + e] = a.bias ? bf16_bits_to_f32((uint16_t)(b[e >> 1] >> (16 * (e & 1)))) : 0.f;
  }
  const int orow = a.glu ? lane >> 2 : lane >> 3, ochunk = a.glu ? lane & 3 : lane & 7;
  const int passes = a.glu ? 2 : 4, step = a.glu ? 16 : 8;   // rows to a pass
  const bool inside = n0 + ochunk * (a.glu ? 16 : 8) < a.N;
  const uint32_t out_off = (uint32_t)orow * (uint32_t)ld + ochunk * 8;
#pragma unroll 1
  for (int m = 0; m < kWM; m += 32) {
#pragma unroll 1
    for (int h = 0; h < 2; ++h) {
      const int row = h * 16 + (lane & 15);
      float v[4 * kNT];
      // one copy of what follows, whichever part of the tile: the instruction cache is shared by two CUs
#pragma unroll
      for (int i = 0; i < kMT; ++i)
        if (m + h * 16 == i * 16) {
#pragma unroll
          for (int e = 0; e < 4 * kNT; ++e) v[e] = acc[i][e >> 2][e & 3] + bv[e];
        }
      if (a.glu) {   // (gate, up) pairs; gate, up and activation rounded to bf16 as the reference does
        float g[2 * kNT];
#pragma unroll
        for (int e = 0; e < 2 * kNT; ++e) g[e] = bf16_bits_to_f32(f32_to_bf16_bits(v[2 * e]));
        act_n<2 * kNT>(act, g, 0, 0);
#pragma unroll
        for (int e = 0; e < 2 * kNT; ++e) g[e] = bf16_bits_to_f32(f32_to_bf16_bits(g[e])) * bf16_bits_to_f32(f32_to_bf16_bits(v[2 * e + 1]));
#pragma unroll
        for (int j = 0; j < kNT; ++j) *reinterpret_cast<uint32_t *>(staging + row * 64 + ((j ^ ((row >> 2) & 3)) << 4) + 4 * (lane >> 4)) = pack_bf16x2(g[2 * j], g[2 * j + 1]);
        continue;
      }
      act_n<4 * kNT>(act, v, 0, 0);
#pragma unroll
      for (int j = 0; j < kNT; ++j)
        *reinterpret_cast<u32x2 *>(staging + row * 128 + (((j * 2 + (lane >> 5)) ^ ((row >> 1) & 7)) << 4) + 8 * ((lane >> 4) & 1)) =
            u32x2{pack_bf16x2(v[4 * j], v[4 * j + 1]), pack_bf16x2(v[4 * j + 2], v[4 * j + 3])};
    }
    // LDS operations of one wave complete in order; no block barrier is needed for a wave-private region
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      if (p >= passes) break;
      const int r = p * step + orow;
      const u32x4 x = *reinterpret_cast<const u32x4 *>(staging + (a.glu ? r * 64 + ((ochunk ^ ((r >> 2) & 3)) << 4) : r * 128 + ((ochunk ^ ((r >> 1) & 7)) << 4)));
      if (inside && m0 + m + r < a.M) store_rows(out + (m + p * step) * ld + out_off, x, past);
    }
  }
}

// The same with a residual and no bias, activation or gate: what comes after the first 32 rows is asked for at once.
__device__ __forceinline__ void write_residual(const LinearArgs &a, Acc acc, char *staging, int m0, int n0) {
  const int lane = lane_again();
  const int orow = lane >> 3, ochunk = lane & 7;
  u32x4 more[kWM / 32 - 1][4];
#pragma unroll
  for (int b = 1; b < kWM / 32; ++b)
#pragma unroll
    for (int p = 0; p < 4; ++p) more[b - 1][p] = *reinterpret_cast<const u32x4 *>(residual_piece(a, m0 + b * 32 + p * 8 + orow, n0 + ochunk * 8));
  const bool second = n0 >= a.n_split;
  const int64_t ld = second ? a.ld2 : a.ld1;
  uint16_t *out = second ? (uint16_t *)a.out2 + (n0 - a.n_split) : (uint16_t *)a.out1 + n0;
  out += m0 * ld;
  const bool past = whole_pieces(out, ld);
  const bool inside = n0 + ochunk * 8 < a.N;
  const uint32_t out_off = (uint32_t)orow * (uint32_t)ld + ochunk * 8;
#pragma unroll
  for (int b = 0; b < kWM / 32; ++b) {
    if (b > 0) {
#pragma unroll
      for (int p = 0; p < 4; ++p) *reinterpret_cast<u32x4 *>(staging + (p * 8 + orow) * 128 + ((ochunk ^ (((p * 8 + orow) >> 1) & 7)) << 4)) = more[b - 1][p];
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int j = 0; j < kNT; ++j) {
        const int row = h * 16 + (lane & 15);
        u32x2 *at = reinterpret_cast<u32x2 *>(staging + row * 128 + (((j * 2 + (lane >> 5)) ^ ((row >> 1) & 7)) << 4) + 8 * ((lane >> 4) & 1));
        const u32x2 x = *at;
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = acc[2 * b + h][j][e] + bf16_bits_to_f32((uint16_t)(x[e >> 1] >> (16 * (e & 1))));
        *at = u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
      }
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const int r = p * 8 + orow;
      const u32x4 x = *reinterpret_cast<const u32x4 *>(staging + r * 128 + ((ochunk ^ ((r >> 1) & 7)) << 4));
      if (inside && m0 + b * 32 + r < a.M) store_rows(out + (b * 32 + p * 8) * ld + out_off, x, past);
    }
  }
}

// Any other: 16 rows of f32 through LDS, 16-byte chunk c of row r at c ^ r, 8 columns of a row to a lane.
__device__ __forceinline__ void write_rows(const LinearArgs &a, Acc acc, float *staging, int m0, int n0) {
  const int lane = lane_again();
  const bool vec_out = rows_store_16(a);
  const int n = n0 + (lane & 7) * 8;
  const bool whole = n + 8 <= a.N;
  float bv[8];
  load_bias8(a, n, bv);
#pragma unroll 1
  for (int q = 0; q < kMT; ++q) {
#pragma unroll
    for (int i = 0; i < kMT; ++i)
      if (q == i) {
#pragma unroll
        for (int j = 0; j < kNT; ++j) *reinterpret_cast<f32x4 *>(staging + (lane & 15) * kWN + (((j * 4 + (lane >> 4)) ^ (lane & 15)) << 2)) = acc[i][j];
      }
#pragma unroll 1
    for (int p = 0; p < 2; ++p) {
      const int r = p * 8 + (lane >> 3), m = m0 + q * 16 + r;
      const f32x4 v0 = *reinterpret_cast<const f32x4 *>(staging + r * kWN + ((((lane & 7) * 2) ^ r) << 2));
      const f32x4 v1 = *reinterpret_cast<const f32x4 *>(staging + r * kWN + ((((lane & 7) * 2 + 1) ^ r) << 2));
      if (m < a.M && n < a.N) store_row8(a, v0, v1, bv, m, n, whole, vec_out);
    }
  }
}

// Tile rows lie in LDS as in dma_tile_mainloop_k64 (gemm_mfma.hip): 128 bytes, 16-byte chunk c of row r at c ^ ((r >> 1) & 7).
// SHARED: some tiles are shared out.
template <int OUT, bool SHARED> __global__ void __launch_bounds__(kThreads) k_gemm_bf16_mfma_persist(LinearArgs a, StreamKArgs sk) {
  extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 2, wn = wave & 3;
  float *staging = reinterpret_cast<float *>(lds + 2 * kStageElems);
  const int tiles_m = (a.M + kTileDim - 1) / kTileDim, tiles_n = (a.N + kTileDim - 1) / kTileDim;
  const int stages = a.K / kStageK;
  // Blocks go to the XCDs in turn.  An XCD has a run of the shared part and a run of the whole tiles, and its blocks step
  // through the latter side by side, so that the tiles in the works at one time share their panels in its L2.
  const int xcd = blockIdx.x % kXcds, per_xcd = gridDim.x / kXcds, p = xcd * per_xcd + blockIdx.x / kXcds;
  const int wholes = tiles_m * tiles_n - sk.sk_tiles, run = (wholes + kXcds - 1) / kXcds;
  Walk todo;
  todo.u = SHARED ? sk_start(sk, p) : 0;
  todo.u_end = SHARED ? sk_start(sk, p + 1) : 0;
  todo.whole = sk.sk_tiles + xcd * run + blockIdx.x / kXcds;
  todo.whole_end = sk.sk_tiles + ((xcd + 1) * run < wholes ? (xcd + 1) * run : wholes);
  todo.step = per_xcd;
  todo.stages = stages;

  // ---- the loading side: two stages ahead of the multiplies, in the same sequence
  Walk ahead = todo;
  const char *src_a = nullptr, *src_w = nullptr;
  uint32_t off_a[kLoads], off_w[kLoads];
  int left = 0;   // stages of its segment still to be requested
  auto advance = [&] {
    Segment s;
    if (left > 0 || !ahead.next(s)) return;
    int tile_m, tile_n;
    tile_coords(s.tile, tiles_m, tiles_n, &tile_m, &tile_n);
    const int m0 = tile_m * kTileDim, n0 = tile_n * kTileDim;
    const int lane = lane_again();
    src_a = (const char *)a.A + ((int64_t)m0 * a.lda + s.k0 * kStageK) * 2;
    src_w = (const char *)a.W + ((int64_t)n0 * a.ldw + s.k0 * kStageK) * 2;
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      const int r = (wave * kLoads + j) * 8 + (lane >> 3);
      const uint32_t chunk = ((lane & 7) ^ ((r >> 1) & 7)) * 16;
      off_a[j] = (uint32_t)(m0 + r < a.M ? r : a.M - 1 - m0) * (uint32_t)(2 * a.lda) + chunk;   // rows beyond the last: that row
      off_w[j] = (uint32_t)(n0 + r < a.N ? r : a.N - 1 - n0) * (uint32_t)(2 * a.ldw) + chunk;
    }
    left = s.n;
  };
  uint16_t *dst = lds + wave * kLoads * 8 * kStageK;
  auto request_part = [&](int buf, int j) __attribute__((always_inline)) {
    uint16_t *da = dst + buf * kStageElems, *dw = da + kTileDim * kStageK;
    __builtin_amdgcn_global_load_lds((const void *)(src_a + off_a[j]), (lds_ptr)(da + j * 8 * kStageK), 16, 0, 0);
    __builtin_amdgcn_global_load_lds((const void *)(src_w + off_w[j]), (lds_ptr)(dw + j * 8 * kStageK), 16, 0, 0);
  };
  auto step = [&] {
    --left;
    src_a += left > 0 ? 2 * kStageK : 0;   // (behind a segment's last stage: where it was, should nothing follow)
    src_w += left > 0 ? 2 * kStageK : 0;
  };
  auto request = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < kLoads; ++j) request_part(buf, j);
  };

  Segment seg;
  if (!todo.next(seg)) return;
  advance();
  request(0);
  step();
  advance();
  if (left > 0) {
    request(1);
    step();
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * kLoads) : "memory");
  } else {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
  __builtin_amdgcn_s_barrier();

  // ---- the multiplying side
  const int frow = (lane & 15) * kStageK, sw = (lane >> 1) & 7;
  int coff[2];   // the four chunks of 8 of an MFMA's 32 of K
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) coff[ks] = ((ks * 4 + (lane >> 4)) ^ sw) << 3;
  const int a_off = wm * kWM * kStageK + frow, w_off = kTileDim * kStageK + wn * kWN * kStageK + frow;
  bf16x8 fa[kMT], fb[kNT];
  f32x4 acc[kMT][kNT];
#define RAI_READ(BUF, KS)                                                                                                      \
  do {                                                                                                                         \
    const uint16_t *as_ = lds + (BUF) * kStageElems + a_off + coff[KS], *bs_ = lds + (BUF) * kStageElems + w_off + coff[KS];   \
    _Pragma("unroll") for (int j = 0; j < kNT; ++j) fb[j] = *reinterpret_cast<const bf16x8 *>(bs_ + j * 16 * kStageK);         \
    _Pragma("unroll") for (int i = 0; i < kMT; ++i) fa[i] = *reinterpret_cast<const bf16x8 *>(as_ + i * 16 * kStageK);         \
  } while (0)
#define RAI_MUL(I0, I1)                                                                        \
  do {                                                                                         \
    _Pragma("unroll") for (int i = I0; i < I1; ++i)                                            \
      _Pragma("unroll") for (int j = 0; j < kNT; ++j)                                          \
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[j], fa[i], acc[i][j], 0, 0, 0); \
  } while (0)
// (the multiplies stay on their side)
#define RAI_BAR() do { __builtin_amdgcn_sched_barrier(0); __builtin_amdgcn_s_barrier(); __builtin_amdgcn_sched_barrier(0); } while (0)
#define RAI_WAIT(x) asm volatile("s_waitcnt " x ::: "memory")
  // The waves of the tile's lower half run one phase behind those of its upper half, one of each on every SIMD: while one
  // reads the fragments of 32 of K the other has the matrix cores to itself, and at every barrier they change places.  A
  // buffer is free once the late waves have read it: they ask for its next stage while they multiply, the early ones, a
  // barrier later in their own sequence, before they read.  All have it three phases on, ahead of the early ones' first read.
  const bool late = wave >= kWaves / 2;
  int cur = 0, m0 = 0, n0 = 0;
  auto stage = [&](bool last) __attribute__((always_inline)) {
    if (OUT != kRows && last) ask_for(a, reinterpret_cast<char *>(staging + wave * kStagingFloats), m0, n0);
    RAI_READ(cur, 0);
    RAI_BAR();
    __builtin_amdgcn_s_setprio(1);
    RAI_MUL(0, 8);
    __builtin_amdgcn_s_setprio(0);
    RAI_BAR();
    RAI_READ(cur, 1);
    advance();
    if (late) RAI_WAIT("vmcnt(0) lgkmcnt(0)");
    else RAI_WAIT("lgkmcnt(0)");
    RAI_BAR();
    __builtin_amdgcn_s_setprio(1);
    RAI_MUL(0, 2);
    __builtin_amdgcn_sched_barrier(0);
    if (late) request_part(cur, 0);
    RAI_MUL(2, 4);
    __builtin_amdgcn_sched_barrier(0);
    if (late) request_part(cur, 1);
    RAI_MUL(4, 6);
    __builtin_amdgcn_sched_barrier(0);
    if (late) request_part(cur, 2);
    RAI_MUL(6, 8);
    __builtin_amdgcn_sched_barrier(0);
    if (late) request_part(cur, 3);
    else RAI_WAIT("vmcnt(0)");
    __builtin_amdgcn_s_setprio(0);
    RAI_BAR();
    if (!late) request(cur);
    step();
    cur ^= 1;
  };
  if (late) RAI_BAR();
  for (;;) {
    int tile_m, tile_n;
    tile_coords(seg.tile, tiles_m, tiles_n, &tile_m, &tile_n);
    m0 = tile_m * kTileDim + wm * kWM;
    n0 = tile_n * kTileDim + wn * kWN;
    const f32x4 zero = {};
#pragma unroll
    for (int i = 0; i < kMT; ++i)
#pragma unroll
      for (int j = 0; j < kNT; ++j) acc[i][j] = zero;
    stage(seg.n == 1 && !SHARED);
    for (int st = 1; st < seg.n; ++st) stage(SHARED ? st + 1 == stages : st + 1 == seg.n);
    if (!late) RAI_BAR();   // both halves write their outputs side by side
    char *mine = reinterpret_cast<char *>(staging + wave * kStagingFloats);
    bool write = true;
    if (SHARED && seg.n != stages) {
      write = sum_shares(sk, acc, reinterpret_cast<int *>(staging), seg.tile, stages, p, wave, lane_again());
      if (write && OUT != kRows) {
        ask_for(a, mine, m0, n0);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      }
    }
    if (write) {
      if constexpr (OUT == kPlain) write_plain(a, acc, mine, m0, n0);
      else if constexpr (OUT == kPlainResidual) write_residual(a, acc, mine, m0, n0);
      else write_rows(a, acc, reinterpret_cast<float *>(mine), m0, n0);
    }
    if (!todo.next(seg)) break;
    if (late) RAI_BAR();
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // what was asked for behind the last stage lands before the LDS is another's
#undef RAI_READ
#undef RAI_MUL
#undef RAI_BAR
#undef RAI_WAIT
}

}  // namespace

template <int OUT, bool SHARED> static int launch_persist(hipStream_t st, const LinearArgs &a, const StreamKArgs &sk, int dev, int grid) {
  static bool attr_set[64];
  if (!attr_set[dev]) {
    RAI_HIP_TRY(hipFuncSetAttribute((const void *)k_gemm_bf16_mfma_persist<OUT, SHARED>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsBytes));
    attr_set[dev] = true;
  }
  hipLaunchKernelGGL((k_gemm_bf16_mfma_persist<OUT, SHARED>), dim3(grid), dim3(kThreads), kLdsBytes, st, a, sk);
  return launch_check("gemm_bf16_mfma_persist");
}

int launch_gemm_bf16_persist(hipStream_t st, const LinearArgs &a, const StreamKArgs &sk) {
  int dev = a.dev;
  if (dev < 0) RAI_HIP_TRY(hipGetDevice(&dev));
  RAI_REQUIRE(dev >= 0 && dev < 64, RAI_ERR_BAD_ARG, "device %d out of range", dev);
  const int tiles = ((a.M + kTileDim - 1) / kTileDim) * ((a.N + kTileDim - 1) / kTileDim);
  const int grid = sk.sk_tiles || tiles >= kNumCU ? kNumCU : (tiles + kXcds - 1) / kXcds * kXcds;
  const int out = gemm_persist_plain(a) ? a.residual ? kPlainResidual : kPlain : kRows;
  if (sk.sk_tiles)
    return out == kPlain ? launch_persist<kPlain, true>(st, a, sk, dev, grid) : out == kRows ? launch_persist<kRows, true>(st, a, sk, dev, grid)
                                                                                             : launch_persist<kPlainResidual, true>(st, a, sk, dev, grid);
  return out == kPlain ? launch_persist<kPlain, false>(st, a, sk, dev, grid) : out == kRows ? launch_persist<kRows, false>(st, a, sk, dev, grid)
                                                                                            : launch_persist<kPlainResidual, false>(st, a, sk, dev, grid);
}

}  // namespace rai
