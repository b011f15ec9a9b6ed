// bf16 x bf16 -> f32 MFMA GEMM for the Linear layout (out = A[M,K] . W[N,K]^T),
// gfx950 v_mfma_f32_32x32x16_bf16.
//
//   - block tile BM x BN, 4 waves in a 2x2 grid, each wave (BM/2) x (BN/2) made of
//     32x32 MFMA tiles; K step BK.
//   - global -> registers -> LDS with a two-deep LDS buffer: the loads of tile
//     k+1 are in flight while tile k is multiplied; one barrier per K step.
//     Rows are clamped instead of predicated, so the main loop has no branches.
//   - LDS rows are padded by 16 bytes: the 16-byte fragment reads of 16 lanes hit
//     64 distinct banks.
//   - blockIdx -> tile mapping is XCD-aware: hardware hands consecutive blocks to
//     the 8 XCDs round-robin, so each XCD is given a contiguous run of tiles and
//     the tiles that share a weight panel share one L2.
//   - epilogue through LDS: every wave stages 32 x (BN/2) accumulators at a time
//     and writes 16-byte rows with bias / activation / residual applied (or raw
//     f32 partial sums when K is split over several blocks).
#include <cstring>
#include <type_traits>

#include "gemm_device.h"
#include "latent.h"
#include "rai_hip_peaks.h"

namespace rai {

// LDS a tile kernel needs: two stages of A and B tiles, or the epilogue staging area if that is larger.
template <int BM, int BN, int PITCH, int WGN = 2, int WGM = 2> constexpr int gemm_lds_bytes() {
  constexpr int tiles = 2 * (BM + BN) * PITCH * 2, staging = WGM * WGN * 32 * (BN / WGN + 4) * 4;
  return tiles > staging ? tiles : staging;
}

// LDS of the LDS-DMA tile kernels: NS stages of 32 of K, or (NS == 2, or SH == 0) of 64.
template <int BM, int BN, int NS, int WGN, int WGM = 2, int SH = 2> constexpr int dma_lds_bytes() {
  return gemm_lds_bytes<BM, BN, NS == 2 || SH == 0 ? 32 * NS : 32 * NS / 2, WGN, WGM>();
}

// Tile epilogue shared by the tile kernels: every wave stages 32 x WN accumulators at a time in
// LDS (the tile buffers are free by then) and writes 16-byte rows with bias / activation /
// residual applied, or raw f32 partial sums when K is split over several blocks.
// (WGM x WGN = waves along M and N; WGM = 2 except for the 256 x 192 tile.)
template <int BM, int BN, int LDS_BYTES, int WGN = 2, int WGM = 2>
__device__ __forceinline__ void gemm_tile_epilogue(const LinearArgs &a, f32x16 (&acc)[BM / (32 * WGM)][BN / (32 * WGN)],
                                                   uint16_t *lds, int m0, int n0, int wave, int lane, int split,
                                                   float *partial) {
  constexpr int WM = BM / WGM, WN = BN / WGN;
  constexpr int MT = WM / 32, NT = WN / 32;
  constexpr int EP = WN + 4;                // epilogue staging pitch (floats)
  const int wm = wave / WGN, wn = wave % WGN;
  // ---- epilogue: stage 32 x WN accumulators per wave in LDS, write 8 columns per lane
  float *stage = reinterpret_cast<float *>(lds) + wave * 32 * EP;
  static_assert(WGM * WGN * 32 * EP * 4 <= LDS_BYTES, "epilogue staging does not fit the tile buffers");
  constexpr int CG = WN / 8;                 // 8-column groups per staged row
  // rows per pass: a lane keeps its column group from pass to pass, so a pass covers a power-of-two number of whole
  // rows (CG = 12, the 96-column wave tile, leaves 16 of the 64 lanes idle)
  constexpr int RP = 64 / CG >= 16 ? 16 : 64 / CG >= 8 ? 8 : 64 / CG >= 4 ? 4 : 2;
  constexpr int ITEMS = 32 / RP;             // passes
  const bool vec_out = rows_store_16(a);
  // A lane serves the same 8 columns in every pass: their bias values are fetched once, ahead of the passes, not
  // inside each of them, where the load's latency (about a microsecond under load) sat between the LDS read and the
  // store of every pass.
  static_assert(RP * CG <= 64 && 32 % RP == 0, "a pass is RP whole rows of CG column groups");
  const int n = n0 + wn * WN + (lane % CG) * 8;
  const bool whole = n + 8 <= a.N;
  float bv[8] = {};
  if (!partial) load_bias8(a, n, bv);
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    // accumulator register r of lane l is C[8*(r/4) + 4*(l/32) + r%4][l%32]
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        stage[(8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)) * EP + j * 32 + (lane & 31)] = acc[i][j][r];
    // LDS operations of one wave complete in order; no block barrier is needed for a wave-private region
#pragma unroll 1
    for (int it = 0; it < ITEMS; ++it) {
      const int row = lane / CG + it * RP, cg = lane % CG;
      const int m = m0 + wm * WM + i * 32 + row;
      if (lane >= RP * CG || m >= a.M || n >= a.N) continue;
      const f32x4 v0 = *reinterpret_cast<const f32x4 *>(stage + row * EP + cg * 8);
      const f32x4 v1 = *reinterpret_cast<const f32x4 *>(stage + row * EP + cg * 8 + 4);
      if (partial) {
        float *p = partial + ((int64_t)split * a.M + m) * a.N + n;
        if (a.N % 4 == 0) {
          *reinterpret_cast<f32x4 *>(p) = v0;
          if (n + 4 < a.N) *reinterpret_cast<f32x4 *>(p + 4) = v1;
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (n + e < a.N) p[e] = e < 4 ? v0[e & 3] : v1[e & 3];
        }
        continue;
      }
      store_row8(a, v0, v1, bv, m, n, whole, vec_out);
    }
  }
}

template <int BM, int BN, int BK, int SH = 0>
__global__ void __launch_bounds__(256) k_gemm_bf16_mfma(LinearArgs a, int splits, int k_per_split, float *partial) {
  // SH == 0: rows padded by 16 bytes.  SH > 0: unpadded rows, the 16-byte chunk c of row r stored at
  // chunk c ^ ((r >> SH) & (BK/8 - 1)), so that both the row-wise stores and the column-wise
  // fragment reads spread over the banks.
  constexpr int PITCH = SH ? BK : BK + 8;
  constexpr int CMASK = BK / 8 - 1;
  constexpr int WM = BM / 2, WN = BN / 2;
  constexpr int MT = WM / 32, NT = WN / 32;
  constexpr int CPR = BK / 8;               // 16-byte chunks per tile row
  constexpr int A_CH = BM * CPR / 256;      // chunks per thread
  constexpr int B_CH = BN * CPR / 256;
  static_assert(A_CH >= 1 && B_CH >= 1, "tile too small for 256 threads");
  extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
  uint16_t *As = lds;                       // [2][BM][PITCH]
  uint16_t *Bs = lds + 2 * BM * PITCH;      // [2][BN][PITCH]

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int tiles_m = (a.M + BM - 1) / BM, tiles_n = (a.N + BN - 1) / BN;
  const int total = tiles_m * tiles_n;
  const int tile = xcd_remap(blockIdx.x, total);
  if (tile >= total) return;
  int tile_m, tile_n;
  tile_coords(tile, tiles_m, tiles_n, &tile_m, &tile_n);
  const int m0 = tile_m * BM, n0 = tile_n * BN;
  const int split = blockIdx.y;
  const int k_begin = split * k_per_split;
  const int k_end = k_begin + k_per_split < a.K ? k_begin + k_per_split : a.K;
  const int KT = (k_end - k_begin) / BK;

  // per-thread source pointers (rows clamped into range; results of clamped rows are never stored)
  const uint16_t *ga[A_CH], *gb[B_CH];
  int sa[A_CH], sb[B_CH];
#pragma unroll
  for (int i = 0; i < A_CH; ++i) {
    const int c = tid + i * 256, row = c / CPR, kc = (c % CPR) * 8;
    int m = m0 + row;
    m = m < a.M ? m : a.M - 1;
    ga[i] = (const uint16_t *)a.A + (int64_t)m * a.lda + k_begin + kc;
    sa[i] = row * PITCH + (SH ? (((kc >> 3) ^ ((row >> SH) & CMASK)) << 3) : kc);
  }
#pragma unroll
  for (int i = 0; i < B_CH; ++i) {
    const int c = tid + i * 256, row = c / CPR, kc = (c % CPR) * 8;
    int n = n0 + row;
    n = n < a.N ? n : a.N - 1;
    gb[i] = (const uint16_t *)a.W + (int64_t)n * a.ldw + k_begin + kc;
    sb[i] = row * PITCH + (SH ? (((kc >> 3) ^ ((row >> SH) & CMASK)) << 3) : kc);
  }

  f32x16 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  u32x4 ra[A_CH], rb[B_CH];
#pragma unroll
  for (int i = 0; i < A_CH; ++i) ra[i] = *reinterpret_cast<const u32x4 *>(ga[i]);
#pragma unroll
  for (int i = 0; i < B_CH; ++i) rb[i] = *reinterpret_cast<const u32x4 *>(gb[i]);
#pragma unroll
  for (int i = 0; i < A_CH; ++i) *reinterpret_cast<u32x4 *>(As + sa[i]) = ra[i];
#pragma unroll
  for (int i = 0; i < B_CH; ++i) *reinterpret_cast<u32x4 *>(Bs + sb[i]) = rb[i];
  __syncthreads();

  const int frag = (lane & 31) * PITCH + (SH ? 0 : (lane >> 5) * 8);
  const int rsw = SH ? (((lane & 31) >> SH) & CMASK) : 0;
  for (int kt = 0; kt < KT; ++kt) {
    const int buf = kt & 1;
    const bool more = kt + 1 < KT;
    if (more) {
#pragma unroll
      for (int i = 0; i < A_CH; ++i) ra[i] = *reinterpret_cast<const u32x4 *>(ga[i] + (kt + 1) * BK);
#pragma unroll
      for (int i = 0; i < B_CH; ++i) rb[i] = *reinterpret_cast<const u32x4 *>(gb[i] + (kt + 1) * BK);
    }
    const uint16_t *as = As + buf * BM * PITCH + wm * WM * PITCH + frag;
    const uint16_t *bs = Bs + buf * BN * PITCH + wn * WN * PITCH + frag;
#pragma unroll
    for (int ks = 0; ks < BK / 16; ++ks) {
      bf16x8 fa[MT], fb[NT];
#pragma unroll
      for (int i = 0; i < MT; ++i)
        fa[i] = *reinterpret_cast<const bf16x8 *>(as + i * 32 * PITCH + (SH ? (((ks * 2 + (lane >> 5)) ^ rsw) << 3) : ks * 16));
#pragma unroll
      for (int j = 0; j < NT; ++j)
        fb[j] = *reinterpret_cast<const bf16x8 *>(bs + j * 32 * PITCH + (SH ? (((ks * 2 + (lane >> 5)) ^ rsw) << 3) : ks * 16));
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);
    }
    if (more) {
      uint16_t *ad = As + (buf ^ 1) * BM * PITCH, *bd = Bs + (buf ^ 1) * BN * PITCH;
#pragma unroll
      for (int i = 0; i < A_CH; ++i) *reinterpret_cast<u32x4 *>(ad + sa[i]) = ra[i];
#pragma unroll
      for (int i = 0; i < B_CH; ++i) *reinterpret_cast<u32x4 *>(bd + sb[i]) = rb[i];
    }
    __syncthreads();
  }

  gemm_tile_epilogue<BM, BN, gemm_lds_bytes<BM, BN, PITCH>()>(a, acc, lds, m0, n0, wave, lane, split, partial);
}

// Tile kernel with direct global -> LDS loads (global_load_lds_dwordx4): no registers and no
// ds_write instructions are spent on staging, so NS LDS stages are cheap and the loads run
// NS-1 K tiles ahead of the multiplies, which is what hides HBM/L2 latency at 2-3 blocks per CU.
//   - one load instruction moves 64 lanes x 16 bytes into 1 KB of consecutive LDS, i.e. 16
//     unpadded tile rows of BK = 32 bf16; bank spreading comes from a swizzle instead of padding:
//     the 16-byte chunk c of row r lives at chunk position c ^ ((r >> SH) & 3), applied by choosing
//     which global chunk each lane fetches;
//   - every wave issues (BM + BN) / 64 loads per K tile; `s_waitcnt vmcnt(loads * (NS - 3))` then a
//     bare s_barrier make tile t+1 visible to the block (and retire stage t-1 for refilling) with one
//     barrier per K tile.  The barrier carries no fence: a fence would wait for every outstanding
//     LDS load, i.e. drain the pipeline.
// K loop of the LDS-DMA tile kernels: acc = A[m0.., k_begin..] . W[n0.., k_begin..]^T over KT tiles of 32, with the
// software pipeline described above.  Ends with every load landed and the block synchronised, so the caller may reuse
// the LDS stages.
template <int BM, int BN, int NS, int SH, int WGN>
__device__ __forceinline__ void dma_tile_mainloop(const LinearArgs &a, uint16_t *lds, int m0, int n0, int k_begin, int KT,
                                                  int wave, int lane, f32x16 (&acc)[BM / 64][BN / (32 * WGN)]) {
  constexpr int BK = 32, PITCH = BK;
  constexpr int WM = BM / 2, WN = BN / WGN;
  constexpr int MT = WM / 32, NT = WN / 32;
  constexpr int LA = BM / (32 * WGN), LB = BN / (32 * WGN);   // loads per wave per K tile (16 rows each)
  constexpr int STAGE = (BM + BN) * BK;              // elements per stage: A rows then B rows
  const int wm = wave / WGN, wn = wave % WGN;
  // lane -> (row within the 16-row group, swizzled chunk)
  const int lrow = lane >> 2;
  const uint16_t *gpa[LA], *gpb[LB];
#pragma unroll
  for (int j = 0; j < LA; ++j) {
    const int r = (wave * LA + j) * 16 + lrow;   // row within the tile
    int m = m0 + r;
    m = m < a.M ? m : a.M - 1;
    gpa[j] = (const uint16_t *)a.A + (int64_t)m * a.lda + k_begin + (((lane & 3) ^ ((r >> SH) & 3)) << 3);
  }
#pragma unroll
  for (int j = 0; j < LB; ++j) {
    const int r = (wave * LB + j) * 16 + lrow;
    int n = n0 + r;
    n = n < a.N ? n : a.N - 1;
    gpb[j] = (const uint16_t *)a.W + (int64_t)n * a.ldw + k_begin + (((lane & 3) ^ ((r >> SH) & 3)) << 3);
  }
  typedef __attribute__((address_space(3))) void *lds_ptr;
  auto issue = [&](int kt, int stage) {
    kt = kt < KT ? kt : KT - 1;   // past the end: refetch the last tile into a stage nobody reads again
    uint16_t *sa = lds + stage * STAGE + wave * LA * 16 * BK;
    uint16_t *sb = lds + stage * STAGE + BM * BK + wave * LB * 16 * BK;
#pragma unroll
    for (int j = 0; j < LA; ++j)
      __builtin_amdgcn_global_load_lds((const void *)(gpa[j] + kt * BK), (lds_ptr)(sa + j * 16 * BK), 16, 0, 0);
#pragma unroll
    for (int j = 0; j < LB; ++j)
      __builtin_amdgcn_global_load_lds((const void *)(gpb[j] + kt * BK), (lds_ptr)(sb + j * 16 * BK), 16, 0, 0);
  };

#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

#pragma unroll
  for (int t = 0; t < NS - 1; ++t) issue(t, t);

  // Software pipeline of one K tile (BK = 32 = two MFMA K steps, fragment sets F0 and F1):
  //   top:  read F1 (tile t, step 1)            | multiply F0 (tile t, step 0)
  //   mid:  wait for tile t+1, barrier, issue the loads of tile t+NS-1, read F0 (tile t+1, step 0)
  //                                             | multiply F1
  // so LDS reads always run one fragment set ahead of the MFMAs, the barrier sits between two
  // batches of multiplies that are already in the pipe, and global loads are NS-2 tiles ahead.
  const int frow = (lane & 31) * PITCH;
  const int rsw = ((lane & 31) >> SH) & 3;
  const int coff0 = ((0 + (lane >> 5)) ^ rsw) << 3, coff1 = ((2 + (lane >> 5)) ^ rsw) << 3;
  const int a_off = wm * WM * PITCH + frow, b_off = BM * BK + wn * WN * PITCH + frow;
  bf16x8 fa0[MT], fb0[NT], fa1[MT], fb1[NT];
#define RAI_DMA_WAIT(n)                                                                        \
  do {                                                                                         \
    if constexpr ((n) == 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                   \
    else if constexpr ((n) == 4) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");              \
    else if constexpr ((n) == 6) asm volatile("s_waitcnt vmcnt(6)" ::: "memory");              \
    else if constexpr ((n) == 8) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");              \
    else if constexpr ((n) == 12) asm volatile("s_waitcnt vmcnt(12)" ::: "memory");            \
    else if constexpr ((n) == 16) asm volatile("s_waitcnt vmcnt(16)" ::: "memory");            \
    else static_assert((n) < 0, "add the vmcnt immediate for this configuration");             \
  } while (0)
  RAI_DMA_WAIT((LA + LB) * (NS - 2));   // tile 0 has landed (this wave's part)
  __builtin_amdgcn_s_barrier();
  {
    const uint16_t *as = lds + a_off, *bs = lds + b_off;
#pragma unroll
    for (int i = 0; i < MT; ++i) fa0[i] = *reinterpret_cast<const bf16x8 *>(as + i * 32 * PITCH + coff0);
#pragma unroll
    for (int j = 0; j < NT; ++j) fb0[j] = *reinterpret_cast<const bf16x8 *>(bs + j * 32 * PITCH + coff0);
  }
  int cur = 0, nxt = NS - 1;
  // A wave issues in order and an MFMA issue blocks until the matrix pipe is free, so anything placed
  // between two batches of MFMAs runs with the pipe idle.  The LDS reads and the load issues are
  // therefore interleaved one by one between the MFMAs of each half (sched_group_barrier patterns).
  for (int kt = 0; kt < KT; ++kt) {
    {
      const uint16_t *as = lds + cur * STAGE + a_off, *bs = lds + cur * STAGE + b_off;
#pragma unroll
      for (int i = 0; i < MT; ++i) fa1[i] = *reinterpret_cast<const bf16x8 *>(as + i * 32 * PITCH + coff1);
#pragma unroll
      for (int j = 0; j < NT; ++j) fb1[j] = *reinterpret_cast<const bf16x8 *>(bs + j * 32 * PITCH + coff1);
    }
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa0[i], fb0[j], acc[i][j], 0, 0, 0);
#pragma unroll
    for (int g = 0; g < MT + NT; ++g) {
      __builtin_amdgcn_sched_group_barrier(0x008, MT * NT / (MT + NT) > 0 ? MT * NT / (MT + NT) : 1, 0);  // MFMA
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);                                                  // one LDS read
    }
    __builtin_amdgcn_sched_barrier(0);
    RAI_DMA_WAIT((LA + LB) * (NS - 3));  // tile kt+1 has landed; NS-3 younger tiles stay in flight
    __builtin_amdgcn_s_barrier();
    issue(kt + NS - 1, nxt);               // into the stage of tile kt-1, which every wave has left
    cur = cur + 1 == NS ? 0 : cur + 1;
    nxt = nxt + 1 == NS ? 0 : nxt + 1;
    {
      const uint16_t *as = lds + cur * STAGE + a_off, *bs = lds + cur * STAGE + b_off;
#pragma unroll
      for (int i = 0; i < MT; ++i) fa0[i] = *reinterpret_cast<const bf16x8 *>(as + i * 32 * PITCH + coff0);
#pragma unroll
      for (int j = 0; j < NT; ++j) fb0[j] = *reinterpret_cast<const bf16x8 *>(bs + j * 32 * PITCH + coff0);
    }
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa1[i], fb1[j], acc[i][j], 0, 0, 0);
#pragma unroll
    for (int g = 0; g < MT + NT; ++g) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // MFMA
      __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);   // one global -> LDS load
      __builtin_amdgcn_sched_group_barrier(0x008, MT * NT / (MT + NT) > 1 ? MT * NT / (MT + NT) - 1 : 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);   // one LDS read
    }
    __builtin_amdgcn_sched_barrier(0);
  }
#undef RAI_DMA_WAIT
  // the refetches issued past the end must land before the stages are reused for the epilogue
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
}

// The same K loop with K tiles of 64: a tile row is 128 bytes in LDS and one load instruction moves 8 rows x 128 bytes,
// so every request the L1 sends to L2 is a whole 128-byte line instead of half of one (the L2s deliver 1.7x the bytes
// per clock that way with all CUs asking, measured with the loads alone), and there is one barrier per 64 of K.  Two
// stages (the same 128 KB for a 256 x 256 tile as four stages of 32): stage s+1 is requested when stage s-1 has been
// left by every wave, a whole stage of multiplies before it is needed.  A small tile multiplies a stage in less time than
// its loads take: three or four stages (NS) keep two or three of them in flight.
//   - 16-byte chunk c (0..7) of row r lives at chunk position c ^ ((r >> 1) & 7): the 8 lanes that fetch one row swap
//     places within their 128-byte line, and a fragment read's 16 lanes per LDS cycle (16 rows at one chunk index; two
//     rows span the 64 banks) land on 16 different 16-byte slots.  (Swizzling by r & 7 left rows r and r + 8 on the
//     same banks: SQ_LDS_BANK_CONFLICT at 23 % of the kernel's cycles.)
//   - fragment sets alternate F0 / F1 over the four K steps of a stage; the reads run one set ahead of the multiplies.
//   - `half`: stage 0 begins 32 before the operands' rows do, and reads zeros there (K of an odd number of 32s: ODD, kernels of their own).
//     The first stage and not the last: it is asked for outside the loop, which need not know.  (With both ways to ask in one kernel the loop
//     of 128 x 256 tiles came out in another order: 1024 x 8192 x 8192 131.6 us, so 130.0; the other tiles' times are the same.)
static __device__ uint4 g_k_zeros[1];   // (sixteen bytes that nobody writes)
template <int BM, int BN, int WGN, int WGM = 2, int NS = 2>
__device__ __forceinline__ void dma_tile_mainloop_k64(const LinearArgs &a, uint16_t *lds, int m0, int n0, int k_begin, int KT,
                                                      int wave, int lane, f32x16 (&acc)[BM / (32 * WGM)][BN / (32 * WGN)], bool half = false) {
  constexpr int BK = 64;
  constexpr int WM = BM / WGM, WN = BN / WGN;
  constexpr int MT = WM / 32, NT = WN / 32;
  constexpr int NW = WGM * WGN;
  constexpr int LA = BM / (8 * NW), LB = BN / (8 * NW);   // loads per wave per stage (8 rows each)
  constexpr int STAGE = (BM + BN) * BK;
  static_assert(BM % (8 * NW) == 0 && BN % (8 * NW) == 0, "every wave loads whole groups of 8 rows");
  static_assert((LA + LB) * (NS - 1) <= 63, "the wait counts the stages' loads");
  const int wm = wave / WGN, wn = wave % WGN;
  const int lrow = lane >> 3;
  const uint16_t *gpa[LA], *gpb[LB];
#pragma unroll
  for (int j = 0; j < LA; ++j) {
    const int r = (wave * LA + j) * 8 + lrow;     // row within the tile
    int m = m0 + r;
    m = m < a.M ? m : a.M - 1;
    gpa[j] = (const uint16_t *)a.A + (int64_t)m * a.lda + k_begin + (((lane & 7) ^ ((r >> 1) & 7)) << 3);
  }
#pragma unroll
  for (int j = 0; j < LB; ++j) {
    const int r = (wave * LB + j) * 8 + lrow;
    int n = n0 + r;
    n = n < a.N ? n : a.N - 1;
    gpb[j] = (const uint16_t *)a.W + (int64_t)n * a.ldw + k_begin + (((lane & 7) ^ ((r >> 1) & 7)) << 3);
  }
  typedef __attribute__((address_space(3))) void *lds_ptr;
  auto issue = [&](int st, int buf) {
    uint16_t *sa = lds + buf * STAGE + wave * LA * 8 * BK;
    uint16_t *sb = lds + buf * STAGE + BM * BK + wave * LB * 8 * BK;
#pragma unroll
    for (int j = 0; j < LA; ++j)
      __builtin_amdgcn_global_load_lds((const void *)(gpa[j] + st * BK), (lds_ptr)(sa + j * 8 * BK), 16, 0, 0);
#pragma unroll
    for (int j = 0; j < LB; ++j)
      __builtin_amdgcn_global_load_lds((const void *)(gpb[j] + st * BK), (lds_ptr)(sb + j * 8 * BK), 16, 0, 0);
  };

#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  if (!half) {
    issue(0, 0);
  } else {
    uint16_t *sa = lds + wave * LA * 8 * BK, *sb = lds + BM * BK + wave * LB * 8 * BK;
    auto source = [&](const uint16_t *p, int r) { return ((lane & 7) ^ ((r >> 1) & 7)) < 4 ? (const uint16_t *)g_k_zeros : p; };
#pragma unroll
    for (int j = 0; j < LA; ++j) __builtin_amdgcn_global_load_lds((const void *)source(gpa[j], (wave * LA + j) * 8 + lrow), (lds_ptr)(sa + j * 8 * BK), 16, 0, 0);
#pragma unroll
    for (int j = 0; j < LB; ++j) __builtin_amdgcn_global_load_lds((const void *)source(gpb[j], (wave * LB + j) * 8 + lrow), (lds_ptr)(sb + j * 8 * BK), 16, 0, 0);
  }
#pragma unroll
  for (int st = 1; st < NS; ++st) issue(st < KT ? st : KT - 1, st);   // (half: two stages or more)
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NS - 1) * (LA + LB)) : "memory");   // stage 0 has landed (this wave's part)
  __builtin_amdgcn_s_barrier();

  const int frow = (lane & 31) * BK, sw = (lane >> 1) & 7, hi = lane >> 5;   // fragment rows start at multiples of 32
  int coff[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) coff[ks] = ((ks * 2 + hi) ^ sw) << 3;
  const int a_off = wm * WM * BK + frow, b_off = BM * BK + wn * WN * BK + frow;
  bf16x8 fa0[MT], fb0[NT], fa1[MT], fb1[NT];
#define RAI_K64_READ(FA, FB, BUF, KS)                                                                     \
  do {                                                                                                    \
    const uint16_t *as_ = lds + (BUF) * STAGE + a_off + coff[KS], *bs_ = lds + (BUF) * STAGE + b_off + coff[KS]; \
    _Pragma("unroll") for (int i = 0; i < MT; ++i) FA[i] = *reinterpret_cast<const bf16x8 *>(as_ + i * 32 * BK); \
    _Pragma("unroll") for (int j = 0; j < NT; ++j) FB[j] = *reinterpret_cast<const bf16x8 *>(bs_ + j * 32 * BK); \
  } while (0)
#define RAI_K64_MUL(FA, FB)                                                                    \
  do {                                                                                         \
    _Pragma("unroll") for (int i = 0; i < MT; ++i)                                             \
      _Pragma("unroll") for (int j = 0; j < NT; ++j)                                           \
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(FA[i], FB[j], acc[i][j], 0, 0, 0); \
  } while (0)
  // one LDS read between every MT*NT/(MT+NT) multiplies: a wave issues in order, so whatever sits between two
  // batches of MFMAs runs with the matrix pipe idle
#define RAI_K64_MIX_READS()                                                                                \
  do {                                                                                                     \
    _Pragma("unroll") for (int g = 0; g < MT + NT; ++g) {                                                  \
      __builtin_amdgcn_sched_group_barrier(0x008, MT * NT / (MT + NT) > 0 ? MT * NT / (MT + NT) : 1, 0);   \
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);                                                   \
    }                                                                                                      \
    __builtin_amdgcn_sched_barrier(0);                                                                     \
  } while (0)
  RAI_K64_READ(fa0, fb0, 0, 0);
  // Every stage but the last in one straight-line block (a branch around the multiplies would split the
  // scheduling region and leave copies of the accumulators at the join).
  int cur = 0;
  for (int st = 0; st + 1 < KT; ++st) {
    const int next = NS == 2 ? cur ^ 1 : cur + 1 < NS ? cur + 1 : 0;
    RAI_K64_READ(fa1, fb1, cur, 1);
    RAI_K64_MUL(fa0, fb0);
    RAI_K64_MIX_READS();
    RAI_K64_READ(fa0, fb0, cur, 2);
    RAI_K64_MUL(fa1, fb1);
    RAI_K64_MIX_READS();
    RAI_K64_READ(fa1, fb1, cur, 3);
    RAI_K64_MUL(fa0, fb0);
    RAI_K64_MIX_READS();
    // stage st+1 has landed (requested NS-1 stages ago) and this wave's reads of stage st are done: after the barrier
    // stage st belongs to the loads of stage st+NS (past the end: the last stage once more, into a buffer nobody reads)
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((NS - 2) * (LA + LB)) : "memory");
    __builtin_amdgcn_s_barrier();
    issue(st + NS < KT ? st + NS : KT - 1, cur);
    RAI_K64_READ(fa0, fb0, next, 0);
    RAI_K64_MUL(fa1, fb1);
#pragma unroll
    for (int g = 0; g < MT + NT; ++g) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // MFMA
      __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);   // one global -> LDS load
      __builtin_amdgcn_sched_group_barrier(0x008, MT * NT / (MT + NT) > 1 ? MT * NT / (MT + NT) - 1 : 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);   // one LDS read
    }
    __builtin_amdgcn_sched_barrier(0);
    cur = next;
  }
  {
    RAI_K64_READ(fa1, fb1, cur, 1);
    RAI_K64_MUL(fa0, fb0);
    RAI_K64_MIX_READS();
    RAI_K64_READ(fa0, fb0, cur, 2);
    RAI_K64_MUL(fa1, fb1);
    RAI_K64_MIX_READS();
    RAI_K64_READ(fa1, fb1, cur, 3);
    RAI_K64_MUL(fa0, fb0);
    RAI_K64_MIX_READS();
    RAI_K64_MUL(fa1, fb1);
  }
#undef RAI_K64_READ
#undef RAI_K64_MUL
#undef RAI_K64_MIX_READS
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
}

template <int BM, int BN, int NS, int SH, int WGN, int WGM, bool ODD>
__global__ void __launch_bounds__(64 * WGM * WGN) k_gemm_bf16_mfma_dma(LinearArgs a, int longer, int k_per_split, float *partial) {
  // block = 2 x WGN waves.  WGN = 4 (eight waves, wave tile (BM/2) x (BN/4)) keeps two waves on every SIMD: one
  // multiplies while the other sits in its wait for the next tile, and twice as many waves issue loads.
  constexpr int BK = 32, PITCH = BK;
  extern __shared__ __attribute__((aligned(16))) uint16_t lds[];

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tiles_m = (a.M + BM - 1) / BM, tiles_n = (a.N + BN - 1) / BN;
  const int total = tiles_m * tiles_n;
  const int tile = xcd_remap(blockIdx.x, total);
  if (tile >= total) return;
  int tile_m, tile_n;
  tile_coords(tile, tiles_m, tiles_n, &tile_m, &tile_n);
  const int m0 = tile_m * BM, n0 = tile_n * BN;
  const int split = blockIdx.y;
  int k_begin = split * k_per_split, k_span = k_per_split;
  if constexpr (SH == 0) {   // stages of 64: the first `longer` parts take one more (parts of 32s count none: 0.5 us)
    k_begin += (split < longer ? split : longer) * 64;
    k_span += split < longer ? 64 : 0;
  }
  // (stages of 64: K in whole stages, of which the first may begin 32 before it; ODD: 32, but with the constant small products take 0.1 to
  // 0.2 us more, 500 x 1000 x 992 8.6, 8.9)
  const int early = SH == 0 && ODD ? a.K & 32 : 0;
  const int k_end = k_begin + k_span < a.K + early ? k_begin + k_span : a.K + early;
  const int KT = (k_end - k_begin) / BK;

  f32x16 acc[BM / (32 * WGM)][BN / (32 * WGN)];
  if constexpr (SH == 0) {   // stages of 64 (the launcher sends splits of whole stages here)
    dma_tile_mainloop_k64<BM, BN, WGN, WGM, NS>(a, lds, m0, n0, k_begin - early, KT / 2, wave, lane, acc, early && split == 0);
  } else {
    static_assert(WGM == 2, "the K-32 loop is written for two waves along M");
    dma_tile_mainloop<BM, BN, NS, SH, WGN>(a, lds, m0, n0, k_begin, KT, wave, lane, acc);
  }
  gemm_tile_epilogue<BM, BN, dma_lds_bytes<BM, BN, NS, WGN, WGM, SH>(), WGN, WGM>(a, acc, lds, m0, n0, wave, lane, split, partial);
}

// The same tile over the rows of one expert (see MoePlan): a block finds its expert and rows in the device-side table,
// whose length only the device knows; the grid covers the largest it can be and the blocks behind the end leave.
template <int BM, int BN, int WGN>
__global__ void __launch_bounds__(128 * WGN) k_gemm_bf16_mfma_grouped(LinearArgs a, int64_t w_stride, const int4 *table, const int *n_tiles) {
  extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tiles_m = *n_tiles, tiles_n = (a.N + BN - 1) / BN;
  const int total = tiles_m * tiles_n;
  if ((int)blockIdx.x >= (total + kXcds - 1) / kXcds * kXcds) return;
  const int tile = xcd_remap(blockIdx.x, total);
  if (tile >= total) return;
  // an XCD's run walks all column tiles of one row tile group: the experts' weights are read once, their rows from L2
  int tile_m, tile_n;
  tile_coords(tile, tiles_m, tiles_n, &tile_m, &tile_n);
  const int4 t = table[tile_m];
  a.A = (const uint16_t *)a.A + (int64_t)t.y * a.lda;
  a.W = (const uint16_t *)a.W + (int64_t)t.x * w_stride;
  a.out1 = (uint16_t *)a.out1 + (int64_t)t.y * a.ld1;
  a.M = t.z;
  f32x16 acc[BM / 64][BN / (32 * WGN)];
  dma_tile_mainloop_k64<BM, BN, WGN>(a, lds, 0, tile_n * BN, 0, a.K / 64, wave, lane, acc);
  gemm_tile_epilogue<BM, BN, dma_lds_bytes<BM, BN, 2, WGN>(), WGN>(a, acc, lds, 0, tile_n * BN, wave, lane, 0, nullptr);
}

// ---- stream-K form of the eight-wave 256x256 tile kernel ---------------------------------------------------------
// One block per CU.  When the tile count is not a multiple of the CU count, the last partial round would leave CUs
// idle for a whole tile time (140 tiles on 256 CUs: 45 % of the machine).  Here the K tiles of those `sk_tiles` tiles
// are dealt out evenly instead: block p (in XCD order, so neighbours share an L2) takes units [start(p), start(p+1))
// of the sk_tiles * KT (tile, K tile) units, i.e. the tail of one tile and the head of the next.  A tile is then the
// work of two or three blocks: each stores its f32 accumulators to its slot of the workspace in register order
// with device-scope stores and counts itself in; the block that arrives
// last adds the slots in slot order (so the sum does not depend on who was last) and runs the epilogue.  It alone
// waits, for stores under way, and not for ever.  The remaining tiles follow in whole rounds, one tile per block as before.
//   With stages of 64 this is the form for operands that stay in no cache (persists() below), else gemm_persist.hip's.
template <int NS>   // four stages of 32, two of 64
__global__ void __launch_bounds__(512) k_gemm_bf16_mfma_dma_streamk(LinearArgs a, StreamKArgs sk) {
  constexpr int BM = 256, BN = 256, SH = 2, WGN = 4, BK = NS == 2 ? 64 : 32;   // the unit of sharing is one K tile of the main loop
  constexpr int MT = BM / 64, NT = BN / (32 * WGN);
  constexpr int LDS_BYTES = dma_lds_bytes<BM, BN, NS, WGN>();
  extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
  __shared__ int s_ticket;

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tiles_m = (a.M + BM - 1) / BM, tiles_n = (a.N + BN - 1) / BN;
  const int total = tiles_m * tiles_n;
  const int KT = a.K / BK;
  const int P = gridDim.x;
  const int p = xcd_remap(blockIdx.x, P);   // P is a multiple of the XCD count
  f32x16 acc[MT][NT];

  // one loop over this block's segments (shares of tiles first, then whole tiles), so that the K loop and the
  // epilogue are instantiated once
  int u = sk_start(sk, p);
  const int u_end = sk_start(sk, p + 1);
  int whole = sk.sk_tiles + p;
  for (;;) {
    int tile, kt0, kt1;
    if (u < u_end) {
      tile = u / KT;
      kt0 = u - tile * KT;
      kt1 = kt0 + (u_end - u) < KT ? kt0 + (u_end - u) : KT;
      u += kt1 - kt0;
    } else if (whole < total) {
      tile = whole;
      kt0 = 0;
      kt1 = KT;
      whole += P;
    } else {
      break;
    }
    int tile_m, tile_n;
    tile_coords(tile, tiles_m, tiles_n, &tile_m, &tile_n);
    const int m0 = tile_m * BM, n0 = tile_n * BN;
    __syncthreads();   // the previous segment's epilogue staging is done with the LDS
    if constexpr (NS == 2) dma_tile_mainloop_k64<BM, BN, WGN>(a, lds, m0, n0, kt0 * BK, kt1 - kt0, wave, lane, acc);
    else dma_tile_mainloop<BM, BN, NS, SH, WGN>(a, lds, m0, n0, kt0 * BK, kt1 - kt0, wave, lane, acc);
    if (kt1 - kt0 != KT && !sum_shares(sk, acc, &s_ticket, tile, KT, p, wave, lane)) continue;
    gemm_tile_epilogue<BM, BN, LDS_BYTES, WGN>(a, acc, lds, m0, n0, wave, lane, 0, nullptr);
  }
}

// Sums the per-split partial products and applies the Linear epilogue: four columns of a row to a thread, P of its parts asked for at a time
// and added in their order.  Bound by the partial sums' way through the caches.  Measured
// against an element at a time, the whole product (us): 333 x 8960 x 1536 of five parts 26.5 -> 24.4, 131 x 8512 x 5936 38.6 -> 36.4, 70 x 3072 x 1000
// 10.1 -> 9.2, 800 x 16384 x 2048 71.4 -> 68.9.
typedef __attribute__((ext_vector_type(2))) uint32_t sum_u32x2;
template <int P>
__global__ void __launch_bounds__(256) k_splitk_epilogue(LinearArgs a, int splits, const float *partial) {
  const uint32_t total = (uint32_t)a.M * (uint32_t)a.N, row_quads = (uint32_t)a.N / 4, q = blockIdx.x * 256 + threadIdx.x;   // (fewer than 2^32 floats)
  if (q >= total / 4) return;
  const int m = (int)(q / row_quads), n = (int)(q % row_quads) * 4;
  const uint16_t *bias = (const uint16_t *)a.bias, *bias2 = (const uint16_t *)a.bias2, *res = (const uint16_t *)a.residual;
  sum_u32x2 b1 = {0u, 0u}, b2 = {0u, 0u}, rb = {0u, 0u};   // zero bits where there is none: +0.0
  f32x4 rf = {0.f, 0.f, 0.f, 0.f};
  if (bias) b1 = *reinterpret_cast<const sum_u32x2 *>(bias + n);
  if (bias2) b2 = *reinterpret_cast<const sum_u32x2 *>(bias2 + n);
  if (a.residual && a.f32_out) rf = *reinterpret_cast<const f32x4 *>((const float *)a.residual + (int64_t)m * a.ldr + n);
  else if (a.residual) rb = *reinterpret_cast<const sum_u32x2 *>(res + (int64_t)m * a.ldr + n);
  float x[4] = {0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < splits; s0 += P) {
    f32x4 p[P];
#pragma unroll
    for (int u = 0; u < P; ++u) p[u] = *reinterpret_cast<const f32x4 *>(partial + (size_t)min(s0 + u, splits - 1) * total + 4 * (size_t)q);
#pragma unroll
    for (int u = 0; u < P; ++u)
      if (s0 + u < splits) {
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] += p[u][e];
      }
  }
  auto half = [](sum_u32x2 v, int e) { return bf16_bits_to_f32((uint16_t)(v[e >> 1] >> (e & 1) * 16)); };
  if (a.glu) {   // two (gate, up) pairs
    uint32_t o = 0;
#pragma unroll
    for (int e = 0; e < 4; e += 2) o |= (uint32_t)f32_to_bf16_bits(glu_bf16(a, x[e] + half(b1, e), x[e + 1] + half(b1, e + 1))) << 8 * e;
    *reinterpret_cast<uint32_t *>((uint16_t *)a.out1 + (int64_t)m * a.ld1 + (n >> 1)) = o;
    return;
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) x[e] += half(b1, e) + half(b2, e);
  if (a.act >= 0) act_exact<4>(a.act, x, n, a.act_from);
  if (a.f32_out) {
    f32x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = fmaf(a.out_scale, x[e], rf[e]);
    *reinterpret_cast<f32x4 *>((float *)a.out1 + (int64_t)m * a.ld1 + n) = o;
    return;
  }
  if (res) {
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] += half(rb, e);
  }
  const sum_u32x2 o = {(uint32_t)f32_to_bf16_bits(x[0]) | (uint32_t)f32_to_bf16_bits(x[1]) << 16,
                   (uint32_t)f32_to_bf16_bits(x[2]) | (uint32_t)f32_to_bf16_bits(x[3]) << 16};
  uint16_t *dst = n < a.n_split ? (uint16_t *)a.out1 + (int64_t)m * a.ld1 + n : (uint16_t *)a.out2 + (int64_t)m * a.ld2 + (n - a.n_split);
  *reinterpret_cast<sum_u32x2 *>(dst) = o;
}

// The same an element at a time: where a piece below would be cut or off its boundary.
__global__ void __launch_bounds__(256) k_splitk_epilogue_any(LinearArgs a, int splits, const float *partial) {
  const int64_t total = (int64_t)a.M * a.N;
  const uint16_t *bias = (const uint16_t *)a.bias;
  const uint16_t *bias2 = (const uint16_t *)a.bias2;
  const uint16_t *res = (const uint16_t *)a.residual;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total; e += (int64_t)gridDim.x * blockDim.x) {
    const int m = (int)(e / a.N), n = (int)(e % a.N);
    if (a.glu) {
      if (n & 1) continue;
      float g = 0.f, u = 0.f;
      for (int s = 0; s < splits; ++s) { g += partial[(int64_t)s * total + e]; u += partial[(int64_t)s * total + e + 1]; }
      g += bias ? bf16_bits_to_f32(bias[n]) : 0.f;
      u += bias ? bf16_bits_to_f32(bias[n + 1]) : 0.f;
      ((uint16_t *)a.out1)[(int64_t)m * a.ld1 + (n >> 1)] = f32_to_bf16_bits(glu_bf16(a, g, u));
      continue;
    }
    float x = 0.f;
    for (int s = 0; s < splits; ++s) x += partial[(int64_t)s * total + e];
    x += (bias ? bf16_bits_to_f32(bias[n]) : 0.f) + (bias2 ? bf16_bits_to_f32(bias2[n]) : 0.f);
    if (a.act >= 0 && n >= a.act_from) x = act_eval(a.act, x);
    if (a.f32_out) {
      ((float *)a.out1)[(int64_t)m * a.ld1 + n] = fmaf(a.out_scale, x, res ? ((const float *)a.residual)[(int64_t)m * a.ldr + n] : 0.f);
      continue;
    }
    if (res) x += bf16_bits_to_f32(res[(int64_t)m * a.ldr + n]);
    if (n < a.n_split) ((uint16_t *)a.out1)[(int64_t)m * a.ld1 + n] = f32_to_bf16_bits(x);
    else ((uint16_t *)a.out2)[(int64_t)m * a.ld2 + (n - a.n_split)] = f32_to_bf16_bits(x);
  }
}

// The same pass for a Linear whose output rows are normalised next.  A block of four waves owns a row (N <= 512 *
// ITEMS columns).  The sums over the partial products, bias / activation / residual and the bf16 store are element
// by element, so they are shared out: every wave takes a quarter of the row's 16-byte packs (512 rows are then eight
// waves per CU with one round of loads each, instead of two waves with two rounds).  The stored (rounded) row goes
// through LDS to the block, which runs LayerNorm on it with the arithmetic of the stand-alone norm kernel's block form -- same
// order in a thread, same reductions -- so fusing changes no bit (rai-nn/src/layer_norm.rs:32-42) as long as that form serves the rows.
template <int ITEMS>
__global__ void __launch_bounds__(256) k_splitk_epilogue_ln(LinearArgs a, int splits, const float *partial) {
  constexpr int NWV = 4;                                 // waves per row
  constexpr int JT = (ITEMS * 64 / NWV + 63) / 64;       // packs per lane in the summing part
  constexpr int NI = (ITEMS + 3) / 4;                    // packs per thread in the norm
  __shared__ u32x4 rowbuf[64 * ITEMS];
  __shared__ float sums[2][4];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int row = blockIdx.x;
  const int packs = a.N / 8;
  const uint16_t *lw = (const uint16_t *)a.post_ln_w, *lb = (const uint16_t *)a.post_ln_b;
  u32x4 lwr[NI], lbr[NI];   // the norm's weights, asked for with everything else
#pragma unroll
  for (int it = 0; it < NI; ++it) {
    const int p = threadIdx.x + it * 256 < packs ? threadIdx.x + it * 256 : 0;
    if (lw) lwr[it] = *reinterpret_cast<const u32x4 *>(lw + p * 8);
    if (lb) lbr[it] = *reinterpret_cast<const u32x4 *>(lb + p * 8);
  }
  const int quarter = (packs + NWV - 1) / NWV;
  const int64_t total = (int64_t)a.M * a.N;
  const uint16_t *bias = (const uint16_t *)a.bias, *bias2 = (const uint16_t *)a.bias2;
  const uint16_t *res = (const uint16_t *)a.residual;
  {
    // loads are issued as early and as many at a time as the registers allow: bias and residual first, then the
    // partial products of all the lane's packs (six splits each), while every element's additions stay in split order
    int pk[JT];
    bool on[JT];
    u32x4 braw[JT], b2raw[JT], rraw[JT];
    float x[JT][8];
#pragma unroll
    for (int j = 0; j < JT; ++j) {
      const int q = lane + j * 64;
      pk[j] = wv * quarter + q;
      on[j] = q < quarter && pk[j] < packs;
      if (!on[j]) pk[j] = 0;   // a clamped pack is loaded and never used
      const int n = pk[j] * 8;
      braw[j] = b2raw[j] = rraw[j] = u32x4{0u, 0u, 0u, 0u};
      if (bias) braw[j] = *reinterpret_cast<const u32x4 *>(bias + n);
      if (bias2) b2raw[j] = *reinterpret_cast<const u32x4 *>(bias2 + n);
      if (res) rraw[j] = *reinterpret_cast<const u32x4 *>(res + (int64_t)row * a.ldr + n);
#pragma unroll
      for (int e = 0; e < 8; ++e) x[j][e] = 0.f;
    }
    for (int s0 = 0; s0 < splits; s0 += 6) {
      f32x4 p0[JT][6], p1[JT][6];
#pragma unroll
      for (int j = 0; j < JT; ++j)
#pragma unroll
        for (int u = 0; u < 6; ++u) {
          const int sp = s0 + u < splits ? s0 + u : splits - 1;
          const float *pp = partial + (int64_t)sp * total + (int64_t)row * a.N + pk[j] * 8;
          p0[j][u] = *reinterpret_cast<const f32x4 *>(pp);
          p1[j][u] = *reinterpret_cast<const f32x4 *>(pp + 4);
        }
#pragma unroll
      for (int j = 0; j < JT; ++j)
#pragma unroll
        for (int u = 0; u < 6; ++u) {
          if (s0 + u < splits) {
            x[j][0] += p0[j][u].x; x[j][1] += p0[j][u].y; x[j][2] += p0[j][u].z; x[j][3] += p0[j][u].w;
            x[j][4] += p1[j][u].x; x[j][5] += p1[j][u].y; x[j][6] += p1[j][u].z; x[j][7] += p1[j][u].w;
          }
        }
    }
#pragma unroll
    for (int j = 0; j < JT; ++j) {
      if (on[j]) {
        const int n = pk[j] * 8;
        float b1[8], b2[8];
        unpack8(braw[j], b1);     // zero bits where there is no bias: +0.0
        unpack8(b2raw[j], b2);
#pragma unroll
        for (int e = 0; e < 8; ++e) x[j][e] += b1[e] + b2[e];
        if (a.act >= 0) act8(a.act, x[j], n, a.act_from);
        if (res) {
          float rv[8];
          unpack8(rraw[j], rv);
#pragma unroll
          for (int e = 0; e < 8; ++e) x[j][e] += rv[e];
        }
        u32x4 o;
        o.x = (uint32_t)f32_to_bf16_bits(x[j][0]) | ((uint32_t)f32_to_bf16_bits(x[j][1]) << 16);
        o.y = (uint32_t)f32_to_bf16_bits(x[j][2]) | ((uint32_t)f32_to_bf16_bits(x[j][3]) << 16);
        o.z = (uint32_t)f32_to_bf16_bits(x[j][4]) | ((uint32_t)f32_to_bf16_bits(x[j][5]) << 16);
        o.w = (uint32_t)f32_to_bf16_bits(x[j][6]) | ((uint32_t)f32_to_bf16_bits(x[j][7]) << 16);
        *reinterpret_cast<u32x4 *>((uint16_t *)a.out1 + (int64_t)row * a.ld1 + n) = o;
        rowbuf[pk[j]] = o;
      }
    }
  }
  __syncthreads();
  // ---- LayerNorm of the stored row: thread t has packs t, t + 256, ..
  float v[NI][8], s = 0.f;
#pragma unroll
  for (int it = 0; it < NI; ++it) {
    const int p = threadIdx.x + it * 256;
    if (p < packs) unpack8(rowbuf[p], v[it]);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      if (p >= packs) v[it][e] = 0.f;
      s += v[it][e];
    }
  }
  auto block_sum = [&](float x, float (&part)[4]) {
    x = wave_sum(x);
    if (lane == 0) part[wv] = x;
    __syncthreads();
    return (part[0] + part[1]) + (part[2] + part[3]);
  };
  const float mean = block_sum(s, sums[0]) / (float)a.N;
  s = 0.f;
#pragma unroll
  for (int it = 0; it < NI; ++it)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float d = threadIdx.x + it * 256 < packs ? v[it][e] - mean : 0.f;
      s += d * d;
    }
  const float scale = 1.0f / sqrtf(block_sum(s, sums[1]) / (float)a.N + a.post_ln_eps);
#pragma unroll
  for (int it = 0; it < NI; ++it) {
    const int p = threadIdx.x + it * 256;
    if (p < packs) {
      float wf[8], bf[8];
      if (lw) unpack8(lwr[it], wf);
      if (lb) unpack8(lbr[it], bf);
      uint32_t h[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float y = (v[it][e] - mean) * scale;
        if (lw) y *= wf[e];
        if (lb) y += bf[e];
        h[e] = f32_to_bf16_bits(y);
      }
      u32x4 o = {h[0] | (h[1] << 16), h[2] | (h[3] << 16), h[4] | (h[5] << 16), h[6] | (h[7] << 16)};
      *reinterpret_cast<u32x4 *>((uint16_t *)a.post_ln_out + (int64_t)row * a.N + p * 8) = o;
    }
  }
}

// Whether the pass over the partial sums can also normalise the rows: one ungated output, whole 16-byte packs.
static bool post_norm_fits(const LinearArgs &a) {
  auto al16 = [](const void *p) { return ((uintptr_t)p & 15) == 0; };
  return a.post_ln_out && !a.glu && !a.f32_out && a.n_split >= a.N && a.N % 8 == 0 && a.N <= 4096 && a.ld1 % 8 == 0 && al16(a.out1) &&
         al16(a.post_ln_out) && (!a.bias || al16(a.bias)) && (!a.bias2 || al16(a.bias2)) &&
         (!a.residual || (a.ldr % 8 == 0 && al16(a.residual))) && (!a.post_ln_w || al16(a.post_ln_w)) &&
         (!a.post_ln_b || al16(a.post_ln_b)) && a.splitk_ws && ((uintptr_t)a.splitk_ws & 15) == 0;
}
// Whether whole pieces of four columns lie on their boundaries in the partial sums and everything they meet.
static bool quads_fit(const LinearArgs &a, const float *partial) {
  auto al = [](const void *p, int64_t ld, unsigned bytes, unsigned size) { return ((uintptr_t)p & (bytes - 1)) == 0 && ld * size % bytes == 0; };
  if (a.N % 4 || (int64_t)a.M * a.N >= (int64_t)1 << 32 || ((uintptr_t)partial & 15) || !al(a.bias, 0, 8, 2) || !al(a.bias2, 0, 8, 2)) return false;
  if (a.glu) return al(a.out1, a.ld1, 4, 2);
  if (a.f32_out) return al(a.out1, a.ld1, 16, 4) && al(a.residual, a.residual ? a.ldr : 0, 16, 4);
  return al(a.out1, a.ld1, 8, 2) && al(a.residual, a.residual ? a.ldr : 0, 8, 2) && (a.n_split >= a.N || (a.n_split % 4 == 0 && al(a.out2, a.ld2, 8, 2)));
}
static int launch_sum_of_parts(hipStream_t st, const LinearArgs &a, int splits, const float *partial) {
  const int64_t total = (int64_t)a.M * a.N;
  if (quads_fit(a, partial)) {
    const dim3 grid((unsigned)((total / 4 + 255) / 256)), block(256);
    if (splits == 2) hipLaunchKernelGGL(k_splitk_epilogue<2>, grid, block, 0, st, a, splits, partial);
    else if (splits == 3) hipLaunchKernelGGL(k_splitk_epilogue<3>, grid, block, 0, st, a, splits, partial);
    else hipLaunchKernelGGL(k_splitk_epilogue<4>, grid, block, 0, st, a, splits, partial);
    return launch_check("splitk_epilogue");
  }
  const int blocks = (int)((total + 255) / 256 < 4096 ? (total + 255) / 256 : 4096);
  hipLaunchKernelGGL(k_splitk_epilogue_any, dim3(blocks), dim3(256), 0, st, a, splits, partial);
  return launch_check("splitk_epilogue");
}
// Sums the partial products of a tile GEMM that split K (and normalises the rows when asked to and possible).
static int launch_splitk_epilogue(hipStream_t st, const LinearArgs &a, int splits, const float *partial) {
  if (post_norm_fits(a)) {
    const int items = (a.N / 8 + 63) / 64;
    const dim3 grid(a.M), block(256);
    if (items <= 2) hipLaunchKernelGGL(k_splitk_epilogue_ln<2>, grid, block, 0, st, a, splits, partial);
    else if (items <= 5) hipLaunchKernelGGL(k_splitk_epilogue_ln<5>, grid, block, 0, st, a, splits, partial);
    else hipLaunchKernelGGL(k_splitk_epilogue_ln<8>, grid, block, 0, st, a, splits, partial);
    return launch_check("splitk_epilogue_ln");
  }
  return launch_sum_of_parts(st, a, splits, partial);
}

template <int BM, int BN, int BK, int SH = 0> static int launch_cfg(hipStream_t st, const LinearArgs &a, int splits) {
  constexpr size_t lds = gemm_lds_bytes<BM, BN, (SH ? BK : BK + 8)>();
  static bool attr_set = false;
  if (lds > 64 * 1024 && !attr_set) {
    RAI_HIP_TRY(hipFuncSetAttribute((const void *)k_gemm_bf16_mfma<BM, BN, BK, SH>,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    attr_set = true;
  }
  const int tiles = ((a.M + BM - 1) / BM) * ((a.N + BN - 1) / BN);
  const int grid_x = ((tiles + kXcds - 1) / kXcds) * kXcds;  // whole rounds over the XCDs
  int k_per_split = a.K;
  float *partial = nullptr;
  if (splits > 1) {
    const int k_tiles = a.K / BK, per = (k_tiles + splits - 1) / splits;
    splits = (k_tiles + per - 1) / per;  // every split gets at least one K tile
    k_per_split = per * BK;
    partial = (float *)a.splitk_ws;
  }
  hipLaunchKernelGGL((k_gemm_bf16_mfma<BM, BN, BK, SH>), dim3(grid_x, splits), dim3(256), lds, st, a, splits, k_per_split,
                     partial);
  RAI_TRY(launch_check("gemm_bf16_mfma"));
  if (splits > 1) RAI_TRY(launch_splitk_epilogue(st, a, splits, (const float *)partial));
  return RAI_OK;
}

template <int BM, int BN, int NS, int SH, int WGN, int WGM, bool ODD>
static int launch_cfg_dma_k(hipStream_t st, const LinearArgs &a, int splits) {
  constexpr size_t lds = dma_lds_bytes<BM, BN, NS, WGN, WGM, SH>();
  static bool attr_set = false;
  if (lds > 64 * 1024 && !attr_set) {
    RAI_HIP_TRY(hipFuncSetAttribute((const void *)k_gemm_bf16_mfma_dma<BM, BN, NS, SH, WGN, WGM, ODD>,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    attr_set = true;
  }
  const int tiles = ((a.M + BM - 1) / BM) * ((a.N + BN - 1) / BN);
  const int grid_x = ((tiles + kXcds - 1) / kXcds) * kXcds;
  const int stages = (a.K + 32) / 64;
  int k_per_split = SH == 0 ? stages * 64 : a.K, longer = 0;
  const int most = stages - ODD;   // the part whose first stage begins before the rows has a second one
  if (SH == 0 && splits > most) splits = most;
  if (splits > 1) {
    if constexpr (SH == 0) {   // stages of 64, dealt out evenly
      k_per_split = stages / splits * 64;
      longer = stages % splits;
    } else {
      const int k_tiles = a.K / 32, per = (k_tiles + splits - 1) / splits;
      splits = (k_tiles + per - 1) / per;
      k_per_split = per * 32;
    }
  }
  float *partial = splits > 1 ? (float *)a.splitk_ws : nullptr;
  hipLaunchKernelGGL((k_gemm_bf16_mfma_dma<BM, BN, NS, SH, WGN, WGM, ODD>), dim3(grid_x, splits), dim3(64 * WGM * WGN), lds, st, a,
                     longer, k_per_split, partial);
  RAI_TRY(launch_check("gemm_bf16_mfma_dma"));
  if (splits > 1) RAI_TRY(launch_splitk_epilogue(st, a, splits, (const float *)partial));
  return RAI_OK;
}
template <int BM, int BN, int NS, int SH, int WGN = 2, int WGM = 2> static int launch_cfg_dma(hipStream_t st, const LinearArgs &a, int splits) {
  if constexpr (SH == 0) {
    if (a.K % 64) return launch_cfg_dma_k<BM, BN, NS, SH, WGN, WGM, true>(st, a, splits);
  }
  return launch_cfg_dma_k<BM, BN, NS, SH, WGN, WGM, false>(st, a, splits);
}

// Arrival counters of the stream-K kernel, one per shared tile; every launch leaves them at zero.
static __device__ int g_streamk_counters[4 * kNumCU];

// How the stream-K kernel would share out an M x N x K product: false when it does not apply (tile count a multiple
// of the CU count, too few tiles, or a tile would be the work of more than three blocks).  Whether it pays: streamk_us,
// streamk_pays_k32.
struct StreamKPlan {
  StreamKArgs k;
  size_t ws_bytes;
};
static bool streamk_plan(int M, int N, int K, int bk, StreamKPlan *plan) {
  const int P = kNumCU, KT = K / bk;
  const int T = ((M + 255) / 256) * ((N + 255) / 256);
  const int full = T / P, left = T % P;
  if (left == 0 || K / 32 < 8) return false;
  int sk_tiles = left;
  if (left < P / 2) {
    if (full == 0) return false;
    sk_tiles = left + P;   // a whole round joins the shared part: every block then works on two tiles at most
  }
  const long long units = (long long)sk_tiles * KT;
  StreamKArgs k;
  k.sk_tiles = sk_tiles;
  k.q = (int)(units / P);
  k.rem = (int)(units % P);
  if (k.q < 1) return false;
  auto block_of = [&](int u) {
    const int big = k.rem * (k.q + 1);
    return u < big ? u / (k.q + 1) : k.rem + (u - big) / k.q;
  };
  int max_parts = 1;
  for (int t = 0; t < sk_tiles; ++t) {
    const int parts = block_of(t * KT + KT - 1) - block_of(t * KT) + 1;
    if (parts > max_parts) max_parts = parts;
  }
  if (max_parts > 3 || sk_tiles > 2 * kNumCU) return false;
  k.max_parts = max_parts;
  k.ws = nullptr;
  k.counters = nullptr;
  plan->k = k;
  plan->ws_bytes = (size_t)sk_tiles * max_parts * 256 * 256 * sizeof(float);
  return true;
}

static int linear_device(const LinearArgs &a, int *dev) {
  *dev = a.dev;
  if (*dev < 0) RAI_HIP_TRY(hipGetDevice(dev));
  RAI_REQUIRE(*dev >= 0 && *dev < 64, RAI_ERR_BAD_ARG, "device %d out of range", *dev);
  return RAI_OK;
}

// True when the stream-K kernel can serve this Linear (plain tile epilogue, workspace large enough, not switched off).
static bool streamk_applies(const LinearArgs &a, int bk, StreamKPlan *plan) {
  const char *off = getenv("RAI_HIP_NO_STREAMK");   // read per call: tests compare both forms in one process
  if (off && *off && *off != '0') return false;
  if (!a.splitk_ws || ((uintptr_t)a.splitk_ws & 15) || a.post_ln_out) return false;
  // one block per CU of a 256-CU part: the plan, the counter array and the XCD order are laid out for that grid
  int dev = -1;
  if (linear_device(a, &dev) != RAI_OK || device_cu_count(dev) != kNumCU) return false;
  return a.K % bk == 0 && streamk_plan(a.M, a.N, a.K, bk, plan) && plan->ws_bytes <= a.splitk_ws_bytes;
}

// every GPU holds its own copy of a __device__ array at its own address: looked up once per device
template <typename Sym> static int *device_ints_of(int dev, int *(&cache)[64], const Sym &symbol) {
  if (dev < 0 || dev >= 64) return nullptr;
  if (!cache[dev]) {
    int cur = -1;
    void *p = nullptr;
    if (hipGetDevice(&cur) != hipSuccess || (cur != dev && hipSetDevice(dev) != hipSuccess)) return nullptr;
    if (hipGetSymbolAddress(&p, symbol) == hipSuccess) cache[dev] = (int *)p;
    if (cur != dev) (void)hipSetDevice(cur);
  }
  return cache[dev];
}
static int *streamk_counters_of(int dev) {
  static int *counters[64];
  return device_ints_of(dev, counters, HIP_SYMBOL(g_streamk_counters));
}
// Tickets of the small-M streaming Linear's K split, one per group of weight tiles; zero between launches (the block
// that takes a group's last ticket puts it back).  Launches that overlap on one GPU would share them: the library
// runs a device's work on one stream.
static __device__ int g_splitk_tickets[kSplitTickets];
static int *splitk_tickets_of(int dev) {
  static int *tickets[64];
  return device_ints_of(dev, tickets, HIP_SYMBOL(g_splitk_tickets));
}

int *splitk_tickets(const LinearArgs &a) {
  int dev = -1;
  return linear_device(a, &dev) == RAI_OK ? splitk_tickets_of(dev) : nullptr;
}

int streamk_counters_reset(int dev, hipStream_t st) {
  int *c = streamk_counters_of(dev), *t = splitk_tickets_of(dev);
  RAI_REQUIRE(c && t, RAI_ERR_HIP, "stream-K counters of device %d not found", dev);
  RAI_HIP_TRY(hipMemsetAsync(c, 0, sizeof(int) * 4 * kNumCU, st));
  RAI_HIP_TRY(hipMemsetAsync(t, 0, sizeof(int) * kSplitTickets, st));
  return RAI_OK;
}

template <int NS> static int launch_streamk_blocks(hipStream_t st, const LinearArgs &a, const StreamKArgs &sk, int dev) {
  constexpr size_t lds = dma_lds_bytes<256, 256, NS, 4>();
  static bool attr_set[64];
  if (!attr_set[dev]) {
    RAI_HIP_TRY(hipFuncSetAttribute((const void *)k_gemm_bf16_mfma_dma_streamk<NS>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    attr_set[dev] = true;
  }
  hipLaunchKernelGGL(k_gemm_bf16_mfma_dma_streamk<NS>, dim3(kNumCU), dim3(512), lds, st, a, sk);
  return launch_check("gemm_bf16_mfma_dma_streamk");
}

// Whether the 256 x 256 tiles of stages of 64 are those of one block per CU (gemm_persist.hip); otherwise a block has one tile, or stream-K's
// shares.  Those ask for a stage as soon as the one before the last is let go, all waves at once, and that is worth more where the operands
// outgrow the memory-side cache of 256 MB and come from HBM again and again.  Measured (us, blocks / one per CU): stream-K 16384 x 1536 x 8960
// (321 MB) 378, 386, 8032 x 8984 x 8832 (300 MB) 1019, 1051; whole 4318 x 16496 x 10432 (434 MB) 1269, 1277, 3784 x 15064 x 7680 (290 MB) 745, 760,
// 4426 x 6392 x 12544 (271 MB) 601, 611.  From 200 MB on either may be ahead (8803 x 5064 x 7744, 215 MB, 560, 543; 16384 x 1536 x 6144, 220 MB, by
// stream-K 260, 267), below one per CU is (4096 x 4096 x 12288 312, 289; 8192 x 7168 x 4096 397, 370).
//   With a residual one per CU has no such loss: a block's epilogue waits for its rows, there they are on their way (the same products 390,
// 386; 1066, 1074; 1325, 1313; 780, 771; 625, 620).  Behind other work 16384 x 1536 x 8960 is further ahead: four layers of width 1536, 16 x 1024
// tokens, 6680 us with blocks, 6575 with one per CU.
//   With stream-K's shares, which begin at different columns of K and so share less in the L2s, the line lies earlier, unless two whole rounds
// follow (us, blocks / one per CU): 1.5 rounds, 16384 x 1536 x 4608 (165 MB) 199, 200, x 5632 (202 MB) 235, 242, x 6144 258,
// 267, x 7168 304, 312, 8192 x 3072 x 8192 (185 MB) 320, 305, x 9216 (208 MB) 358, 366, x 10240 401, 418, 4096 x 6144 x 8192 (168 MB) 320, 304,
// x 10240 393, 393, x 12288 (252 MB) 471, 478; 2.5 rounds, 4096 x 10240 x 7168 (206 MB) 462, 463, x 8192 (235 MB) 526, 518.  With new_gelu x 1536 x 5632 249,
// 250, 8192 x 3072 x 9216 374, 378, x 10240 417, 426.
constexpr int64_t kPersistBytes = 256 << 20, kPersistShareBytes = 192 << 20;
static bool persists(const LinearArgs &a, bool shares = false) {
  const bool few = ((a.M + 255) / 256) * ((a.N + 255) / 256) < 2 * kNumCU;   // (shares and less than two whole rounds)
  return a.K % 64 == 0 && gemm_persist_serves(a) &&
         (((int64_t)a.M + a.N) * a.K * 2 <= (shares && few ? kPersistShareBytes : kPersistBytes) || (a.residual && gemm_persist_plain(a)));
}

static int launch_streamk(hipStream_t st, const LinearArgs &a, StreamKPlan plan, int bk) {
  int dev = 0;
  RAI_TRY(linear_device(a, &dev));
  plan.k.ws = (float *)a.splitk_ws;
  plan.k.counters = streamk_counters_of(dev);
  plan.k.fault = kernel_fault_word(dev);
  RAI_REQUIRE(plan.k.counters && plan.k.fault, RAI_ERR_HIP, "stream-K: device %d has no counters / fault word", dev);
  plan.k.spin_limit = 1 << 20;
  plan.k.drop_tile = -1;
  // RAI_HIP_STREAMK_TEST="<spin limit>,<tile>": a tiny wait and one tile whose shares are never counted, so that the
  // expiry path runs with every wave still exiting normally (read per launch; the tests set it around one call)
  if (const char *t = getenv("RAI_HIP_STREAMK_TEST")) {
    int lim = 0, tile = -1;
    if (sscanf(t, "%d,%d", &lim, &tile) == 2 && lim > 0) { plan.k.spin_limit = lim; plan.k.drop_tile = tile; }
  }
  if (bk == 32) return launch_streamk_blocks<4>(st, a, plan.k, dev);
  return persists(a, true) ? launch_gemm_bf16_persist(st, a, plan.k) : launch_streamk_blocks<2>(st, a, plan.k, dev);
}

// ---- small M (9..64 rows): weight streaming through 16x16x32 MFMA -----------------------
// The activations are tiny and the weights are read exactly once, so the kernel is a
// stream over W: every wave owns 16 weight rows and reads them straight from global
// memory in MFMA fragment order (lane l: row l%16, 8 consecutive k at 8*(l/16)), U
// fragments ahead of the multiply.  The activation rows sit in LDS (16-byte padded
// pitch: the fragment reads of 16 lanes hit distinct banks) and are the B operand, so
// accumulator register r of lane l is out[m = l%16][n = 4*(l/16) + r]: four consecutive
// columns per lane.  K may be split over blockIdx.y (f32 partial sums, summed by
// k_splitk_epilogue) so that narrow outputs still fill the chip.
template <int MT, int U>
__global__ void __launch_bounds__(256) k_linear_bf16_mfma_skinny(LinearArgs a, int k_per_split, int k_chunk,
                                                                 float *partial) {
  extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int split = blockIdx.y;
  const int kb = split * k_per_split;
  const int ke = kb + k_per_split < a.K ? kb + k_per_split : a.K;
  const int pitch = k_chunk + 8;
  const int n0 = (blockIdx.x * 4 + wave) * 16;
  int nrow = n0 + (lane & 15);
  nrow = nrow < a.N ? nrow : a.N - 1;  // clamped rows are computed and never stored
  const uint16_t *wrow = (const uint16_t *)a.W + (int64_t)nrow * a.ldw + (lane >> 4) * 8;
  const uint16_t *xfrag = lds + (lane & 15) * pitch + (lane >> 4) * 8;

  f32x4 acc[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};

  for (int kc0 = kb; kc0 < ke; kc0 += k_chunk) {
    const int clen = ke - kc0 < k_chunk ? ke - kc0 : k_chunk;  // multiple of 32
    const int cpr = clen >> 3;
    if (kc0 != kb) __syncthreads();
    for (int c = tid; c < MT * 16 * cpr; c += 256) {
      const int row = c / cpr, kc = (c - row * cpr) * 8;
      u32x4 v = {0u, 0u, 0u, 0u};
      if (row < a.M) v = *reinterpret_cast<const u32x4 *>((const uint16_t *)a.A + (int64_t)row * a.lda + kc0 + kc);
      *reinterpret_cast<u32x4 *>(lds + row * pitch + kc) = v;
    }
    const uint16_t *wp = wrow + kc0;
    bf16x8 w[U];
    const int full = clen / (32 * U);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (full > 0) w[u] = __builtin_nontemporal_load(reinterpret_cast<const bf16x8 *>(wp + u * 32));
    __syncthreads();
    int k = 0;
    for (int it = 0; it < full; ++it, k += 32 * U) {
      bf16x8 cur[U];
#pragma unroll
      for (int u = 0; u < U; ++u) cur[u] = w[u];
      if (it + 1 < full) {
#pragma unroll
        for (int u = 0; u < U; ++u)
          w[u] = __builtin_nontemporal_load(reinterpret_cast<const bf16x8 *>(wp + k + 32 * U + u * 32));
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          const bf16x8 x = *reinterpret_cast<const bf16x8 *>(xfrag + i * 16 * pitch + k + u * 32);
          acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(cur[u], x, acc[i], 0, 0, 0);
        }
    }
    for (; k < clen; k += 32) {
      const bf16x8 wv = __builtin_nontemporal_load(reinterpret_cast<const bf16x8 *>(wp + k));
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const bf16x8 x = *reinterpret_cast<const bf16x8 *>(xfrag + i * 16 * pitch + k);
        acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv, x, acc[i], 0, 0, 0);
      }
    }
  }

  const int n = n0 + 4 * (lane >> 4);
  if (n >= a.N) return;
  const uint16_t *bias = (const uint16_t *)a.bias;
  const uint16_t *bias2 = (const uint16_t *)a.bias2;
  const uint16_t *res = (const uint16_t *)a.residual;
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int m = i * 16 + (lane & 15);
    if (m >= a.M) continue;
    const float v[4] = {acc[i][0], acc[i][1], acc[i][2], acc[i][3]};
    if (partial) {
      float *p = partial + ((int64_t)split * a.M + m) * a.N + n;
      if (a.N % 4 == 0) *reinterpret_cast<f32x4 *>(p) = acc[i];
      else for (int e = 0; e < 4 && n + e < a.N; ++e) p[e] = v[e];
      continue;
    }
    if (a.glu) {  // columns n..n+3 are two (gate, up) pairs
      uint16_t *dst = (uint16_t *)a.out1 + (int64_t)m * a.ld1 + (n >> 1);
      for (int e = 0; e < 4 && n + e + 1 < a.N; e += 2) {
        const float g = v[e] + (bias ? bf16_bits_to_f32(bias[n + e]) : 0.f);
        const float u = v[e + 1] + (bias ? bf16_bits_to_f32(bias[n + e + 1]) : 0.f);
        dst[e >> 1] = f32_to_bf16_bits(glu_bf16(a, g, u));
      }
      continue;
    }
    for (int e = 0; e < 4 && n + e < a.N; ++e) {
      const int nn = n + e;
      float x = v[e] + (bias ? bf16_bits_to_f32(bias[nn]) : 0.f) + (bias2 ? bf16_bits_to_f32(bias2[nn]) : 0.f);
      if (a.act >= 0 && nn >= a.act_from) x = act_eval(a.act, x);
      if (a.f32_out) {
        ((float *)a.out1)[(int64_t)m * a.ld1 + nn] = fmaf(a.out_scale, x, res ? ((const float *)a.residual)[(int64_t)m * a.ldr + nn] : 0.f);
        continue;
      }
      if (res) x += bf16_bits_to_f32(res[(int64_t)m * a.ldr + nn]);
      if (nn < a.n_split) ((uint16_t *)a.out1)[(int64_t)m * a.ld1 + nn] = f32_to_bf16_bits(x);
      else ((uint16_t *)a.out2)[(int64_t)m * a.ld2 + (nn - a.n_split)] = f32_to_bf16_bits(x);
    }
  }
}

template <int MT> static int launch_mfma_skinny(hipStream_t st, const LinearArgs &a) {
  constexpr int U = 8;
  constexpr int kcap = MT == 1 ? 2048 : MT == 2 ? 1024 : 512;  // LDS: MT*16 rows of (chunk + 8) bf16, about 64 KB
  const int blocks_x = ((a.N + 15) / 16 + 3) / 4;
  // Split K until there are about four blocks per CU, keeping at least 256 columns per split.
  int splits = 1;
  if (a.splitk_ws) {
    while (blocks_x * splits < 4 * kNumCU && a.K / (splits * 2) >= 256 &&
           (size_t)(splits * 2) * a.M * a.N * sizeof(float) <= a.splitk_ws_bytes)
      splits *= 2;
  }
  int kps = (a.K + splits - 1) / splits;
  kps = (kps + 127) / 128 * 128;
  splits = (a.K + kps - 1) / kps;
  const int chunk = kps < kcap ? kps : kcap;
  const size_t lds = (size_t)MT * 16 * (chunk + 8) * sizeof(uint16_t);
  static bool attr_set = false;
  if (!attr_set) {
    RAI_HIP_TRY(hipFuncSetAttribute((const void *)k_linear_bf16_mfma_skinny<MT, U>,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, 80 * 1024));
    attr_set = true;
  }
  float *partial = splits > 1 ? (float *)a.splitk_ws : nullptr;
  hipLaunchKernelGGL((k_linear_bf16_mfma_skinny<MT, U>), dim3(blocks_x, splits), dim3(256), lds, st, a, kps, chunk,
                     partial);
  RAI_TRY(launch_check("linear_bf16_mfma_skinny"));
  if (splits > 1) {
    RAI_TRY(launch_sum_of_parts(st, a, splits, partial));
  }
  return RAI_OK;
}

// ---- small M, second form: activations in registers, K split over the waves of a block ----
// Block = 8 waves; wave w owns K columns [k0 + w*32*KS, k0 + (w+1)*32*KS) of the block's
// K span and keeps the activation fragments of that slice in registers for the whole
// launch (MT*KS fragments).  The block walks over 16-row weight tiles: every wave reads
// its slice of the tile's rows straight into MFMA A fragments (one tile ahead of the
// multiply), so the block as a whole reads one contiguous 16-row panel after another and
// nothing is staged through LDS.  After G tiles the eight partial accumulators of each
// output are summed through LDS and the Linear epilogue is applied.  A K span of
// 256*KS covers K = 2048 (M <= 32) without splitting K over blocks, so the qkv / dense
// shapes of a batched decode step need neither a partial-sum buffer nor a second kernel.
// Fragment-major copy of W: element j of lane l of (row tile t, K step s) is W[16 t + l % 16][32 s + 8 (l / 16) + j].
__global__ void __launch_bounds__(256) k_linear_fragment_layout(bf16x8 *out, const uint16_t *W, int64_t ldw, int N, int ksteps,
                                                                int64_t total) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
    const int lane = (int)(i & 63);
    const int64_t ts = i >> 6;
    const int s = (int)(ts % ksteps);
    const int64_t t = ts / ksteps;
    const int64_t n = t * 16 + (lane & 15);
    bf16x8 v = {};
    if (n < N) v = *reinterpret_cast<const bf16x8 *>(W + n * ldw + s * 32 + (lane >> 4) * 8);
    out[i] = v;
  }
}
size_t linear_fragment_elems(int N, int K) { return (size_t)((N + 15) / 16) * 16 * (size_t)K; }
int launch_linear_fragment_layout(hipStream_t st, const void *W, int64_t ldw, int N, int K, void *Wfrag) {
  RAI_REQUIRE(K % 32 == 0 && ldw % 8 == 0 && (uintptr_t)W % 16 == 0 && (uintptr_t)Wfrag % 16 == 0, RAI_ERR_BAD_STRIDE,
              "fragment layout: K must be a multiple of 32 and the operands 16-byte aligned");
  const int64_t total = (int64_t)((N + 15) / 16) * (K / 32) * 64;
  const int64_t blocks = (total + 255) / 256;
  hipLaunchKernelGGL(k_linear_fragment_layout, dim3((unsigned)(blocks < 65535 ? blocks : 65535)), dim3(256), 0, st,
                     (bf16x8 *)Wfrag, (const uint16_t *)W, ldw, N, K / 32, total);
  return launch_check("linear_fragment_layout");
}

// F32O: the f32 output of LinearArgs::f32_out (fragment-order weights only; a branch in the bf16 form costs it 1 %)
template <int MT, int KS, int G, bool FRAG, bool F32O>
__global__ void __launch_bounds__(512) k_linear_bf16_mfma_stream(LinearArgs a, int tiles, float *partial, int *tickets) {
  __shared__ int s_ticket;
  constexpr int NW = 8;
  extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
  constexpr int PCH = 4 * G + 1;                       // row pitch of the parked accumulators, in f32x4
  f32x4 *red = reinterpret_cast<f32x4 *>(lds);        // [NW][MT * 16 rows][PCH]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lrow = lane & 15, lq = lane >> 4;
  const int split = blockIdx.y;
  const int k0 = (split * NW + wave) * KS * 32;

  int koff[KS];   // K steps beyond K read column 0 (their activation fragments are zero)
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) koff[ks] = k0 + ks * 32 < a.K ? k0 + ks * 32 : 0;
  const uint16_t *wbase = (const uint16_t *)a.W + lq * 8;
  const bf16x8 *fbase = reinterpret_cast<const bf16x8 *>(a.Wfrag) + lane;
  const int ksteps = a.K / 32;

  // A ring of tile buffers: while tile t is multiplied, the next RING-1 tiles are in flight.  Long streams (four
  // tiles per group, i.e. at least four tiles per block) take three buffers and loads that bypass the caches
  // (measured on a 1 GB matrix: 232 -> 193 us); short ones keep two buffers and cached loads, which a 10 MB matrix on
  // 160 blocks prefers by 1-2 us.  The ring turns by G positions per group, so the group body exists in RING rotations.
  constexpr int RING = G >= 4 ? 3 : 2;
  constexpr bool NT = G >= 4;
  bf16x8 w[RING][KS];
  auto load_tile = [&](bf16x8 (&wt)[KS], int tile) {
    tile = tile < tiles ? tile : tiles - 1;
    if constexpr (FRAG) {   // one instruction reads 1 KB of consecutive memory
      const bf16x8 *p = fbase + (int64_t)tile * ksteps * 64;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) wt[ks] = NT ? __builtin_nontemporal_load(p + (koff[ks] >> 5) * 64) : p[(koff[ks] >> 5) * 64];
    } else {
      int n = tile * 16 + lrow;
      n = n < a.N ? n : a.N - 1;
      const uint16_t *p = wbase + (int64_t)n * a.ldw;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        wt[ks] = NT ? __builtin_nontemporal_load(reinterpret_cast<const bf16x8 *>(p + koff[ks])) : *reinterpret_cast<const bf16x8 *>(p + koff[ks]);
    }
    // keep the whole tile's loads together and ahead of the multiplies that follow: left alone,
    // the scheduler sinks each load to just before its use and the prefetch distance collapses
    __builtin_amdgcn_sched_barrier(0);
  };
  const int stride = gridDim.x * G;
  // tile at position pos (0 .. G + RING - 2) counted from the start of the group that begins at tile g0
  auto tile_at = [&](int g0, int pos) { return g0 + (pos / G) * stride + pos % G; };
  // The block's first tiles are asked for behind the activation fragments (which come from the L2 and are needed
  // first: loads return in order) and, with a fused norm, before its statistics go round the block.
  int g0 = blockIdx.x * G;
  auto first_tiles = [&]() {
#pragma unroll
    for (int pos = 0; pos + 1 < RING; ++pos) load_tile(w[pos], tile_at(g0, pos));
  };
  // activation fragments of this wave's K slice (zero beyond M and K)
  bf16x8 xf[MT][KS];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int m = mt * 16 + lrow, k = k0 + ks * 32;
      bf16x8 z = {};
      if (m < a.M && k < a.K)
        z = *reinterpret_cast<const bf16x8 *>((const uint16_t *)a.A + (int64_t)m * a.lda + k + lq * 8);
      xf[mt][ks] = z;
    }
  // Optional RMSNorm of the activation rows (ln_kind 1: x * w / rms, 2: x * (1 + w) / rms), K not split
  // over blocks: the sum of squares of a row is gathered from the four lanes and eight waves that hold
  // its pieces, then every fragment is scaled and rounded to bf16 exactly as the stand-alone kernel does.  Every block norms all rows, so
  // its vector instructions count: squares on the matrix cores, the weight widened once for all row tiles and asked for ahead of
  // the weight tiles (24 x 2560 x 2048 10.8 to 9.8 us, 16 x 16384 x 2048 gated 17.2 to 16.0).
  if (a.ln_kind > 0) {
    float *rs = reinterpret_cast<float *>(lds);   // [8 waves][MT * 16 rows]; the accumulator area is not in use yet
    const uint16_t *lw = (const uint16_t *)a.ln_w;
    bf16x8 wv[KS];   // ahead of the weight tiles
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) wv[ks] = *reinterpret_cast<const bf16x8 *>(lw + koff[ks] + lq * 8);
    first_tiles();   // on their way while the row statistics go round the block
    // (the sum of squares is the diagonal of X X^T: lane (row, quarter) holds row 4 quarter + r of column `row`)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      f32x4 xx = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) xx = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf[mt][ks], xf[mt][ks], xx, 0, 0, 0);
      const float lo = lrow & 1 ? xx.y : xx.x, hi = lrow & 1 ? xx.w : xx.z;
      if (lq == lrow >> 2) rs[wave * (MT * 16) + mt * 16 + lrow] = lrow & 2 ? hi : lo;
    }
    // the widened values of the statistics pass are not kept for the scaling pass (256 registers: they would spill)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(xf[mt][ks]));
    __syncthreads();
    if (k0 + KS * 32 > a.K) {   // an infinite weight, read in their place, would make the zeros beyond K NaN
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        if (k0 + ks * 32 >= a.K) wv[ks] = bf16x8{};
    }
    float scale[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      float tot = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) tot += rs[w * (MT * 16) + mt * 16 + lrow];
      scale[mt] = 1.0f / sqrtf(tot / (float)a.K + a.ln_eps);
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)   // (beyond K: zeros stay zeros)
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float wf = a.ln_kind == 2 ? 1.0f + (float)wv[ks][j] : (float)wv[ks][j];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) xf[mt][ks][j] = (__bf16)((float)xf[mt][ks][j] * scale[mt] * wf);
      }
    __syncthreads();   // the statistics have been read before the area is reused
  } else {
    first_tiles();
  }
  const uint16_t *bias = (const uint16_t *)a.bias;
  const uint16_t *bias2 = (const uint16_t *)a.bias2;
  const uint16_t *res = (const uint16_t *)a.residual;
  // bias, activation / gated pair, residual and the bf16 store of four consecutive columns n .. n+3 of row m
  // (rv: the residual's four columns, asked for ahead of the sums that they are added to: 24 x 2048 x 2048 7.4 to 6.9 us)
  typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;
  auto residual4 = [&](int m, int n) __attribute__((always_inline)) {
    u32x2 rv = {0u, 0u};
    if (F32O || !res || m >= a.M || n >= a.N) return rv;
    const uint16_t *p = res + (int64_t)m * a.ldr + n;
    if (n + 4 <= a.N && ((uintptr_t)p & 7) == 0) return *reinterpret_cast<const u32x2 *>(p);
    const int lim = a.N - n < 4 ? a.N - n : 4;
    rv.x = (uint32_t)p[0] | (lim > 1 ? (uint32_t)p[1] << 16 : 0u);
    rv.y = (lim > 2 ? (uint32_t)p[2] : 0u) | (lim > 3 ? (uint32_t)p[3] << 16 : 0u);
    return rv;
  };
  auto finish = [&](int m, int n, f32x4 s4, u32x2 rv) __attribute__((always_inline)) {
    const float x[4] = {s4.x, s4.y, s4.z, s4.w};
    const int lim = a.N - n < 4 ? a.N - n : 4;
    if (a.glu) {   // columns (n, n+1) and (n+2, n+3) are (gate, up) pairs (N is a multiple of 8)
      uint16_t o[2];
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const float gt = x[2 * e] + (bias ? bf16_bits_to_f32(bias[n + 2 * e]) : 0.f);
        const float up = x[2 * e + 1] + (bias ? bf16_bits_to_f32(bias[n + 2 * e + 1]) : 0.f);
        o[e] = f32_to_bf16_bits(glu_bf16(a, gt, up));
      }
      uint16_t *dst = (uint16_t *)a.out1 + (int64_t)m * a.ld1 + (n >> 1);
      if (((uintptr_t)dst & 3) == 0) *reinterpret_cast<uint32_t *>(dst) = (uint32_t)o[0] | ((uint32_t)o[1] << 16);
      else { dst[0] = o[0]; dst[1] = o[1]; }
      return;
    }
    if constexpr (F32O) {
      float *dst = (float *)a.out1 + (int64_t)m * a.ld1 + n;
      const float *rsrc = res ? (const float *)a.residual + (int64_t)m * a.ldr + n : nullptr;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (e < lim) {
          float y = x[e] + ((bias ? bf16_bits_to_f32(bias[n + e]) : 0.f) + (bias2 ? bf16_bits_to_f32(bias2[n + e]) : 0.f));
          if (a.act >= 0 && n + e >= a.act_from) y = act_eval(a.act, y);
          dst[e] = fmaf(a.out_scale, y, rsrc ? rsrc[e] : 0.f);
        }
      }
      return;
    }
    uint16_t o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int nn = e < lim ? n + e : n;
      float y = x[e] + ((bias ? bf16_bits_to_f32(bias[nn]) : 0.f) + (bias2 ? bf16_bits_to_f32(bias2[nn]) : 0.f));
      if (a.act >= 0 && nn >= a.act_from) y = act_eval(a.act, y);
      if (res) y += bf16_bits_to_f32((uint16_t)((e < 2 ? rv.x : rv.y) >> (16 * (e & 1))));
      o[e] = f32_to_bf16_bits(y);
    }
    // all four columns in one output and the destination 8-byte aligned: one store
    const bool first = n + 3 < a.n_split, second = n >= a.n_split;
    uint16_t *dst = second ? (uint16_t *)a.out2 + (int64_t)m * a.ld2 + (n - a.n_split) : (uint16_t *)a.out1 + (int64_t)m * a.ld1 + n;
    if (lim == 4 && (first || second) && ((uintptr_t)dst & 7) == 0) {
      const u32x2 pk = {(uint32_t)o[0] | ((uint32_t)o[1] << 16), (uint32_t)o[2] | ((uint32_t)o[3] << 16)};
      *reinterpret_cast<u32x2 *>(dst) = pk;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (e < lim) {
          const int nn = n + e;
          if (nn < a.n_split) ((uint16_t *)a.out1)[(int64_t)m * a.ld1 + nn] = o[e];
          else ((uint16_t *)a.out2)[(int64_t)m * a.ld2 + (nn - a.n_split)] = o[e];
        }
      }
    }
  };
  auto group = [&](auto rot, const int g0) {
    constexpr int R = decltype(rot)::value;
    f32x4 acc[G][MT];
#pragma unroll
    for (int j = 0; j < G; ++j)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) acc[j][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int tc = tid % (G * 4);
    const u32x2 first_rv = partial ? u32x2{0u, 0u} : residual4(tid / (G * 4), (g0 + (tc >> 2)) * 16 + 4 * (tc & 3));
#pragma unroll
    for (int j = 0; j < G; ++j) {
      load_tile(w[(R + j + RING - 1) % RING], tile_at(g0, j + RING - 1));
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          acc[j][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[(R + j) % RING][ks], xf[mt][ks], acc[j][mt], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    // ---- sum the eight K slices and write G tiles of 16 columns x 16*MT rows.
    // Every wave parks its accumulators as [row m][G tiles x 4 column quads] (pitch PCH = 4 G + 1 chunks of 16 bytes,
    // odd, so that the 16 lanes of a quad, one row each, hit distinct banks); a thread then owns four consecutive
    // columns of one row: eight 16-byte reads, one store of four bf16, and 16 neighbouring threads cover 64 columns of
    // a row.  (One 4-byte read per wave and element and 2-byte stores a row apart took as long as streaming the
    // group's weights.)
    __syncthreads();   // the previous group's sums have been read
#pragma unroll
    for (int j = 0; j < G; ++j)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) red[(wave * MT * 16 + mt * 16 + lrow) * PCH + j * 4 + lq] = acc[j][mt];
    __syncthreads();
    for (int v = tid; v < MT * G * 64; v += 512) {
      const int m = v / (G * 4), c = v - m * (G * 4);
      const int tile = g0 + (c >> 2);
      const int n = tile * 16 + 4 * (c & 3);
      if (tile >= tiles || n >= a.N || m >= a.M) continue;
      f32x4 s4 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        const f32x4 t = red[(w * MT * 16 + m) * PCH + c];
        s4.x += t.x; s4.y += t.y; s4.z += t.z; s4.w += t.w;
      }
      if (partial) {
        float *p = partial + ((int64_t)split * a.M + m) * a.N + n;
        if (tickets) {   // read by another block of this launch: past the L2 (N is a multiple of 4, checked on the host)
          store_f32x4_device(p, s4);
        } else if (a.N - n >= 4 && a.N % 4 == 0) {
          *reinterpret_cast<f32x4 *>(p) = s4;
        } else {
          const float x[4] = {s4.x, s4.y, s4.z, s4.w};
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (n + e < a.N) p[e] = x[e];
        }
        continue;
      }
      finish(m, n, s4, v == tid ? first_rv : residual4(m, n));
    }
    if (partial && tickets) {
      // K split over blocks without a second launch: a block counts itself in once its partial sums have reached
      // memory, and the block that counts last -- whichever it is -- adds all of them in split order (the order of
      // the separate summing pass, so the result is the same bit for bit) and runs the epilogue.  Nobody waits.
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      int *ticket = tickets + g0 / G;
      if (tid == 0) s_ticket = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __syncthreads();
      if (s_ticket == (int)gridDim.y - 1) {
        if (tid == 0) __hip_atomic_store(ticket, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // for the next launch
        for (int v = tid; v < MT * G * 64; v += 512) {
          const int m = v / (G * 4), c = v - m * (G * 4);
          const int tile = g0 + (c >> 2);
          const int n = tile * 16 + 4 * (c & 3);
          if (tile >= tiles || n >= a.N || m >= a.M) continue;
          const u32x2 rv = residual4(m, n);
          f32x4 s4 = {0.f, 0.f, 0.f, 0.f};
          const float *p = partial + (int64_t)m * a.N + n;
          const int64_t each = (int64_t)a.M * a.N;
          // so many splits by one trip to memory, the residual with them (one after the other: 24 x 2048 x 16384 21.0 us, now 19.7)
          auto add = [&](auto count, int sp) {
            constexpr int B = decltype(count)::value;
            f32x4 t[B];
#pragma unroll
            for (int i = 0; i < B; ++i) t[i] = load_f32x4_device(p + (sp + i) * each);
#pragma unroll
            for (int i = 0; i < B; ++i) { s4.x += t[i].x; s4.y += t[i].y; s4.z += t[i].z; s4.w += t[i].w; }
          };
          int sp = 0;
          for (; sp + 8 <= (int)gridDim.y; sp += 8) add(std::integral_constant<int, 8>{}, sp);
          if (gridDim.y & 4) { add(std::integral_constant<int, 4>{}, sp); sp += 4; }
          if (gridDim.y & 2) { add(std::integral_constant<int, 2>{}, sp); sp += 2; }
          if (gridDim.y & 1) add(std::integral_constant<int, 1>{}, sp);
          finish(m, n, s4, rv);
        }
      }
    }
  };
  for (;;) {
    group(std::integral_constant<int, 0>{}, g0);
    if ((g0 += stride) >= tiles) break;
    group(std::integral_constant<int, G % RING>{}, g0);
    if ((g0 += stride) >= tiles) break;
    if constexpr (RING == 3) {
      group(std::integral_constant<int, (2 * G) % RING>{}, g0);
      if ((g0 += stride) >= tiles) break;
    }
  }
}

template <int MT, int KS, int G, bool FRAG = false, bool F32O = false>
static int launch_mfma_stream_cfg(hipStream_t st, const LinearArgs &a, int splits) {
  if constexpr (!FRAG) {
    if (a.f32_out) return launch_mfma_stream_cfg<MT, KS, G, true, true>(st, a, splits);
    if (a.Wfrag) return launch_mfma_stream_cfg<MT, KS, G, true>(st, a, splits);
  }
  const int tiles = (a.N + 15) / 16;
  const int groups = (tiles + G - 1) / G;
  int blocks_x = kNumCU / splits;
  if (blocks_x < 1) blocks_x = 1;
  if (blocks_x > groups) blocks_x = groups;
  const size_t lds = (size_t)8 * MT * 16 * (4 * G + 1) * sizeof(f32x4);
  static bool attr_set = false;
  if (lds > 64 * 1024 && !attr_set) {
    RAI_HIP_TRY(hipFuncSetAttribute((const void *)k_linear_bf16_mfma_stream<MT, KS, G, FRAG, F32O>,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    attr_set = true;
  }
  float *partial = splits > 1 ? (float *)a.splitk_ws : nullptr;
  // K split: the block that finishes a group last sums the partial products and runs the epilogue itself (no second
  // launch) when the tickets reach and the partial rows are 16-byte aligned; RAI_HIP_NO_FUSED_SPLITK=1 keeps the
  // separate summing pass (the tests compare the two: same bits).
  int *tickets = nullptr;
  if (splits > 1 && groups <= kSplitTickets && a.N % 4 == 0 && ((uintptr_t)partial & 15) == 0 && !getenv("RAI_HIP_NO_FUSED_SPLITK")) tickets = splitk_tickets(a);
  hipLaunchKernelGGL((k_linear_bf16_mfma_stream<MT, KS, G, FRAG, F32O>), dim3(blocks_x, splits), dim3(512), lds, st, a, tiles,
                     partial, tickets);
  RAI_TRY(launch_check("linear_bf16_mfma_stream"));
  if (splits > 1 && !tickets) {
    RAI_TRY(launch_sum_of_parts(st, a, splits, partial));
  }
  return RAI_OK;
}

// False when the shape needs a K split and no (or too small a) workspace was lent.
template <int MT, int KS> static bool mfma_stream_fits(const LinearArgs &a, int *splits) {
  const int span = 8 * KS * 32;
  *splits = (a.K + span - 1) / span;
  return *splits == 1 || (a.splitk_ws && (size_t)*splits * a.M * a.N * sizeof(float) <= a.splitk_ws_bytes);
}

template <int MT, int KS> static int launch_mfma_stream(hipStream_t st, const LinearArgs &a, int splits) {
  const int tiles = (a.N + 15) / 16;
  const int per_block = tiles * splits / kNumCU;   // tiles per block when every CU holds one block
  if (per_block >= 4) return launch_mfma_stream_cfg<MT, KS, 4>(st, a, splits);
  if (per_block >= 2) return launch_mfma_stream_cfg<MT, KS, 2>(st, a, splits);
  return launch_mfma_stream_cfg<MT, KS, 1>(st, a, splits);
}

// True when the small-M streaming kernel can apply the RMSNorm of the activation rows itself.
bool linear_mfma_fuses_norm(int M, int K, int ln_kind) {
  // read per call (three getenv are nothing next to a launch): tests force the fallback kernels within one process
  const bool off = getenv("RAI_HIP_NO_MFMA_STREAM") != nullptr || getenv("RAI_HIP_NO_MFMA_SKINNY") != nullptr ||
                   getenv("RAI_HIP_NO_FUSED_NORM") != nullptr;
  if (off || (ln_kind != 1 && ln_kind != 2) || M <= 8 || M > 64 || K % 32) return false;
  return K <= (M <= 32 ? 8 * 8 * 32 : 8 * 4 * 32);   // one block's K span: no split over blocks
}

static bool no_k64() {   // read per call: tests compare both forms in one process
  const char *e = getenv("RAI_HIP_NO_K64");
  return e && *e && *e != '0';
}

// 256 x 256 tiles cover a good half of the CUs.
static bool has_huge_tiles(const LinearArgs &a) { return 32 * (((a.M + 255) / 256) * ((a.N + 255) / 256)) >= 17 * kNumCU; }

// Which of the tiles with K stages of 64 serves a product, and over how many parts of K, by what the kernels' own times make
// of it.  The constants are fitted to 1276 products (random ones of 9 to 16384 rows, and the widths of the decoders' layers by twelve
// numbers of rows; every tile, one to twelve parts, weights from the caches and from HBM); over 654 others what is picked takes 0.7 %
// more than the best of them in the mean, over a twentieth more at 34 and over a tenth at 9 (600 of other days: 0.8 to 0.9 %).  The
// worst of all: 1221 x 328 x 3776 (18.8 us for 14.8), 1226 x 536 x 8128 (41.6 for 33.8), 512 x 1536 x 8960 (five parts 37.3, four 31.8),
// 6863 x 2368 x 2176 (102.5 for 87.3 by stream-K, see below).
// An XCD has 32 CUs and a run of tiles of its own, so rounds are counted there: over the whole chip 36 tiles in seven parts look like one
// round of 256 CUs, but five tiles on an XCD are 35 blocks and two rounds (333 x 8960 x 1536: 38.7 us, in five parts 26.9).  Blocks
// share a CU: `stage` is the time of 64 of K with one, two, three of them on it, `end` what a tile takes besides, to start and to write
// its outputs, `cut` the same where it writes partial sums.  A K split adds a launch and the partial sums' own time, and leaves every
// part four stages; of more than 80 MB of partial sums none was the best (beyond 160 MB they took 0.15 us a MB more than counted
// here); partial sums in rows off 16-byte boundaries cost 2.2 us per MB of outputs more.  A norm of the finished rows rides on the pass
// that sums the parts and is a launch of 5 us without one.
// 128 x 128 with eight waves (4 x 2, 32 x 64 each, two to a SIMD) took the place of four waves in two and four stages: 333 x 8960 x 1536
// 20.5 to 18.9 us, 2000 x 2048 x 2048 22.7 to 21.1.  128 x 256 and 192 x 256 (eight waves, three and two stages) serve where 256 x 256
// leaves a last round nearly empty: 1200 x 16384 x 2048 108 to 97 us, 3000 x 4096 x 4096 105 to 88, 777 x 22528 x 2048 114 to 91.
// Whole 256 x 256 tiles on one block per CU that keeps its pipeline full from tile to tile (gemm_persist.hip; persists()) cost kPersistEnd
// besides (over 320 products with 100 such tiles and more what is picked takes 0.4 % more than the best in the mean, 1.2 % by the
// figure of a block per tile).  K of an odd number of 32s, K parts and, without a residual, operands that no cache holds are blocks' work.
enum { kTile128 = 0, kTile128x64, kTile64, kTile128x256, kTile256x192, kTile192x256, kTile256, kTileStreamK };
struct TileCost { int bm, bn, share; float stage[3], end, cut; };
static const TileCost kTileCosts[] = {{128, 128, 1, {0.482f}, 3.24f, 1.46f}, {128, 64, 2, {0.36f, 0.568f}, 2.02f, 0.929f}, {64, 64, 3, {0.256f, 0.382f, 0.614f}, 0.81f, 0.428f},
                                      {128, 256, 1, {0.785f}, 6.77f, 2.27f}, {256, 192, 1, {1.21f}, 7.82f, 0.293f},        {192, 256, 1, {1.16f}, 7.58f, 0.472f},
                                      {256, 256, 1, {1.33f}, 10.1f, 0.493f}};
constexpr float kPersistEnd = 8.f, kLaunchUs = 2.43f, kCutUs = 4.04f, kPartUsPerMB = 0.555f, kMostPartMB = 80.f, kShareUs = 20.9f, kPersistShareUs = 25.f;

// Stream-K over 256 x 256 tiles, where its last round is exactly half full and so each of that round's tiles the work of two CUs, a half of
// K each: no CU is left idle, for an exchange of the halves (us, stream-K, the best whole tiles, all as blocks of a tile each: 4096 x 10240 x 2560
// 200, 212; 16384 x 1536 x 8960 374, 419; 1200 x 32768 x 2048 168, 174).  Shares that begin anywhere in K lose more in the L2s, where blocks no longer read
// the same columns together, than they win in idle CUs: of 168 such products with 40 stages and more the median took 1.14 times the best
// whole tiles' time (7770 x 2560 x 10240 476 us for 369, 7443 x 2560 x 2560 133 for 104), three less than 0.96 of it (14476 x 1536 x 8960
// 344 for 388).  On one block per CU a shared tile costs what a block's does, a whole one less, and the exchange is the dearer for it
// (2827 x 24480 x 2048 263, whole 246; 884 x 40776 x 2048 158, 146; 1341 x 16320 x 3584 151, on 192 x 256 tiles 138; but 16384 x 1536 x 4096 169, 178).
// 0: does not pay or does not apply.
static float streamk_us(const LinearArgs &a) {
  const int tiles = ((a.M + 255) / 256) * ((a.N + 255) / 256);
  StreamKPlan plan;
  if (!has_huge_tiles(a) || tiles % kNumCU != kNumCU / 2 || a.K / 64 % 2 || !streamk_applies(a, 64, &plan)) return 0.f;
  const bool persist = persists(a);
  const float multiply = kTileCosts[kTile256].stage[0] * ((float)a.K / 64), end = kTileCosts[kTile256].end;
  const float shared = (end + multiply) * ((float)tiles / kNumCU) + (persists(a, true) ? kPersistShareUs : kShareUs);
  return shared < ((persist ? kPersistEnd : end) + multiply) * ((tiles + kNumCU - 1) / kNumCU) ? kLaunchUs + shared : 0.f;
}
// With K stages of 32 (K no multiple of 64) whole 256 x 256 tiles are all there is beside it, and any shares pay where the CU time saved
// exceeds the exchange of two or three to a tile; a K tile of 32 takes some 1 us with all CUs busy (us, stream-K, whole tiles: 16384 x
// 1536 x 8928 464, 586; 8192 x 2560 x 5152 235, 306; 7770 x 2560 x 10272 475, 495; 4096 x 2560 x 10272 235, 286).
static bool streamk_pays_k32(const LinearArgs &a, StreamKPlan *plan) {
  if (!streamk_applies(a, 32, plan)) return false;
  const int left = ((a.M + 255) / 256) * ((a.N + 255) / 256) % kNumCU;
  return (float)(kNumCU - left) / kNumCU * (a.K / 32) >= 1.3f * (plan->k.max_parts <= 2 ? 18.f : 39.f);
}

struct TilePlan { int tile, splits; };
static TilePlan tile_plan_k64(const LinearArgs &a, int first = kTile128, int last = kTileStreamK) {
  const int stages = (a.K + 32) / 64;
  const float part_mb = (float)a.M * a.N * 4e-6f;
  TilePlan best = {first, 1};
  float least = 0.f;
  for (int t = first; t <= last && t < kTileStreamK; ++t) {
    const TileCost &c = kTileCosts[t];
    const int64_t tiles = (int64_t)((a.M + c.bm - 1) / c.bm) * ((a.N + c.bn - 1) / c.bn);
    for (int s = 1; s <= 12; ++s) {
      if (s > 1 && (a.force_splits == 1 || stages / s < 4 || s * part_mb > kMostPartMB || !a.splitk_ws || (size_t)s * a.M * a.N * sizeof(float) > a.splitk_ws_bytes)) break;
      const int64_t per_cu = ((tiles + kXcds - 1) / kXcds * s + kNumCU / kXcds - 1) / (kNumCU / kXcds);
      const int left = (int)(per_cu % c.share);
      const float stage = per_cu / c.share * c.stage[c.share - 1] + (left ? c.stage[left - 1] : 0.f);
      const float end = t == kTile256 && persists(a) ? kPersistEnd : c.end;
      const float cost = kLaunchUs + stage * ((stages + s - 1) / s) +
                         (s > 1 ? kCutUs + kPartUsPerMB * s * part_mb + (a.N % 4 ? 2.2f * part_mb : 0.f) + per_cu * c.cut : per_cu * end + (a.post_ln_out ? 5.f : 0.f));
      if ((t == first && s == 1) || cost < least) { least = cost; best = {t, s}; }
    }
  }
  if (last == kTileStreamK && a.K % 64 == 0)
    if (const float us = streamk_us(a); us > 0.f && us < least) best = {kTileStreamK, 1};
  return best;
}

// Split K when the tile count alone cannot fill the GPU and a workspace was provided (tiles of 32 of K, or a number of
// splits that the caller asked for).
static int tile_splits(const LinearArgs &a) {
  const int tiles = ((a.M + 127) / 128) * ((a.N + 127) / 128);
  int splits = 1;
  if (a.force_splits > 0) {
    const int kt = a.K / 32;
    int s = a.force_splits < kt ? a.force_splits : kt;
    while (s > 1 && (!a.splitk_ws || (size_t)s * a.M * a.N * sizeof(float) > a.splitk_ws_bytes)) --s;
    return s < 1 ? 1 : s;
  }
  if (a.splitk_ws && tiles < kNumCU) {
    // Cost model in units of one K tile of one block: blocks go round-robin over the CUs, a CU holds up to three,
    // n co-resident blocks share a CU at a combined rate of 0.5 / 0.85 / 1 (one block alone cannot hide its own
    // barriers and memory latency), each block pays ~8 units of prologue + epilogue, and every split adds a pass over
    // the f32 partial sums (~7 units at 512 x 2560).  Measured at 512 x 2560 x 12800: 3, 4, 6, 9, 12 splits give
    // 6.69, 6.64, 6.28, 6.44, 6.79 ms per 32-layer prefill, the order this model predicts.
    const int kt = a.K / 32;
    float best = 0.f;
    for (int s = 1; s <= 12; ++s) {
      if (s > 1 && (kt / s < 8 || (size_t)s * a.M * a.N * sizeof(float) > a.splitk_ws_bytes)) break;
      const float per_block = (float)((kt + s - 1) / s) + 8.f;
      int left = (tiles * s + kNumCU - 1) / kNumCU;   // blocks on the busiest CU
      float cost = (s > 1 ? 7.f * s : 0.f) * ((float)a.M * a.N / (512.f * 2560.f));
      while (left > 0) {
        const int n = left < 3 ? left : 3;
        cost += n * per_block / (n == 1 ? 0.5f : n == 2 ? 0.85f : 1.f);
        left -= n;
      }
      if (s == 1 || cost < best) { best = cost; splits = s; }
    }
  }
  return splits;
}

// RAI_HIP_GEMM_TILE, read per call, and the names of the tiles above in it; a tile that it names gets the split of its own.
static const char *forced_tile() { return getenv("RAI_HIP_GEMM_TILE"); }
static const struct { const char *name; int tile; } kTileNames[] = {{"128x128k64", kTile128},   {"128x128deep", kTile128},  {"128x64", kTile128x64},
                                                                   {"64x64", kTile64},         {"128x256", kTile128x256},  {"192x256", kTile192x256},
                                                                   {"256x192", kTile256x192}, {"256x256k64", kTile256}};
static int named_tile(const char *knob) {   // -1: none of them
  for (const auto &t : kTileNames)
    if (!strcmp(knob, t.name)) return t.tile;
  return -1;
}
// Stages of 64 also where K is an odd number of 32s: half of the first stage is zeros.  Over 280 such products they took 0.75 times the
// time of stages of 32 in the mean (us, stages of 32, of 64: 646 x 608 x 2456 20.9, 8.0; 1024 x 2080 x 2048 35.9, 17.7; 277 x 1376 x 600 11.8,
// 8.9; 16384 x 1504 x 8960 479, 434; 5105 x 672 x 9608 105, 101).  Stages of 32 stay where a short K meets one to two rounds of 128 x 128 tiles,
// which then share CUs (3574 x 160 x 1728 9.7, 11.5; 2405 x 608 x 1744 14.6, 15.9; with 10 stages and more even), and where stream-K saves
// much of a long one (6061 x 9504 x 13584 1501, 1551; but 4096 x 2592 x 10240, with `saved` at 40, 212, 208).
static bool stages_of_64(const LinearArgs &a) {
  if (a.K < 64 || no_k64()) return false;
  if (a.K % 64 == 0) return true;
  const int64_t tiles = (int64_t)((a.M + 127) / 128) * ((a.N + 127) / 128);
  if (a.K <= 12 * 64 && tiles > 224 && tiles <= 2 * kNumCU) return false;
  StreamKPlan plan;
  const int left = (int)((int64_t)((a.M + 255) / 256) * ((a.N + 255) / 256) % kNumCU);
  const float saved = (float)(kNumCU - left) / kNumCU * (a.K / 32);
  return !(saved >= 100.f && has_huge_tiles(a) && streamk_applies(a, 32, &plan));
}
static TilePlan tile_plan(const LinearArgs &a) {
  if (const char *knob = forced_tile()) {
    const int t = named_tile(knob);
    if (t >= 0) return a.K % 64 || a.force_splits > 0 ? TilePlan{t, tile_splits(a)} : tile_plan_k64(a, t, t);
    return {kTile128, tile_splits(a)};
  }
  if (!stages_of_64(a) || a.force_splits > 1) return {kTile128, tile_splits(a)};
  return tile_plan_k64(a);
}

template <int BM, int BN, int WGN>
static int launch_grouped_cfg(hipStream_t st, const LinearArgs &a, int64_t w_stride, const MoePlan &plan) {
  constexpr size_t lds = dma_lds_bytes<BM, BN, 2, WGN>();
  static bool attr_set = false;
  if (lds > 64 * 1024 && !attr_set) {
    RAI_HIP_TRY(hipFuncSetAttribute((const void *)k_gemm_bf16_mfma_grouped<BM, BN, WGN>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    attr_set = true;
  }
  const int total = plan.cap_tiles * ((a.N + BN - 1) / BN);
  hipLaunchKernelGGL((k_gemm_bf16_mfma_grouped<BM, BN, WGN>), dim3((total + kXcds - 1) / kXcds * kXcds), dim3(128 * WGN), lds, st, a, w_stride,
                     plan.tiles, plan.n_tiles);
  return launch_check("gemm_bf16_mfma_grouped");
}
// The eight-wave 256 x 256 tile once the experts have a few such tiles each, so that partly filled ones weigh little.
int linear_grouped_rows(int dtype, int64_t slots, int experts) {
  if (dtype != RAI_BF16) return kGroupedRowsF32;
  return slots >= (int64_t)experts * 4 * 256 ? 256 : kGroupedRowsBf16;
}
int launch_linear_bf16_grouped(hipStream_t st, const LinearArgs &a, int64_t w_stride, const MoePlan &plan, int bm) {
  RAI_REQUIRE(a.K % 64 == 0 && a.lda % 8 == 0 && a.ldw % 8 == 0 && w_stride % 8 == 0 && a.n_split == a.N && !a.residual && !a.f32_out &&
                  (!a.glu || a.N % 8 == 0),
              RAI_ERR_BAD_ARG, "linear grouped: %d x %d not served", a.N, a.K);
  return bm == 256 ? launch_grouped_cfg<256, 256, 4>(st, a, w_stride, plan) : launch_grouped_cfg<128, 128, 2>(st, a, w_stride, plan);
}

bool linear_fuses_post_norm(const LinearArgs &a) {
  // the tile kernels serve more than 64 rows; their split-K pass is the one that can normalise
  // (RAI_HIP_NO_POST_NORM: run the norm as its own launch, for comparison)
  const char *off = getenv("RAI_HIP_NO_POST_NORM");   // read per call: the test switches it within one process
  if (off && *off) return false;
  return a.M > 64 && post_norm_fits(a) && tile_plan(a).splits > 1;
}

static int launch_tile_k64(hipStream_t st, const LinearArgs &a, TilePlan tile) {
  switch (tile.tile) {
    case kTile64: return launch_cfg_dma<64, 64, 3, 0>(st, a, tile.splits);
    case kTile128x64: return launch_cfg_dma<128, 64, 3, 0>(st, a, tile.splits);
    case kTile128x256: return launch_cfg_dma<128, 256, 3, 0, 4, 2>(st, a, tile.splits);
    case kTile256x192: return launch_cfg_dma<256, 192, 2, 0, 2, 4>(st, a, tile.splits);
    case kTile192x256: return launch_cfg_dma<192, 256, 2, 0, 4, 2>(st, a, tile.splits);
    case kTile256:
      if (tile.splits == 1 && persists(a)) return launch_gemm_bf16_persist(st, a, StreamKArgs{});
      return launch_cfg_dma<256, 256, 2, 0, 4>(st, a, tile.splits);
    case kTileStreamK: {
      StreamKPlan plan;
      RAI_REQUIRE(streamk_applies(a, 64, &plan), RAI_ERR_UNSUPPORTED, "linear: stream-K does not apply to %dx%dx%d", a.M, a.N, a.K);
      return launch_streamk(st, a, plan, 64);
    }
    default: return launch_cfg_dma<128, 128, 4, 0, 2, 4>(st, a, tile.splits);
  }
}

int launch_linear_bf16_mfma(hipStream_t st, const LinearArgs &a) {
  RAI_REQUIRE(a.M > 0 && a.N > 0 && a.K > 0, RAI_ERR_BAD_SHAPE, "linear: empty problem %dx%dx%d", a.M, a.N, a.K);
  RAI_REQUIRE(a.A && a.W && a.out1, RAI_ERR_BAD_ARG, "linear: null operand");
  RAI_REQUIRE(a.n_split >= 0 && a.n_split <= a.N && (a.n_split == a.N || a.out2), RAI_ERR_BAD_ARG,
              "linear: bad output split");
  RAI_REQUIRE(a.ln_kind < 0 || linear_mfma_fuses_norm(a.M, a.K, a.ln_kind), RAI_ERR_UNSUPPORTED,
              "linear: fused norm needs M <= 8, or an RMS norm with M <= 64 and K within one block's span");
  if (a.glu) RAI_REQUIRE(a.N % 8 == 0 && !a.residual && a.n_split == a.N && a.act >= 0, RAI_ERR_BAD_ARG,
                         "linear mfma: bad gated-MLP arguments");
  RAI_REQUIRE(!a.f32_out || (a.n_split == a.N && !a.glu), RAI_ERR_BAD_ARG, "linear mfma: an f32 output is a single, ungated one");
  RAI_REQUIRE(a.K % 32 == 0, RAI_ERR_UNSUPPORTED, "linear mfma: K=%d must be a multiple of 32", a.K);
  RAI_REQUIRE(a.lda % 8 == 0 && a.ldw % 8 == 0 && (uintptr_t)a.A % 16 == 0 && (uintptr_t)a.W % 16 == 0,
              RAI_ERR_BAD_STRIDE, "linear mfma: operands must be 16-byte aligned with row strides multiple of 8");
  const bool no_skinny = getenv("RAI_HIP_NO_MFMA_SKINNY") != nullptr;
  const bool no_stream = getenv("RAI_HIP_NO_MFMA_STREAM") != nullptr;
  // A row-major W and 9 to 64 rows (up to 32 those that the streaming form of gemm_stream.hip leaves: a decoder's head on chosen rows, short K,
  // columns in no whole fours, and where it does not pay): the streaming kernel here reads 512-byte pieces of W's rows, at 2 to 3 TB/s; tiles with all of
  // their loads in flight do better once there are enough of them, and split K by themselves (us, stream, tiles, weights from
  // HBM: 16 x 512 x 8960 11.2, 6.2; 16 x 8192 x 8960 45, 35; 64 x 8192 x 8960 77, 40; 64 x 2048 x 2048 9.8, 9.2; 16 x 8192 x 2048 15.2,
  // 14.4; but 16 x 2048 x 2048 7.1, 8.0; 48 x 512 x 2048 4.8, 5.8; 16 x 8192 x 512 9.7, 13.4).  Where K needs no cut in the streaming
  // kernel (2048, beyond 32 rows 1024) it takes more of them (31 x 1728 x 6016 10.6, 12.9; 26 x 2048 x 2944 8.6, 10.0; 48 x 1024 x
  // 4736 7.7, 9.3; 17 to 32 rows x 1025 to 1535 x 4096 to 9000 in the mean 9.0, 10.6, up to 17000 12.8, 11.1; x 513 to 1024 8.6, 8.2;
  // 49 to 64 rows there 8.2, 8.3).
  const bool uncut = a.K <= (a.M <= 32 ? 2048 : 1024);
  const bool wide = a.N >= 4096 && (!uncut || a.N >= 9000 || (a.M <= 32 ? a.K <= 1024 : a.M > 48));
  const bool deep = a.N >= 2048 && !uncut && a.splitk_ws && a.K >= (a.M <= 16 ? 4096 : 1536);
  if (a.M > 8 && a.M <= 64 && !a.Wfrag && a.ln_kind < 0 && !a.f32_out && a.force_splits <= 0 && a.K % 64 == 0 && !no_k64() &&
      !no_skinny && !no_stream && (wide || deep))
    return launch_tile_k64(st, a, tile_plan_k64(a));
  if (a.M <= 64 && !no_skinny && !no_stream && (!a.f32_out || a.Wfrag)) {
    int splits = 1;
    if (a.M <= 16 && mfma_stream_fits<1, 8>(a, &splits)) return launch_mfma_stream<1, 8>(st, a, splits);
    if (a.M > 16 && a.M <= 32 && mfma_stream_fits<2, 8>(a, &splits)) return launch_mfma_stream<2, 8>(st, a, splits);
    if (a.M > 32 && a.M <= 48 && mfma_stream_fits<3, 4>(a, &splits)) return launch_mfma_stream<3, 4>(st, a, splits);
    if (a.M > 48 && mfma_stream_fits<4, 4>(a, &splits)) return launch_mfma_stream<4, 4>(st, a, splits);
  }
  if (a.M <= 64 && !no_skinny) {
    const int mt = (a.M + 15) / 16;
    if (mt == 1) return launch_mfma_skinny<1>(st, a);
    if (mt == 2) return launch_mfma_skinny<2>(st, a);
    if (mt == 3) return launch_mfma_skinny<3>(st, a);
    return launch_mfma_skinny<4>(st, a);
  }
  const TilePlan tile = tile_plan(a);
  const int splits = tile.splits;
  // Tile choice.  The LDS-DMA kernels stream K tiles straight into LDS, with stages of 64 where that pays (whole 128-byte lines per request;
  // RAI_HIP_NO_K64: never; stages_of_64): what tile_plan_k64 says.  Else 256 x 256 in its eight-wave form (one block per CU, 4 LDS stages of 32, two
  // waves per SIMD) or stream-K over it once its tiles cover a good half of the CUs, 128 x 128 with three stages below that.
  // RAI_HIP_GEMM_TILE = "64x64" | "128x64" | "128x128" | "128x128k64" | "128x128deep" (the same) | "128x256" | "192x256" | "256x128" |
  // "256x192" | "256x256" | "256x256k64" | "256x256x8w" | "256x256x8wk64" (256x256k64, K never cut) | "streamk" | "streamk64" | "classic"
  // overrides (tuning aid; a form that does not apply to the shape is an error).
  const char *knob = forced_tile();
  if (knob) {
    if (named_tile(knob) >= 0) {
      RAI_REQUIRE(a.K % 64 == 0, RAI_ERR_UNSUPPORTED, "linear: RAI_HIP_GEMM_TILE=%s needs K %% 64 == 0 (%dx%dx%d)", knob, a.M, a.N, a.K);
      return launch_tile_k64(st, a, tile);
    }
    if (!strcmp(knob, "128x128")) return launch_cfg_dma<128, 128, 3, 2>(st, a, splits);
    if (!strcmp(knob, "256x128")) return launch_cfg_dma<256, 128, 3, 2>(st, a, splits);
    if (!strcmp(knob, "256x256")) return launch_cfg_dma<256, 256, 4, 2>(st, a, splits);
    if (!strcmp(knob, "classic")) return launch_cfg<128, 128, 32>(st, a, splits);
    if (!strcmp(knob, "256x256x8w")) return launch_cfg_dma<256, 256, 4, 2, 4>(st, a, splits);
    if (!strcmp(knob, "256x256x8wk64")) {
      RAI_REQUIRE(splits == 1 && a.K % 64 == 0, RAI_ERR_UNSUPPORTED,
                  "linear: RAI_HIP_GEMM_TILE=256x256x8wk64 needs K %% 64 == 0 and no K split (%dx%dx%d)", a.M, a.N, a.K);
      return launch_tile_k64(st, a, {kTile256, 1});
    }
    if (!strcmp(knob, "streamk") || !strcmp(knob, "streamk64")) {
      const int bk = knob[7] ? 64 : 32;
      StreamKPlan plan;
      RAI_REQUIRE(splits == 1 && streamk_applies(a, bk, &plan), RAI_ERR_UNSUPPORTED,
                  "linear: RAI_HIP_GEMM_TILE=%s does not apply to %dx%dx%d", knob, a.M, a.N, a.K);
      return launch_streamk(st, a, plan, bk);
    }
  }
  if (stages_of_64(a)) return launch_tile_k64(st, a, tile);
  if (splits == 1 && has_huge_tiles(a)) {
    StreamKPlan plan;
    return streamk_pays_k32(a, &plan) ? launch_streamk(st, a, plan, 32) : launch_cfg_dma<256, 256, 4, 2, 4>(st, a, splits);
  }
  return launch_cfg_dma<128, 128, 3, 2>(st, a, splits);
}

}  // namespace rai

extern "C" int rai_hip_linear_plan(int dev, int32_t m, int32_t k, int32_t n, size_t scratch_bytes, char *tile, size_t tile_len, int32_t *k_parts) {
  using namespace rai;
  RAI_REQUIRE(tile && tile_len && k_parts && n > 0, RAI_ERR_BAD_ARG, "linear_plan: null argument");
  RAI_REQUIRE(m > 64 && k > 0 && k % 64 == 0, RAI_ERR_UNSUPPORTED, "linear_plan: %dx%dx%d is not served by one rule", m, n, k);
  LinearArgs a = linear_args_default();
  a.M = m; a.N = n; a.K = k; a.dev = dev;
  a.splitk_ws = scratch_bytes ? (void *)16 : nullptr;   // (looked at, not into)
  a.splitk_ws_bytes = scratch_bytes;
  const TilePlan plan = tile_plan_k64(a);
  const char *name = "streamk64";
  for (const auto &t : kTileNames)
    if (t.tile == plan.tile) { name = t.name; break; }
  snprintf(tile, tile_len, "%s", name);
  *k_parts = plan.splits;
  return RAI_OK;
}
