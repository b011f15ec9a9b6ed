// f32 Linears on the f32 matrix instructions (every product and sum in f32).
//   k_linear_f32_tile    tiles of 64 x 64 or 32 x 128 outputs, operands through LDS, K optionally cut over blocks
//   k_linear_f32_rows    up to four rows (decoding)
//   k_linear_f32_sum     adds the partial products of such a cut and applies the epilogue
//   k_linear_f32_grouped the tile form over the rows of one expert after another
//
// Reference semantics: rai-nn/src/linear.rs:59-69 (x W^T + b).
#include "gemm.h"
#include "latent.h"

namespace rai {

typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;

// ------------------------------------------------------------------ epilogue
__device__ __forceinline__ float f32_bias(const LinearArgs &a, int n) {
  return (a.bias ? ((const float *)a.bias)[n] : 0.f) + (a.bias2 ? ((const float *)a.bias2)[n] : 0.f);
}
__device__ __forceinline__ float f32_gated(const LinearArgs &a, float gate, float up) {
  return a.act == kActClampedGlu ? glu_clamped(gate, up, a.act_limit, a.act_alpha) : act_eval(a.act, gate) * up;
}
// Activation, scale, residual and the store of one output whose bias is already added.
__device__ __forceinline__ void f32_finish(const LinearArgs &a, int m, int n, float v) {
  if (a.act >= 0 && n >= a.act_from) v = act_eval(a.act, v);
  if (a.f32_out) v *= a.out_scale;
  if (a.residual) v += ((const float *)a.residual)[(int64_t)m * a.ldr + n];
  if (n < a.n_split) ((float *)a.out1)[(int64_t)m * a.ld1 + n] = v;
  else ((float *)a.out2)[(int64_t)m * a.ld2 + (n - a.n_split)] = v;
}
// Columns n .. n + 3 of a row, as far as they are below N.
__device__ __forceinline__ bool aligned16(const void *p) { return ((uintptr_t)p & 15) == 0; }
__device__ __forceinline__ f32x4 f32_load_cols(const float *row, int n, int N) {
  if (n + 3 < N && aligned16(row + n)) return *reinterpret_cast<const f32x4 *>(row + n);
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (n + j < N) v[j] = row[n + j];
  return v;
}
__device__ __forceinline__ void f32_store_cols(float *row, int n, int N, f32x4 v) {
  if (n + 3 < N && aligned16(row + n)) { *reinterpret_cast<f32x4 *>(row + n) = v; return; }
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (n + j < N) row[n + j] = v[j];
}
// The whole epilogue of four neighbouring columns, whichever of them exist.
__device__ __forceinline__ void f32_finish4(const LinearArgs &a, int m, int n, f32x4 v) {
  if (a.bias) v += f32_load_cols((const float *)a.bias, n, a.N);
  if (a.bias2) v += f32_load_cols((const float *)a.bias2, n, a.N);
  if (a.glu) {   // interleaved gate and up columns
    float *o = (float *)a.out1 + (int64_t)m * a.ld1 + (n >> 1);
#pragma unroll
    for (int j = 0; j < 4; j += 2)
      if (n + j + 1 < a.N) o[j >> 1] = f32_gated(a, v[j], v[j + 1]);
    return;
  }
  if (n + 3 >= a.N || (n < a.n_split && n + 3 >= a.n_split)) {   // past the end, or across the two outputs
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (n + j < a.N) f32_finish(a, m, n + j, v[j]);
    return;
  }
  if (a.act >= 0) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (n + j >= a.act_from) v[j] = act_eval(a.act, v[j]);
  }
  if (a.f32_out) v *= a.out_scale;
  if (a.residual) v += f32_load_cols((const float *)a.residual + (int64_t)m * a.ldr, n, a.N);
  if (n < a.n_split) f32_store_cols((float *)a.out1 + (int64_t)m * a.ld1, n, a.N, v);
  else f32_store_cols((float *)a.out2 + (int64_t)m * a.ld2 - a.n_split, n, a.N, v);
}

// ------------------------------------------------------------------ tile kernel
// Bound by the matrix units: v_mfma_f32_32x32x2_f32 does 64 flops a clock and SIMD (157 TFLOP/s for the GPU), an eighth
// of what LDS reads of this shape could feed, so the loop is kept simple.  Four waves with one accumulator of 32 x 32 each,
// as 2 x 2 (64 x 64) or side by side (32 x 128, up to 32 rows: half the padding); four or five blocks on a CU cover each
// other's waits.  K tiles of 32 in two LDS stages, loaded into registers one tile ahead without a branch (a branch around a
// load, for the ends of the matrix, made the compiler wait for it: 107 against 123 TFLOP/s) and stored to the other stage
// in the middle of the multiplies, one barrier per K tile.  A lane reads four consecutive k with one 16-byte LDS load and
// feeds them to four MFMAs (k 4h .. 4h + 3 for lane half h, the same order for both operands).  Rows are 36 floats apart
// in LDS: sixteen rows then start in sixteen different 16-byte columns.
//   Measured: 4096 x 2560 x 10240 1745 us = 123 TFLOP/s, MFMAs busy 85 % of the cycles (fused multiply-adds on the vector
// units: 2700 us); 1024 rows 427 us (690); 128 x 12800 x 2560 with K cut 82 us (804); 24 x 2560 x 10240 30 us (162, and 43
// with tiles of 64 x 64).  Tiles of 128 x 128 reach 131 TFLOP/s at 4096 rows and lose more than that to the partial round
// at 1024 (623 us).
//   Operands come in pieces of 16 bytes.  kWhole: rows 16-byte aligned and K a multiple of four.  kRagged: rows that start
// anywhere and any K from four on: the piece that crosses the end of K is read four elements before the end and shifted, so
// no load stands behind a branch (1024 x 8190 x 10240 in rows of 8192 1310 us, in rows of 8190 1340; element by element with
// the ends behind branches 2318 and 2077).  kTiny: element by element.
enum { kTiny, kRagged, kWhole };
template <int BM, int BN>
struct F32Tile {
  static constexpr int BK = 32, PITCH = 36;
  static constexpr int STAGE = (BM + BN) * PITCH;   // floats
  static constexpr int PA = BM / 32, PB = BN / 32;  // 16-byte loads a thread makes per K tile
};

// Four consecutive k of a row, from k on; kTiny: those below k_end and zeros.
template <int LOADS>
__device__ __forceinline__ f32x4 f32_load_k(const float *row, int k, int k_end) {
  f32x4 v;
  if constexpr (LOADS == kTiny) {
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = k + j < k_end ? row[k + j] : 0.f;
  } else if constexpr (LOADS == kRagged) {
    __builtin_memcpy(&v, row + k, 16);
  } else {
    v = *reinterpret_cast<const f32x4 *>(row + k);
  }
  return v;
}
// A piece that was read `past` elements ahead of its place because K ends: what lies past the end is zero.
__device__ __forceinline__ f32x4 f32_end_of_k(f32x4 v, int past) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (past > i) v = f32x4{v[1], v[2], v[3], 0.f};
  return v;
}

// Products over [k_begin, k_end) of the tile at (m0, n0); `finish(m, n, v)` receives them, columns n .. n + 3 (n < N) of
// row m at a time.
template <int BM, int BN, int LOADS, class Finish>
__device__ __forceinline__ void linear_f32_tile(const LinearArgs &a, int m0, int n0, int k_begin, int k_end, float *lds, Finish finish) {
  using T = F32Tile<BM, BN>;
  constexpr int BK = T::BK, PITCH = T::PITCH;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = (wave / (BN / 32)) * 32, wn = (wave % (BN / 32)) * 32;
  const int r = lane & 31, h = lane >> 5;
  const int lrow = tid >> 3, lk = (tid & 7) * 4;   // staging: eight threads a row of 32
  const float *A = (const float *)a.A, *W = (const float *)a.W;
  // rows past the end are read from the last one: they only reach outputs that are not stored
  const float *arow[T::PA], *wrow[T::PB];
#pragma unroll
  for (int p = 0; p < T::PA; ++p) arow[p] = A + (int64_t)min(m0 + lrow + 32 * p, a.M - 1) * a.lda;
#pragma unroll
  for (int p = 0; p < T::PB; ++p) wrow[p] = W + (int64_t)min(n0 + lrow + 32 * p, a.N - 1) * a.ldw;
  f32x4 ra[T::PA], rb[T::PB];
  auto fetch = [&](int k0) {
    const int k = LOADS == kTiny ? k0 + lk : min(k0 + lk, k_end - 4);
#pragma unroll
    for (int p = 0; p < T::PA; ++p) ra[p] = f32_load_k<LOADS>(arow[p], k, k_end);
#pragma unroll
    for (int p = 0; p < T::PB; ++p) rb[p] = f32_load_k<LOADS>(wrow[p], k, k_end);
  };
  auto park = [&](float *st, int k0) {
    // both operands are zero past the end of K
    if (LOADS == kWhole && k0 + BK > k_end && k0 + lk >= k_end) {
#pragma unroll
      for (int p = 0; p < T::PA; ++p) ra[p] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int p = 0; p < T::PB; ++p) rb[p] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    if (LOADS == kRagged && k0 + BK > k_end) {
      const int past = k0 + lk - (k_end - 4);
#pragma unroll
      for (int p = 0; p < T::PA; ++p) ra[p] = f32_end_of_k(ra[p], past);
#pragma unroll
      for (int p = 0; p < T::PB; ++p) rb[p] = f32_end_of_k(rb[p], past);
    }
#pragma unroll
    for (int p = 0; p < T::PA; ++p) *reinterpret_cast<f32x4 *>(st + (lrow + 32 * p) * PITCH + lk) = ra[p];
#pragma unroll
    for (int p = 0; p < T::PB; ++p) *reinterpret_cast<f32x4 *>(st + (BM + lrow + 32 * p) * PITCH + lk) = rb[p];
  };
  f32x16 acc = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};

  const int tiles = (k_end - k_begin + BK - 1) / BK;
  fetch(k_begin);
  park(lds, k_begin);
  if (tiles > 1) fetch(k_begin + BK);
  __syncthreads();
  for (int t = 0; t < tiles; ++t) {
    const float *st = lds + (t & 1) * T::STAGE;
    const float *sa = st + (wm + r) * PITCH + 4 * h, *sb = st + (BM + wn + r) * PITCH + 4 * h;
    f32x4 fa[2], fb[2];   // the next eight k are read while the current ones are multiplied
    auto read = [&](int kk) {
      fa[kk & 1] = *reinterpret_cast<const f32x4 *>(sa + kk * 8);
      fb[kk & 1] = *reinterpret_cast<const f32x4 *>(sb + kk * 8);
    };
    read(0);
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      if (kk < 3) read(kk + 1);
      if (kk == 2 && t + 1 < tiles) {   // to the stage that was read in the previous iteration, which every wave has left
        park(lds + ((t + 1) & 1) * T::STAGE, k_begin + (t + 1) * BK);
        if (t + 2 < tiles) fetch(k_begin + (t + 2) * BK);
      }
#pragma unroll
      for (int s = 0; s < 4; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[kk & 1][s], fb[kk & 1][s], acc, 0, 0, 0);
    }
    __syncthreads();
  }

  // Lane (r, h) holds column r of each accumulator and rows 8 (i / 4) + 4 h + i % 4: through LDS (free after the last
  // barrier), so that a thread finishes four neighbouring columns of a row.
  constexpr int OP = BN + 4;
#pragma unroll
  for (int e = 0; e < 16; ++e) lds[(wm + 8 * (e >> 2) + 4 * h + (e & 3)) * OP + wn + r] = acc[e];
  __syncthreads();
#pragma unroll 1
  for (int e = tid; e < BM * (BN / 4); e += 256) {
    const int row = e / (BN / 4), col = (e % (BN / 4)) * 4;
    if (m0 + row < a.M && n0 + col < a.N) finish(m0 + row, n0 + col, *reinterpret_cast<const f32x4 *>(lds + row * OP + col));
  }
}

// Block -> tile: every XCD (blocks are dealt out to the eight of them in turn) walks a run of tiles of its own, in bands
// of eight tile rows, so that the tiles in flight on it share operand rows in its L2.
__device__ __forceinline__ void f32_tile_of_block(int block, int tiles_m, int tiles_n, int &tm, int &tn) {
  const int tiles = tiles_m * tiles_n, xcd = block & 7, q = tiles >> 3, rem = tiles & 7;
  const int t = xcd * q + (xcd < rem ? xcd : rem) + (block >> 3);
  const int band = t / (8 * tiles_n), rows = tiles_m - 8 * band < 8 ? tiles_m - 8 * band : 8;
  const int in = t - band * 8 * tiles_n;
  tm = band * 8 + in % rows;
  tn = in / rows;
}

template <int BM, int BN, int LOADS, bool PARTIAL>
__global__ void __launch_bounds__(256, 2) k_linear_f32_tile(LinearArgs a, int k_step) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  int tm, tn;
  f32_tile_of_block(blockIdx.x, (a.M + BM - 1) / BM, (a.N + BN - 1) / BN, tm, tn);
  if constexpr (PARTIAL) {
    const int k0 = blockIdx.y * k_step, k1 = k0 + k_step < a.K ? k0 + k_step : a.K;
    float *part = (float *)a.splitk_ws + (int64_t)blockIdx.y * a.M * a.N;
    linear_f32_tile<BM, BN, LOADS>(a, tm * BM, tn * BN, k0, k1, lds, [&](int m, int n, f32x4 v) { f32_store_cols(part + (int64_t)m * a.N, n, a.N, v); });
  } else {
    linear_f32_tile<BM, BN, LOADS>(a, tm * BM, tn * BN, 0, a.K, lds, [&](int m, int n, f32x4 v) { f32_finish4(a, m, n, v); });
  }
}

// Sums the partial products of the K splits in split order and applies the epilogue; a thread owns four columns.
__global__ void __launch_bounds__(256) k_linear_f32_sum(LinearArgs a, int splits) {
  const int quads = (a.N + 3) / 4;
  const int64_t total = (int64_t)a.M * quads, plane = (int64_t)a.M * a.N;
  for (int64_t e = blockIdx.x * 256LL + threadIdx.x; e < total; e += gridDim.x * 256LL) {
    const int m = (int)(e / quads), n = 4 * (int)(e - (int64_t)m * quads);
    const float *p = (const float *)a.splitk_ws + (int64_t)m * a.N;
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int s = 0; s < splits; ++s) v += f32_load_cols(p + s * plane, n, a.N);
    f32_finish4(a, m, n, v);
  }
}

// The 64 x 64 tile over the rows of one expert (see MoePlan): blockIdx.x = column tile, blockIdx.y = row tile.
template <int LOADS>
__global__ void __launch_bounds__(256) k_linear_f32_grouped(LinearArgs a, int64_t w_stride, const int4 *tiles, const int *n_tiles) {
  __shared__ __attribute__((aligned(16))) float lds[2 * F32Tile<64, 64>::STAGE];
  if ((int)blockIdx.y >= *n_tiles) return;
  const int4 t = tiles[blockIdx.y];
  a.A = (const float *)a.A + (int64_t)t.y * a.lda;
  a.W = (const float *)a.W + (int64_t)t.x * w_stride;
  a.out1 = (float *)a.out1 + (int64_t)t.y * a.ld1;
  a.M = t.z;
  linear_f32_tile<64, 64, LOADS>(a, 0, blockIdx.x * 64, 0, a.K, lds, [&](int m, int n, f32x4 v) { f32_finish4(a, m, n, v); });
}

// ------------------------------------------------------------------ few rows
// M <= 4 (decoding): bound by the weight matrix's way from HBM.  A block owns two rows of W, a quarter of K to each of its
// four waves; a wave reads 1 KB of a row with one instruction and multiplies it with the same piece of the M rows of A,
// which come from L2 and stay in registers.  Few bytes per wave and many small waves in flight do best: 27 registers at
// M = 1, eight waves a SIMD.  Measured with weights that no cache holds (us; 1 x 2560 x 32768, 1 x 12800 x 2560, 1 x 2560 x
// 2560): 48.7, 23.2, 7.0 (6.9, 5.6 and 3.7 TB/s), against 57, 23, 8.2 with four pieces of a row requested at a time, 50, 34,
// 9.1 without the cut of K, and 220, 769, 160 with tiles of 64 x 64 over unsplit K.  Eight rows take 36 us at 2560 x 10240,
// where the tile form takes 29; four take 26.
template <int M>
__global__ void __launch_bounds__(256) k_linear_f32_rows(LinearArgs a) {
  constexpr int R = 2, U = 2, KW = 4;
  __shared__ float red[KW][R * M];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = blockIdx.x * R;
  const int chunks = (a.K + 255) / 256, each = (chunks + KW - 1) / KW;
  const int k_end = min((wave + 1) * each * 256, a.K);
  const float *A = (const float *)a.A, *w[R];
#pragma unroll
  for (int i = 0; i < R; ++i) w[i] = (const float *)a.W + (int64_t)min(n0 + i, a.N - 1) * a.ldw;
  float acc[R][M];
#pragma unroll
  for (int i = 0; i < R; ++i)
#pragma unroll
    for (int m = 0; m < M; ++m) acc[i][m] = 0.f;
  for (int k0 = wave * each * 256 + 4 * lane; k0 < k_end; k0 += 256 * U) {
    f32x4 wv[U][R], xv[U][M];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + 256 * u < k_end ? k0 + 256 * u : k0;   // past the end: read again, not added
#pragma unroll
      for (int m = 0; m < M; ++m) xv[u][m] = *reinterpret_cast<const f32x4 *>(A + (int64_t)min(m, a.M - 1) * a.lda + k);
#pragma unroll
      for (int i = 0; i < R; ++i) wv[u][i] = __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(w[i] + k));
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (k0 + 256 * u < k_end) {
#pragma unroll
        for (int i = 0; i < R; ++i)
#pragma unroll
          for (int m = 0; m < M; ++m)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[i][m] = fmaf(wv[u][i][e], xv[u][m][e], acc[i][m]);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < R; ++i)
#pragma unroll
    for (int m = 0; m < M; ++m) acc[i][m] = wave_sum(acc[i][m]);
  if (lane == 0) {
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
      for (int m = 0; m < M; ++m) red[wave][i * M + m] = acc[i][m];
  }
  __syncthreads();
  if (threadIdx.x >= a.M) return;   // thread m finishes row m
  const int m = threadIdx.x;
  float v[R];
#pragma unroll
  for (int i = 0; i < R; ++i) {
    v[i] = red[0][i * M + m];
#pragma unroll
    for (int j = 1; j < KW; ++j) v[i] += red[j][i * M + m];
    if (n0 + i < a.N) v[i] += f32_bias(a, n0 + i);
  }
  if (a.glu) {
    if (n0 + 1 < a.N) ((float *)a.out1)[(int64_t)m * a.ld1 + (n0 >> 1)] = f32_gated(a, v[0], v[1]);
    return;
  }
#pragma unroll
  for (int i = 0; i < R; ++i)
    if (n0 + i < a.N) f32_finish(a, m, n0 + i, v[i]);
}

// ------------------------------------------------------------------ launchers
static bool rows_aligned(const LinearArgs &a) {
  return a.K % 4 == 0 && a.lda % 4 == 0 && a.ldw % 4 == 0 && (uintptr_t)a.A % 16 == 0 && (uintptr_t)a.W % 16 == 0;
}

template <int BM, int BN, int LOADS, bool PARTIAL>
static int launch_tile(hipStream_t st, const LinearArgs &a, int splits, int k_step) {
  constexpr size_t lds = 2 * F32Tile<BM, BN>::STAGE * sizeof(float);
  static bool attr_set = false;
  if (lds > 64 * 1024 && !attr_set) {
    RAI_HIP_TRY(hipFuncSetAttribute((const void *)k_linear_f32_tile<BM, BN, LOADS, PARTIAL>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    attr_set = true;
  }
  const int64_t tiles = (int64_t)((a.M + BM - 1) / BM) * ((a.N + BN - 1) / BN);
  RAI_REQUIRE(tiles < (1LL << 31), RAI_ERR_UNSUPPORTED, "linear f32: %d x %d outputs exceed the grid", a.M, a.N);
  hipLaunchKernelGGL((k_linear_f32_tile<BM, BN, LOADS, PARTIAL>), dim3((unsigned)tiles, splits), dim3(256), lds, st, a, k_step);
  return launch_check("linear_f32_tile");
}

constexpr int kFewRows = 4;
template <int M> static int launch_rows(hipStream_t st, const LinearArgs &a) {
  hipLaunchKernelGGL((k_linear_f32_rows<M>), dim3((a.N + 1) / 2), dim3(256), 0, st, a);
  return launch_check("linear_f32_rows");
}

// How many pieces of K to compute side by side with `room` bytes for their products, by the time the tiles and the summing
// pass would take: a tile of full K is 0.017 us of a busy CU's time per k, a CU needs three or four blocks to be busy, the
// sum is a launch and a trip of the partial products to memory and back.
static bool wide_tiles(const LinearArgs &a) { return a.M <= 32 && rows_aligned(a); }   // 32 x 128 instead of 64 x 64
static int f32_splits(const LinearArgs &a, size_t room) {
  static const double busy[5] = {0, 0.45, 0.75, 0.9, 1.0};   // share of its rate a CU reaches with this many blocks
  const int64_t tiles = wide_tiles(a) ? (a.N + 127) / 128 : (int64_t)((a.M + 63) / 64) * ((a.N + 63) / 64);
  const size_t plane = (size_t)a.M * a.N * sizeof(float);
  int best = 1;
  double least = 0;
  for (int s = 1; s <= 16 && (s == 1 || (s * 256 <= a.K && s * plane <= room)); ++s) {
    const int64_t rounds = (tiles * s + kNumCU - 1) / kNumCU;
    const double us = rounds * 0.017 * a.K / s / busy[rounds < 4 ? rounds : 4] + (s > 1 ? 3.0 + 2.0 * s * plane / 4e6 : 0.0);
    if (s == 1 || us < least) { least = us; best = s; }
  }
  return best;
}
// Where the few-row kernel serves.  A block's end (the sums across its lanes) is paid per two rows of W however short they
// are: 0.36, 0.51 and 1.04 us per 1000 rows of W for one, two and four rows.  Short rows against many are done sooner by
// the tiles, a round of which takes 3.4 us and 0.02 per k (us, this kernel, tiles, K x N; four rows 64 x 10240 13.3, 4.6; 256 x
// 32768 36.5, 10.5; 384 x 10240 13.4, 11.0; two 128 x 16384 11.0, 6.3; one 96 x 32768 13.2, 7.7; multiply-adds on the vector units
// 9.2, 26.6, 28.7, 11.8, 9.5).
static bool few_rows(const LinearArgs &a) {
  if (a.M > kFewRows || !rows_aligned(a)) return false;
  const float per_row = a.M == 1 ? 0.36e-3f : a.M == 2 ? 0.51e-3f : 1.04e-3f;
  return 2.f + per_row * a.N <= 3.4f + 0.02f * a.K * (float)((a.N + 16383) / 16384);
}

size_t linear_f32_workspace_bytes(const LinearArgs &a, size_t room) {
  const int s = few_rows(a) ? 1 : f32_splits(a, room);
  return s > 1 ? (size_t)s * a.M * a.N * sizeof(float) : 0;
}

int launch_linear_f32(hipStream_t st, const LinearArgs &a) {
  RAI_REQUIRE(a.M > 0 && a.N > 0 && a.K > 0, RAI_ERR_BAD_SHAPE, "linear: empty problem");
  RAI_REQUIRE(a.ln_kind < 0, RAI_ERR_UNSUPPORTED, "linear f32: no fused norm");
  if (few_rows(a)) return a.M == 1 ? launch_rows<1>(st, a) : a.M == 2 ? launch_rows<2>(st, a) : launch_rows<4>(st, a);
  const bool vec = rows_aligned(a), wide = wide_tiles(a);
  int splits = f32_splits(a, a.splitk_ws ? a.splitk_ws_bytes : 0);
  if (splits > 1) {
    int k_step = (a.K + splits - 1) / splits;
    k_step = (k_step + 31) / 32 * 32;
    splits = (a.K + k_step - 1) / k_step;
    if (wide) RAI_TRY((launch_tile<32, 128, kWhole, true>(st, a, splits, k_step)));
    else RAI_TRY((vec ? launch_tile<64, 64, kWhole, true>(st, a, splits, k_step) : launch_tile<64, 64, kRagged, true>(st, a, splits, k_step)));
    const int64_t blocks = ((int64_t)a.M * ((a.N + 3) / 4) + 255) / 256;
    hipLaunchKernelGGL(k_linear_f32_sum, dim3((unsigned)(blocks < 4096 ? blocks : 4096)), dim3(256), 0, st, a, splits);
    return launch_check("linear_f32_sum");
  }
  if (wide) return launch_tile<32, 128, kWhole, false>(st, a, 1, 0);
  if (vec) return launch_tile<64, 64, kWhole, false>(st, a, 1, 0);
  return a.K >= 4 ? launch_tile<64, 64, kRagged, false>(st, a, 1, 0) : launch_tile<64, 64, kTiny, false>(st, a, 1, 0);
}

int launch_linear_f32_grouped(hipStream_t st, const LinearArgs &a, int64_t w_stride, const MoePlan &plan) {
  const dim3 grid((a.N + 63) / 64, plan.cap_tiles);
  if (rows_aligned(a) && w_stride % 4 == 0)
    hipLaunchKernelGGL(k_linear_f32_grouped<kWhole>, grid, dim3(256), 0, st, a, w_stride, plan.tiles, plan.n_tiles);
  else if (a.K >= 4)
    hipLaunchKernelGGL(k_linear_f32_grouped<kRagged>, grid, dim3(256), 0, st, a, w_stride, plan.tiles, plan.n_tiles);
  else
    hipLaunchKernelGGL(k_linear_f32_grouped<kTiny>, grid, dim3(256), 0, st, a, w_stride, plan.tiles, plan.n_tiles);
  return launch_check("linear_f32_grouped");
}

}  // namespace rai
