// Batched products of strided operands on the matrix instructions: f32, bf16 and f16, each operand contiguous along K or
// along its other axis, any batch strides.  (Products whose right operand is one shared, K-contiguous matrix are Linears;
// f64 and operands without a unit stride stay with k_matmul_generic.)
//
// Reference semantics: rai-core/src/backend/candle.rs:327-443 (MatMul, stride rule).
#include "gemm.h"

namespace rai {

typedef __attribute__((ext_vector_type(16))) float mm_f32x16;
typedef __attribute__((ext_vector_type(4))) float mm_f32x4;
typedef __attribute__((ext_vector_type(8))) __bf16 mm_bf16x8;
typedef __attribute__((ext_vector_type(8))) _Float16 mm_f16x8;
typedef __attribute__((ext_vector_type(4))) uint32_t mm_chunk;   // 16 bytes of an operand

// acc += a b over the chunk's four (f32) or eight consecutive k of each lane half: 32 x 32 outputs.
template <typename T> __device__ __forceinline__ mm_f32x16 mm_mfma(mm_chunk a, mm_chunk b, mm_f32x16 acc);
template <> __device__ __forceinline__ mm_f32x16 mm_mfma<float>(mm_chunk a, mm_chunk b, mm_f32x16 acc) {
  const mm_f32x4 x = __builtin_bit_cast(mm_f32x4, a), y = __builtin_bit_cast(mm_f32x4, b);
#pragma unroll
  for (int s = 0; s < 4; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x[s], y[s], acc, 0, 0, 0);
  return acc;
}
template <> __device__ __forceinline__ mm_f32x16 mm_mfma<bf16_raw>(mm_chunk a, mm_chunk b, mm_f32x16 acc) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(mm_bf16x8, a), __builtin_bit_cast(mm_bf16x8, b), acc, 0, 0, 0);
}
template <> __device__ __forceinline__ mm_f32x16 mm_mfma<f16_raw>(mm_chunk a, mm_chunk b, mm_f32x16 acc) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(mm_f16x8, a), __builtin_bit_cast(mm_f16x8, b), acc, 0, 0, 0);
}

// One operand's tile of ROWS outputs x KB bytes of K.  KC (contiguous along K): in LDS as rows of KB + 16 bytes.  Otherwise
// as it lies, BK rows of ROWS elements + 16 bytes, and the fragments are put together on the way out: 16-bit elements
// with the transposing LDS read (lane i of 16 receives element i % 4 of the 8 bytes that lanes 4j + i / 4, j = 0..3, point
// at: with lane a pointing at row a / 4, columns 4 (a % 4), it receives column i of four rows), f32 one by one.
// Memory is read in pieces of 16 bytes whatever their alignment, every one of them whole: a piece that would reach past an end
// is read as much earlier, and moved down and filled up with zeros on its way into LDS.  (A load under a mask, or in one of two
// branches, is waited for where those end: the second operand's loads then begin when the first's have come.)  Only a K, or a
// row of outputs, of less than a piece is read by pairs or elements.
template <typename T, int ROWS, bool KC, int KB, int R, bool TINY>
struct MmOperand {
  static constexpr int V = 16 / sizeof(T), BK = KB / sizeof(T), CPR = KC ? KB / 16 : ROWS / V, PIECES = ROWS * KB / 16, P = (PIECES + 255) / 256;
  static constexpr int PITCH = (KC ? KB : ROWS * (int)sizeof(T)) + 16;
  static constexpr int BYTES = (KC ? ROWS : BK) * PITCH;
  const T *base;      // the tile's first output row (column), k = 0
  int64_t stride;     // KC: between outputs; otherwise: between consecutive k
  int valid, K;       // outputs that exist from the tile's first on (the operand has V of them or more); the length of K
  bool tiny;          // (TINY) fewer than V outputs (!KC), a K below V (KC)
  int k_reg[R];       // where in K the pieces held begin
  const T *at[P];     // this thread's pieces at k = 0
  mm_chunk reg[R][P];

  // place of this thread's piece p: KC: (output, chunk of K); otherwise (k, chunk of outputs)
  static __device__ __forceinline__ int row(int p) { return (threadIdx.x + 256 * p) / CPR; }
  static __device__ __forceinline__ int col(int p) { return ((threadIdx.x + 256 * p) % CPR) * V; }

  // The whole tile lies inside the operand (outputs past the end aside, which are read from the last one).
  __device__ __forceinline__ bool whole(int k0) const { return k0 + BK <= K && (KC || valid >= ROWS); }
  __device__ __forceinline__ void begin() {
    if (TINY && tiny) return;
#pragma unroll
    for (int p = 0; p < P; ++p) at[p] = base + (KC ? min(row(p), valid - 1) : min(row(p), K - 1)) * stride + (KC ? 0 : min(col(p), valid - V));
  }
  // !KC: by how much the tile is read earlier, so that all its rows exist (where K has as many)
  __device__ __forceinline__ int back(int k0) const { return K < BK ? k0 : max(k0 + BK - K, 0); }
  __device__ __forceinline__ void fetch(int k0, int set) {   // (past K: the last pieces once more, or the last rows)
    k_reg[set] = k0;
    if (!(TINY && tiny)) {
      const int64_t ahead = KC ? 0 : (k0 - back(k0)) * stride;
#pragma unroll
      for (int p = 0; p < P; ++p) __builtin_memcpy(&reg[set][p], at[p] + (KC ? (int64_t)min(k0 + col(p), K - V) : ahead), 16);
      return;
    }
#pragma unroll
    for (int p = 0; p < P; ++p) {   // zeros past K, the last output repeated
      const int k = KC ? k0 + col(p) : k0 + row(p), o = KC ? min(row(p), valid - 1) : col(p);
      if (k >= K) {
        reg[set][p] = mm_chunk{0u, 0u, 0u, 0u};
      } else if (KC && sizeof(T) == 2 && K > 1) {   // by pairs (by elements up to 1.1 us more: 11 x 1 x 11 x 93 in bf16 5.3, now 4.5)
        const T *at_o = base + (int64_t)o * stride;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          uint32_t two;
          __builtin_memcpy(&two, at_o + min(2 * j, K - 2), 4);
          reg[set][p][j] = 2 * j < K - 1 ? two : 2 * j == K - 1 ? two >> 16 : 0u;
        }
      } else {
        T v[V];
#pragma unroll
        for (int j = 0; j < V; ++j) v[j] = KC ? base[(int64_t)o * stride + min(k + j, K - 1)] : base[(int64_t)k * stride + min(o + j, valid - 1)];
        if (KC) {
#pragma unroll
          for (int j = 0; j < V; ++j)
            if (k + j >= K) v[j] = T{};
        }
        __builtin_memcpy(&reg[set][p], v, 16);
      }
    }
  }
  // A piece that was read `past` elements (below V) ahead of its place: what lies past the end is zero.
  static __device__ __forceinline__ mm_chunk end_of_k(mm_chunk v, int past) {
    const int bits = past * (int)sizeof(T) * 8;
    const uint64_t lo = (uint64_t)v[1] << 32 | v[0], hi = (uint64_t)v[3] << 32 | v[2], up = hi >> (bits & 63);
    const uint64_t a = bits < 64 ? lo >> (bits & 63) | hi << 1 << (63 - (bits & 63)) : up, b = bits < 64 ? up : 0;
    return mm_chunk{(uint32_t)a, (uint32_t)(a >> 32), (uint32_t)b, (uint32_t)(b >> 32)};
  }
  __device__ __forceinline__ void park(char *st, int set) const {
    const bool ends = !whole(k_reg[set]) && !(TINY && tiny), moved = ends && (KC ? K : valid) % V != 0;
    const int k0 = k_reg[set];
#pragma unroll
    for (int p = 0; p < P; ++p) {
      if (PIECES % 256 && (int)threadIdx.x + 256 * p >= PIECES) continue;
      if (!ends) {
        *reinterpret_cast<mm_chunk *>(st + row(p) * PITCH + col(p) * (int)sizeof(T)) = reg[set][p];
        continue;
      }
      mm_chunk v = reg[set][p];
      const int past = KC ? k0 + col(p) + V - K : max(col(p) + V - valid, 0);
      if (moved) v = end_of_k(v, past < 0 || past >= V ? 0 : past);
      int to = row(p);
      bool none = KC ? past >= V : to >= K;
      if (!KC && K >= BK) {   // what was read earlier than its place goes there; rows that were read before make room for zeros
        to -= back(k0);
        none = to < 0;
        if (none) to += BK;
      }
      if (none) v = mm_chunk{0u, 0u, 0u, 0u};
      *reinterpret_cast<mm_chunk *>(st + to * PITCH + col(p) * (int)sizeof(T)) = v;
    }
  }
  // Outputs first .. first + 31, chunk pair kk of K: lane (r, h) gets chunk 2 kk + h of output first + r.
  static __device__ __forceinline__ mm_chunk fragment(const char *st, int first, int kk) {
    const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
    if constexpr (KC) {
      return *reinterpret_cast<const mm_chunk *>(st + (first + r) * PITCH + kk * 32 + h * 16);
    } else if constexpr (sizeof(T) == 2) {
      typedef __attribute__((ext_vector_type(4))) short s16x4;
      typedef __attribute__((address_space(3))) s16x4 *tr_ptr;
      const int i = lane & 15, o = first + 16 * ((lane >> 4) & 1) + 4 * (i & 3);
      const char *at = st + (kk * 16 + h * 8 + (i >> 2)) * PITCH + o * 2;
      const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr)at);
      const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr)(at + 4 * PITCH));
      const __attribute__((ext_vector_type(8))) short f = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      return __builtin_bit_cast(mm_chunk, f);
    } else {
      mm_f32x4 f;
#pragma unroll
      for (int j = 0; j < 4; ++j) f[j] = *reinterpret_cast<const float *>(st + (kk * 8 + h * 4 + j) * PITCH + (first + r) * 4);
      return __builtin_bit_cast(mm_chunk, f);
    }
  }
};

// Four sums as consecutive outputs.
__device__ __forceinline__ void mm_round4(char *dst, mm_f32x4 v, float) { *reinterpret_cast<mm_f32x4 *>(dst) = v; }
__device__ __forceinline__ void mm_round4(char *dst, mm_f32x4 v, bf16_raw) { *reinterpret_cast<uint2 *>(dst) = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])); }
__device__ __forceinline__ void mm_round4(char *dst, mm_f32x4 v, f16_raw) {
  typedef __attribute__((ext_vector_type(4))) _Float16 h4;
  *reinterpret_cast<h4 *>(dst) = h4{(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
}
template <typename T> __device__ __forceinline__ void mm_store(T *dst, mm_chunk w, int n) {   // up to V outputs of a row
  constexpr int V = 16 / sizeof(T);
  if (n >= V) {
    __builtin_memcpy(dst, &w, 16);
  } else {
    asm volatile("" : "+v"(w));   // (or the last store of both branches becomes one, and the whole piece three)
    T v[V];
    __builtin_memcpy(v, &w, 16);
#pragma unroll
    for (int j = 0; j < V; ++j)
      if (j < n) dst[j] = v[j];
  }
}

// Four waves as 2 x 2, each F x F accumulators of 32 x 32 (tiles of 64 F).  Two LDS stages of KB bytes of K, loaded into
// registers one tile ahead (R: two), one barrier per tile, or (ONE: K fits) a single one.  The products are formed as B^T A^T, so
// that a lane's four sums in a row of registers are four outputs in a row: they are rounded, and go through LDS and out 16 bytes
// at a time.  Attention-sized products are bound by the vector instructions around a tile's few MFMAs (eight waves to a SIMD at 32 x
// 512 x 80 x 512, each with some hundreds) and by the chain of trips, long ones by the L2: hence large tiles wherever they
// leave no CU idle, addresses that are made once, loads without conditions, and the scalars asked for together.
//   Measured (us; before that, with tiles of 64, masked loads and f32 through LDS): bf16 32 x 512 x 80 x 512 (scores) 10.8 -> 7.3, 32 x
// 1024 x 128 x 1024 30.3 -> 21.3, 32 x 512 x 512 x 80 (values, [K, N]) 12.5 -> 7.9, 32 x 512 x 256 x 512 16.8 -> 9.9, odd 16 x 410 x 141 x 349
// 8.4 -> 7.0, one row against 32 x 777 x 128 9.3 -> 8.0; f32 32 x 512 x 80 x 512 25 -> 20.8, 32 x 1024 x 80 x 1024 76 -> 62.
template <typename T, bool AKC, bool BKC, int F, int KB, bool ONE, bool TINY = false>
__global__ void __launch_bounds__(256, F == 2 ? 2 : 3) k_matmul_mfma(T *out, const T *A, const T *B, MatmulArgs g, int tiles_m, int tiles_n) {
  constexpr int BT = 64 * F;
  constexpr int R = F == 1 && !ONE && sizeof(T) == 2 ? 2 : 1;   // tiles in registers, on their way
  typedef MmOperand<T, BT, AKC, KB, R, TINY> OpA;
  typedef MmOperand<T, BT, BKC, KB, R, TINY> OpB;
  constexpr int STAGE = OpA::BYTES + OpB::BYTES, OP = BT * (int)sizeof(T) + 16, PAIRS = KB / 32;
  constexpr int LDS = (ONE ? 1 : 2) * STAGE > BT * OP ? (ONE ? 1 : 2) * STAGE : BT * OP;
  __shared__ __attribute__((aligned(16))) char lds[LDS];
  // (asked for together: a dependent chain of scalar loads is a good part of a small tile's time)
  int64_t a_bs = g.a_bs[0], b_bs = g.b_bs[0], as = AKC ? g.a_rs : g.a_cs, bs = BKC ? g.b_cs : g.b_rs;
  asm volatile("" : "+s"(a_bs), "+s"(b_bs), "+s"(as), "+s"(bs));
  // every XCD (blocks are dealt out to the eight of them in turn) walks a run of tiles of its own: the tiles of one batch
  // entry then share its L2
  const int total = gridDim.x, xcd = blockIdx.x & 7, q = total >> 3, rem = total & 7;
  const int t = xcd * q + (xcd < rem ? xcd : rem) + (blockIdx.x >> 3);
  const int z = t / (tiles_m * tiles_n), in = t - z * tiles_m * tiles_n;
  const int m0 = (in % tiles_m) * BT, n0 = (in / tiles_m) * BT;
  int64_t aoff = z * a_bs, boff = z * b_bs;
  if (g.batch_rank > 1) {
    aoff = boff = 0;
    for (int d = g.batch_rank - 1, rest = z; d >= 0; --d) {
      const int n = (int)g.batch_shape[d], i = rest % n;
      rest /= n;
      aoff += i * g.a_bs[d];
      boff += i * g.b_bs[d];
    }
  }
  OpA a;
  a.stride = as;
  a.base = A + aoff + (AKC ? m0 * as : (int64_t)m0);
  a.valid = (int)min<int64_t>(BT, g.M - m0);
  a.K = (int)g.K;
  a.tiny = TINY && (AKC ? g.K : g.M) < OpA::V;
  OpB b;
  b.stride = bs;
  b.base = B + boff + (BKC ? n0 * bs : (int64_t)n0);
  b.valid = (int)min<int64_t>(BT, g.N - n0);
  b.K = (int)g.K;
  b.tiny = TINY && (BKC ? g.K : g.N) < OpB::V;

  const int wave = threadIdx.x >> 6, wm = (wave >> 1) * 32 * F, wn = (wave & 1) * 32 * F;
  mm_f32x16 acc[F][F];
#pragma unroll
  for (int i = 0; i < F; ++i)
#pragma unroll
    for (int j = 0; j < F; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  a.begin();
  b.begin();
  const int steps = ONE ? 1 : ((int)g.K + OpA::BK - 1) / OpA::BK;
#pragma unroll
  for (int i = 0; i < R; ++i) {
    a.fetch(i * OpA::BK, i);
    b.fetch(i * OpA::BK, i);
  }
  a.park(lds, 0);
  b.park(lds + OpA::BYTES, 0);
  if (R > 1 || steps > 1) { a.fetch(R * OpA::BK, 0); b.fetch(R * OpA::BK, 0); }
  __syncthreads();
  auto step = [&](int s, int set) __attribute__((always_inline)) {   // set: what the next tile is in
    const char *sa = lds + (s & 1) * STAGE, *sb = sa + OpA::BYTES;
    mm_chunk fa[2][F], fb[2][F];
    auto read = [&](int kk) {
#pragma unroll
      for (int i = 0; i < F; ++i) fa[kk & 1][i] = OpA::fragment(sa, wm + 32 * i, kk);
#pragma unroll
      for (int j = 0; j < F; ++j) fb[kk & 1][j] = OpB::fragment(sb, wn + 32 * j, kk);
    };
    read(0);
#pragma unroll
    for (int kk = 0; kk < PAIRS; ++kk) {
      if (kk + 1 < PAIRS) read(kk + 1);
      if (!ONE && kk == 2 && (R > 1 || s + 1 < steps)) {   // to the stage that every wave left before the last barrier
        char *next = lds + ((s + 1) & 1) * STAGE;
        a.park(next, set);
        b.park(next + OpA::BYTES, set);
        if (R > 1 || s + 2 < steps) { a.fetch((s + 1 + R) * OpA::BK, set); b.fetch((s + 1 + R) * OpA::BK, set); }
      }
      if (ONE && sizeof(T) == 4 && kk * 8 >= (int)g.K) break;   // (256 cycles to a step of f32)
#pragma unroll
      for (int i = 0; i < F; ++i)
#pragma unroll
        for (int j = 0; j < F; ++j) acc[i][j] = mm_mfma<T>(fb[kk & 1][j], fa[kk & 1][i], acc[i][j]);
    }
    __syncthreads();
  };
  for (int s = 0;;) {   // (with two sets: no request under a condition, whose number the next wait would not know)
    step(s, R - 1);
    if (++s >= steps) break;
    if (R > 1) {
      step(s, 0);
      if (++s >= steps) break;
    }
  }
  // accumulator register e of lane (r, h) is column 8 (e / 4) + 4 h + e % 4, row r: four outputs in a row at a time
  const int r = threadIdx.x & 31, h = (threadIdx.x >> 5) & 1;
  char *mine = lds + (wm + r) * OP + (wn + 4 * h) * (int)sizeof(T);
#pragma unroll
  for (int i = 0; i < F; ++i)
#pragma unroll
    for (int j = 0; j < F; ++j)
#pragma unroll
      for (int e = 0; e < 16; e += 4)
        mm_round4(mine + 32 * i * OP + (32 * j + 2 * e) * (int)sizeof(T), mm_f32x4{acc[i][j][e], acc[i][j][e + 1], acc[i][j][e + 2], acc[i][j][e + 3]}, T());
  __syncthreads();
  constexpr int V = OpA::V, RUN = BT / V, ROWS = 256 / RUN;   // pieces of a row, rows at a time
  const int row = threadIdx.x / RUN, col = threadIdx.x % RUN * V, left = b.valid - col;
  T *o = out + (int64_t)z * g.M * g.N + (int64_t)(m0 + row) * g.N + n0 + col;
  const char *from = lds + row * OP + col * (int)sizeof(T);
  if (left <= 0) return;
#pragma unroll
  for (int e = 0; e < BT / ROWS; ++e) {
    if (row + e * ROWS < a.valid) mm_store<T>(o, *reinterpret_cast<const mm_chunk *>(from + e * ROWS * OP), left);
    o += ROWS * g.N;
  }
}

template <typename T, bool AKC, bool BKC>
static int launch_mm(hipStream_t st, void *out, const void *A, const void *B, const MatmulArgs &g, int64_t batch) {
  // 64 x 64 tiles; 16-bit operands take 128 x 128 (half the operand traffic and a fraction of the instructions per product) once
  // those give every CU two and are not mostly edge (us, 64 and 128: 32 x 512 x 80 x 512 8.5, 7.4; 32 x 512 x 160 x 512 11.2, 10.6 before
  // the loop had two tiles on their way; 32 x 1024 x 64 x 1024 16.4, 14.5; but 32 x 256 x 80 x 256 4.5, 4.8, 64 x 300 x 128 x 300 8.3, 10.5).
  //   As long as a tile's K is short, it needs no second stage: one load phase, and less LDS, so more blocks to a CU (us, two
  // stages, one: 32 x 512 x 80 x 512 with 128 10.5, 7.4; 8 x 900 x 80 x 700 with 64 8.4, 6.7; 16 x 410 x 141 x 349 8.0, 7.0).
  const int64_t t64 = batch * ((g.M + 63) / 64) * ((g.N + 63) / 64), tm128 = (g.M + 127) / 128, tn128 = (g.N + 127) / 128;
  const int kb = (int)(g.K * (int64_t)sizeof(T) < 512 ? g.K * sizeof(T) : 512);
  const int tm = (int)((g.M + 63) / 64), tn = (int)((g.N + 63) / 64);
  auto go = [&](auto kernel, int64_t blocks, int tiles_m, int tiles_n) -> int {
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(256), 0, st, (T *)out, (const T *)A, (const T *)B, g, tiles_m, tiles_n);
    return launch_check("matmul_mfma");
  };
  constexpr int V = 16 / sizeof(T);
  if ((AKC || BKC) && g.K < V || !AKC && g.M < V || !BKC && g.N < V)
    return kb <= 128 ? go(k_matmul_mfma<T, AKC, BKC, 1, 128, true, true>, t64, tm, tn) : go(k_matmul_mfma<T, AKC, BKC, 1, 128, false, true>, t64, tm, tn);
  if constexpr (sizeof(T) == 2) {
    const int64_t t128 = batch * tm128 * tn128;
    auto large = [&](auto kernel) { return go(kernel, t128, (int)tm128, (int)tn128); };
    if (t128 >= 2 * kNumCU && (g.K >= 256 || t128 * 16 <= t64 * 5)) {
      if (kb <= 128) return large(k_matmul_mfma<T, AKC, BKC, 2, 128, true>);
      if (kb <= 160) return large(k_matmul_mfma<T, AKC, BKC, 2, 160, true>);
      if (kb <= 192) return large(k_matmul_mfma<T, AKC, BKC, 2, 192, true>);
      if (kb <= 256) return large(k_matmul_mfma<T, AKC, BKC, 2, 256, true>);
      return large(k_matmul_mfma<T, AKC, BKC, 2, 128, false>);
    }
  }
  if (kb <= 128) return go(k_matmul_mfma<T, AKC, BKC, 1, 128, true>, t64, tm, tn);
  if (kb <= 192) return go(k_matmul_mfma<T, AKC, BKC, 1, 192, true>, t64, tm, tn);
  if (kb <= 256) return go(k_matmul_mfma<T, AKC, BKC, 1, 256, true>, t64, tm, tn);
  if (kb <= 320) return go(k_matmul_mfma<T, AKC, BKC, 1, 320, true>, t64, tm, tn);
  return go(k_matmul_mfma<T, AKC, BKC, 1, 128, false>, t64, tm, tn);
}

bool matmul_mfma_serves(int dtype, const MatmulArgs &g, int64_t batch) {
  const bool a = g.a_cs == 1 || g.a_rs == 1 || g.K == 1 || g.M == 1, b = g.b_rs == 1 || g.b_cs == 1 || g.K == 1 || g.N == 1;
  return (dtype == RAI_F32 || dtype == RAI_BF16 || dtype == RAI_F16) && a && b && g.K < (1 << 30) && g.M < (1LL << 30) && g.N < (1LL << 30) &&
         batch * ((g.M + 63) / 64) * ((g.N + 63) / 64) < (1LL << 31);
}

int launch_matmul_mfma(hipStream_t st, int dtype, void *out, const void *A, const void *B, const MatmulArgs &g0, int64_t batch) {
  MatmulArgs g = g0;
  // batch axes that one stride walks become one, so that most products have no more than one
  int rank = 0;
  for (int d = 0; d < g0.batch_rank; ++d) {
    if (g0.batch_shape[d] == 1) continue;
    const int64_t n = g0.batch_shape[d];
    if (rank && g.a_bs[rank - 1] == g0.a_bs[d] * n && g.b_bs[rank - 1] == g0.b_bs[d] * n) {
      g.batch_shape[rank - 1] *= n;
      --rank;
    } else {
      g.batch_shape[rank] = n;
    }
    g.a_bs[rank] = g0.a_bs[d];
    g.b_bs[rank] = g0.b_bs[d];
    ++rank;
  }
  if (!rank) g.a_bs[0] = g.b_bs[0] = 0;
  g.batch_rank = rank;
  // an axis of one element has no stride of its own
  const bool akc = g.a_cs == 1 || g.K == 1, bkc = g.b_rs == 1 || g.K == 1;
  auto go = [&](auto t) -> int {
    typedef decltype(t) T;
    if (akc) return bkc ? launch_mm<T, true, true>(st, out, A, B, g, batch) : launch_mm<T, true, false>(st, out, A, B, g, batch);
    return bkc ? launch_mm<T, false, true>(st, out, A, B, g, batch) : launch_mm<T, false, false>(st, out, A, B, g, batch);
  };
  if (dtype == RAI_F32) return go(float());
  return dtype == RAI_BF16 ? go(bf16_raw()) : go(f16_raw());
}

}  // namespace rai
