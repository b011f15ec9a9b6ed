// Batched products of strided operands on the matrix instructions: f32, bf16 and f16, each operand contiguous along K or
// along its other axis, any batch strides.  (Products whose right operand is one shared, K-contiguous matrix are Linears;
// f64 and operands without a unit stride stay with k_matmul_generic.)
//
// Reference semantics: rai-core/src/backend/candle.rs:327-443 (MatMul, stride rule).
#include <type_traits>

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
// Memory is read in pieces of 16 bytes whatever their alignment; where K ends inside one (KC), or the outputs do (otherwise), the last 16 bytes of
// the row are read and moved down when they go to LDS, or a K of less than a piece by pairs (element by element, 16-bit operands with K of 9 to 15 took up to
// 1.1 us more than multiply-adds on the vector units: 11 x 1 x 11 x 93 in bf16 4.2 us there, 5.3, now 4.5).
// A K of two stages and more, both operands contiguous along it, of 16 bits and off 16-byte boundaries (OFF): the fetch that asks where a tile ends.  A loop that
// read them without a condition (products formed transposed, 128 x 128 tiles) once gave 130 x 255 x 129 x 241 wrong in one call of three, one piece of one
// operand in one tile, and no cause was found in its source or its assembly: its loads write over their own addresses, but so do those of
// forms that have never failed.  Its single stages did not fail, and none of the other layouts.  What it costs (us): 64 x 1000 x 999 x 1001
// 263, 356; 130 x 255 x 129 x 241 16.4, 18.6; 7 x 481 x 943 x 246 9.1, 9.9.
template <typename T, int ROWS, bool KC, int KB, bool OFF>
struct MmOperand {
  static constexpr int V = 16 / sizeof(T), BK = KB / sizeof(T), CPR = KC ? KB / 16 : ROWS / V, P = ROWS * KB / 16 / 256;
  static constexpr int PITCH = (KC ? KB : ROWS * (int)sizeof(T)) + 16;
  static constexpr int BYTES = (KC ? ROWS : BK) * PITCH;
  const T *base;      // the tile's first output row (column), k = 0
  int64_t stride;     // KC: between outputs; otherwise: between consecutive k
  int valid, K;       // outputs that exist from the tile's first on; the length of K
  int before;         // outputs before the tile's first
  mm_chunk reg[P];

  // place of this thread's piece p: KC: (output, chunk of K); otherwise (k, chunk of outputs)
  static __device__ __forceinline__ int row(int p) { return (threadIdx.x + 256 * p) / CPR; }
  static __device__ __forceinline__ int col(int p) { return ((threadIdx.x + 256 * p) % CPR) * V; }

  // Every row has a piece, so that one can be read for every place.
  __device__ __forceinline__ bool pieces() const { return KC ? K >= V : before + valid >= V; }
  // How a step is fetched and put into LDS: all of it inside the operand; whole in K, where the outputs may end inside; any.  None of these has a
  // branch, so that it stays between the products of the step before.  kGuarded: rows of this operand or the other have no piece, or OFF.
  enum { kInside, kOutputsEnd, kEnds, kGuarded };
  template <int MODE> __device__ __forceinline__ void fetch(int k0) {
    if constexpr (MODE == kGuarded) {
      if (!OFF && pieces()) fetch<kEnds>(k0);
      else fetch_guarded(k0);
    } else {
#pragma unroll
      for (int p = 0; p < P; ++p) {   // at an end: the last 16 bytes of the row, or the last row, again
        const int k = KC ? k0 + col(p) : k0 + row(p), o = KC ? min(row(p), valid - 1) : col(p);
        const T *at = KC ? base + (int64_t)o * stride + (MODE == kEnds ? min(k, K - V) : k)
                         : base + (int64_t)(MODE == kEnds ? min(k, K - 1) : k) * stride + (MODE == kInside ? o : min(o, valid - V));
        __builtin_memcpy(&reg[p], at, 16);
      }
    }
  }
  // To LDS, what was fetched for k0; a piece that was read ahead of its place goes there now.
  template <int MODE> __device__ __forceinline__ void park(char *st, int k0) const {
    if constexpr (MODE == kGuarded) {
      if (!OFF && pieces()) return park<kEnds>(st, k0);
    }
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const int k = KC ? k0 + col(p) : k0 + row(p);
      mm_chunk v = reg[p];
      if (MODE == kEnds || (MODE == kOutputsEnd && !KC)) v = end_of_row(v, KC ? k + V - K : col(p) + V - valid);
      if (MODE == kEnds) v = k < K ? v : mm_chunk{0u, 0u, 0u, 0u};
      *reinterpret_cast<mm_chunk *>(st + row(p) * PITCH + col(p) * (int)sizeof(T)) = v;
    }
  }
  __device__ __forceinline__ void fetch_guarded(int k0) {
    if (KC && OFF && k0 + BK <= K) {
#pragma unroll
      for (int p = 0; p < P; ++p) __builtin_memcpy(&reg[p], base + (int64_t)min(row(p), valid - 1) * stride + k0 + col(p), 16);
      return;
    }
#pragma unroll
    for (int p = 0; p < P; ++p) {   // at the ends, or rows of less than a piece: zeros past K, the last output repeated
      const int k = KC ? k0 + col(p) : k0 + row(p), o = KC ? min(row(p), valid - 1) : col(p);
      if (k >= K) {
        reg[p] = mm_chunk{0u, 0u, 0u, 0u};
      } else if (KC && OFF && k + V <= K) {
        __builtin_memcpy(&reg[p], base + (int64_t)o * stride + k, 16);
      } else if (KC && OFF && K >= V) {   // the piece that ends with K, moved down
        __builtin_memcpy(&reg[p], base + (int64_t)o * stride + (K - V), 16);
        reg[p] = end_of_row(reg[p], k + V - K);
      } else if (KC && sizeof(T) == 2 && K > 1) {   // a shorter K, by pairs
        const T *at_o = base + (int64_t)o * stride;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          uint32_t two;
          __builtin_memcpy(&two, at_o + min(2 * j, K - 2), 4);
          reg[p][j] = 2 * j < K - 1 ? two : 2 * j == K - 1 ? two >> 16 : 0u;
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
        __builtin_memcpy(&reg[p], v, 16);
      }
    }
  }
  // A piece that was read `past` elements (none: past <= 0) ahead of its place: what lies past the end is zero.  (V and more: not zero, of no use.)
  static __device__ __forceinline__ mm_chunk end_of_row(mm_chunk v, int past) {
    past = max(past, 0);
    const int words = past * (int)sizeof(T) / 4;
#pragma unroll
    for (int i = 0; i < 3; ++i)
      if (words > i) v = mm_chunk{v[1], v[2], v[3], 0u};
    if (sizeof(T) == 2 && (past & 1)) v = mm_chunk{v[0] >> 16 | v[1] << 16, v[1] >> 16 | v[2] << 16, v[2] >> 16 | v[3] << 16, v[3] >> 16};
    return v;
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

template <typename T> __device__ __forceinline__ void mm_store(T *dst, const float *src, int n) {   // up to V outputs of a row
  constexpr int V = 16 / sizeof(T);
  T v[V];
#pragma unroll
  for (int j = 0; j < V; ++j) Scalar<T>::store(&v[j], src[j]);
  if (n >= V) {
    __builtin_memcpy(dst, v, 16);
  } else {
#pragma unroll
    for (int j = 0; j < V; ++j)
      if (j < n) dst[j] = v[j];
  }
}

// Four waves as 2 x 2, each F x F accumulators of 32 x 32 (tiles of 64 F).  Two LDS stages of KB bytes of K, loaded into
// registers a tile ahead, one barrier per tile, or (ONE: K fits) a single one; the finished tile goes through LDS so that
// rows are written 16 bytes at a time.  Attention-sized products are bound by a block's chain of trips (operands, LDS,
// MFMAs, LDS, rows out), so what counts is how many blocks share a CU; long ones by the L2.
//   Measured (us; 64 x 64 tiles of multiply-adds on the vector units before): bf16 32 x 512 x 80 x 512 (scores) 11.2 (40.5),
// 32 x 512 x 512 x 80 (values, [K, N]) 13.4 (94.8), 64 x 1024 x 1024 x 1024 200 to 316 (2900 to 3035), one row against 32 x
// 777 x 128 10.4 (77.5), odd 18 x 410 x 141 x 349 10.8 (31.8); f32 32 x 512 x 80 x 512 24.4 (47.9).
//   A step has no branch: the ends of rows are put right by moving what was read, not by asking where it lies (us, with branches, and now): bf16 64 x
// 1024 x 1024 x 1024, [K, N] 300, 207 to 212, K-contiguous 305, 202, 64 x 1000 x 999 x 1001, [K, N] 454, 266, 7 x 481 x 944 x 246 27.9, 11.2,
// 18 x 169 x 639 x 234 19.3, 9.1, 19 x 30 x 192 x 34 6.3, 4.8, f16 5 x 9 x 723 x 56 14.6, 8.0; f32 3 x 15 x 737 x 625 24.1, 21.1, 64 x 128 x 512 x 128
// 16.6, 15.8.  f32, whose products take longer, loads a step ahead from its first products on (from the third: 17.1).  Stages of
// 256 bytes: 0.95 to 1.33 of the time.
template <typename T, bool AKC, bool BKC, int F, int KB, bool ONE, bool OFF = false>
__global__ void __launch_bounds__(256) k_matmul_mfma(T *out, const T *A, const T *B, MatmulArgs g, int tiles_m, int tiles_n) {
  constexpr int BT = 64 * F;
  typedef MmOperand<T, BT, AKC, KB, OFF> OpA;
  typedef MmOperand<T, BT, BKC, KB, OFF> OpB;
  constexpr int STAGE = OpA::BYTES + OpB::BYTES, OP = BT + 4, PAIRS = KB / 32;
  constexpr int LDS = (ONE ? 1 : 2) * STAGE > BT * OP * 4 ? (ONE ? 1 : 2) * STAGE : BT * OP * 4;
  __shared__ __attribute__((aligned(16))) char lds[LDS];
  // every XCD (blocks are dealt out to the eight of them in turn) walks a run of tiles of its own: the tiles of one batch
  // entry then share its L2
  const int total = gridDim.x, xcd = blockIdx.x & 7, q = total >> 3, rem = total & 7;
  const int t = xcd * q + (xcd < rem ? xcd : rem) + (blockIdx.x >> 3);
  const int z = t / (tiles_m * tiles_n), in = t - z * tiles_m * tiles_n;
  const int m0 = (in % tiles_m) * BT, n0 = (in / tiles_m) * BT;
  int64_t aoff = 0, boff = 0;
  for (int d = g.batch_rank - 1, rest = z; d >= 0; --d) {
    const int n = (int)g.batch_shape[d], i = rest % n;
    rest /= n;
    aoff += i * g.a_bs[d];
    boff += i * g.b_bs[d];
  }
  OpA a;
  a.stride = AKC ? g.a_rs : g.a_cs;
  a.base = A + aoff + (AKC ? (int64_t)m0 * g.a_rs : (int64_t)m0);
  a.valid = (int)min<int64_t>(BT, g.M - m0);
  a.K = (int)g.K;
  a.before = m0;
  OpB b;
  b.stride = BKC ? g.b_cs : g.b_rs;
  b.base = B + boff + (BKC ? (int64_t)n0 * g.b_cs : (int64_t)n0);
  b.valid = (int)min<int64_t>(BT, g.N - n0);
  b.K = (int)g.K;
  b.before = n0;

  const int wave = threadIdx.x >> 6, wm = (wave >> 1) * 32 * F, wn = (wave & 1) * 32 * F;
  mm_f32x16 acc[F][F];
#pragma unroll
  for (int i = 0; i < F; ++i)
#pragma unroll
    for (int j = 0; j < F; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  const int steps = ONE ? 1 : ((int)g.K + OpA::BK - 1) / OpA::BK;
  constexpr int kInside = OpA::kInside, kOutputsEnd = OpA::kOutputsEnd, kEnds = OpA::kEnds, kGuarded = OpA::kGuarded;
  const bool pieces = !OFF && a.pieces() && b.pieces();
  auto begin = [&](auto how) __attribute__((always_inline)) {
    constexpr int MODE = decltype(how)::value;
    a.template fetch<MODE>(0);
    b.template fetch<MODE>(0);
    a.template park<MODE>(lds, 0);
    b.template park<MODE>(lds + OpA::BYTES, 0);
    if (steps > 1) { a.template fetch<MODE>(OpA::BK); b.template fetch<MODE>(OpA::BK); }
    __syncthreads();
  };
  int s = 0;
  auto step = [&](auto how) __attribute__((always_inline)) {
    constexpr int MODE = decltype(how)::value;
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
      if (ONE && kk * (32 / (int)sizeof(T)) >= (int)g.K) break;
      if (kk + 1 < PAIRS) read(kk + 1);
      if (kk == (sizeof(T) == 4 ? 0 : 2) && (MODE < kEnds || s + 1 < steps)) {   // to the stage that every wave left before the last barrier
        char *next = lds + ((s + 1) & 1) * STAGE;
        if constexpr (F == 1) __builtin_amdgcn_sched_barrier(0);   // (what the compiler moves across costs short products 1 to 5 %)
        a.template park<MODE>(next, (s + 1) * OpA::BK);
        b.template park<MODE>(next + OpA::BYTES, (s + 1) * OpA::BK);
        if (MODE < kEnds || s + 2 < steps) { a.template fetch<MODE>((s + 2) * OpA::BK); b.template fetch<MODE>((s + 2) * OpA::BK); }
        if constexpr (F == 1) __builtin_amdgcn_sched_barrier(0);   // (what the compiler moves across costs short products 1 to 5 %)
      }
#pragma unroll
      for (int i = 0; i < F; ++i)
#pragma unroll
        for (int j = 0; j < F; ++j) acc[i][j] = mm_mfma<T>(fa[kk & 1][i], fb[kk & 1][j], acc[i][j]);
    }
    __syncthreads();
  };
  if (!pieces) {
    begin(std::integral_constant<int, kGuarded>{});
    for (; s < steps; ++s) step(std::integral_constant<int, kGuarded>{});
  } else {
    begin(std::integral_constant<int, kEnds>{});
    if constexpr (!ONE) {   // the steps that fetch one before the last, whole in K
      if ((AKC || a.valid >= BT) && (BKC || b.valid >= BT)) {
        for (; s + 3 < steps; ++s) step(std::integral_constant<int, kInside>{});
      } else {
        for (; s + 3 < steps; ++s) step(std::integral_constant<int, kOutputsEnd>{});
      }
    }
    for (; s < steps; ++s) step(std::integral_constant<int, kEnds>{});
  }
  // accumulator register e of lane (r, h) is row 8 (e / 4) + 4 h + e % 4, column r
  float *f = reinterpret_cast<float *>(lds);
  const int r = threadIdx.x & 31, h = (threadIdx.x >> 5) & 1;
#pragma unroll
  for (int i = 0; i < F; ++i)
#pragma unroll
    for (int j = 0; j < F; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) f[(wm + 32 * i + 8 * (e >> 2) + 4 * h + (e & 3)) * OP + wn + 32 * j + r] = acc[i][j][e];
  __syncthreads();
  T *o = out + (int64_t)z * g.M * g.N;
  constexpr int V = OpA::V;
#pragma unroll 2
  for (int e = threadIdx.x; e < BT * BT / V; e += 256) {
    const int row = e / (BT / V), col = (e % (BT / V)) * V;
    if (row < a.valid && col < b.valid) mm_store<T>(o + (int64_t)(m0 + row) * g.N + n0 + col, f + row * OP + col, b.valid - col);
  }
}

// Short K in 16 bits (up to 128), both operands contiguous along K and in whole 16-byte pieces: attention scores.  The 64 x 64 form above is bound
// there by the vector instructions around a tile's few MFMAs, some hundreds in each of eight waves to a SIMD at 32 x 512 x 80 x 512.  Here
// tiles are 128 x 128 (F 2) wherever they give every CU one without much of them past the ends, K's pieces are a constant number and all asked for at once, rows beyond the end are the last one
// again, and the product is formed as B A^T, so that a lane's four sums in a row of registers are four outputs in a row: rounded there, they
// go through LDS and out at half the size.
//   Measured (us, the form above, this): bf16 32 x 512 x 80 x 512 10.7, 7.8, x 64 9.5, 7.5, x 128 11.2, 8.4, x 8 9.6, 6.8; 12 x 1024 x 128 x 1024 15.0, 11.0; 3 x 1024 x
// 104 x 1024 6.4, 5.4; f16 63 x 994 x 24 x 304 18.6, 11.4; 40 random ones of 2 to 64 batches 0.87 of the time in the mean, the smallest 0.85 to 0.99.
template <typename T, int F, int KB>
__global__ void __launch_bounds__(256, F == 2 ? 2 : 4) k_matmul_short(T *out, const T *A, const T *B, MatmulArgs g, int tiles_m, int tiles_n) {
  constexpr int BT = 64 * F, CPR = KB / 16, P = BT * CPR / 256, PITCH = KB + 16, STAGE = BT * PITCH, OP = BT * 2 + 16;
  static_assert(BT * CPR % 256 == 0, "every thread has as many pieces");
  constexpr int LDS = 2 * STAGE > BT * OP ? 2 * STAGE : BT * OP;
  __shared__ __attribute__((aligned(16))) char lds[LDS];
  const int total = gridDim.x, xcd = blockIdx.x & 7, q = total >> 3, rem = total & 7;   // runs of tiles by XCD, as above
  const int t = xcd * q + (xcd < rem ? xcd : rem) + (blockIdx.x >> 3);
  const int z = t / (tiles_m * tiles_n), in = t - z * tiles_m * tiles_n;
  const int m0 = (in % tiles_m) * BT, n0 = (in / tiles_m) * BT;
  int64_t aoff = 0, boff = 0;
  for (int d = g.batch_rank - 1, rest = z; d >= 0; --d) {
    const int n = (int)g.batch_shape[d], i = rest % n;
    rest /= n;
    aoff += i * g.a_bs[d];
    boff += i * g.b_bs[d];
  }
  const int rows = (int)min<int64_t>(BT, g.M - m0), cols = (int)min<int64_t>(BT, g.N - n0), pieces = (int)g.K / 8;
  const T *a = A + aoff + m0 * g.a_rs, *b = B + boff + n0 * g.b_cs;
  mm_chunk ra[P], rb[P];
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const int i = threadIdx.x + 256 * p, c = min(i % CPR, pieces - 1) * 8;
    ra[p] = *reinterpret_cast<const mm_chunk *>(a + min(i / CPR, rows - 1) * g.a_rs + c);
  }
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const int i = threadIdx.x + 256 * p, c = min(i % CPR, pieces - 1) * 8;
    rb[p] = *reinterpret_cast<const mm_chunk *>(b + min(i / CPR, cols - 1) * g.b_cs + c);
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int p = 0; p < P; ++p) {   // (what lies past K is zero in both: either may hold what is no number)
    const int i = threadIdx.x + 256 * p;
    *reinterpret_cast<mm_chunk *>(lds + i / CPR * PITCH + i % CPR * 16) = i % CPR < pieces ? ra[p] : mm_chunk{0u, 0u, 0u, 0u};
  }
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const int i = threadIdx.x + 256 * p;
    *reinterpret_cast<mm_chunk *>(lds + STAGE + i / CPR * PITCH + i % CPR * 16) = i % CPR < pieces ? rb[p] : mm_chunk{0u, 0u, 0u, 0u};
  }
  __syncthreads();
  const int wave = threadIdx.x >> 6, wm = (wave >> 1) * 32 * F, wn = (wave & 1) * 32 * F, r = threadIdx.x & 31, h = (threadIdx.x >> 5) & 1;
  mm_f32x16 acc[F][F];
#pragma unroll
  for (int i = 0; i < F; ++i)
#pragma unroll
    for (int j = 0; j < F; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  const char *fa = lds + (wm + r) * PITCH + h * 16, *fb = lds + STAGE + (wn + r) * PITCH + h * 16;
#pragma unroll
  for (int kk = 0; kk < CPR / 2; ++kk) {
    mm_chunk x[F], y[F];
#pragma unroll
    for (int i = 0; i < F; ++i) {
      x[i] = *reinterpret_cast<const mm_chunk *>(fa + i * 32 * PITCH + kk * 32);
      y[i] = *reinterpret_cast<const mm_chunk *>(fb + i * 32 * PITCH + kk * 32);
    }
#pragma unroll
    for (int i = 0; i < F; ++i)
#pragma unroll
      for (int j = 0; j < F; ++j) acc[i][j] = mm_mfma<T>(y[j], x[i], acc[i][j]);
  }
  __syncthreads();   // the operands have been read
  // accumulator register e of lane (r, h) is row r, column 8 (e / 4) + 4 h + e % 4
#pragma unroll
  for (int i = 0; i < F; ++i)
#pragma unroll
    for (int j = 0; j < F; ++j)
#pragma unroll
      for (int e = 0; e < 16; e += 4) {
        T v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) Scalar<T>::store(&v[u], acc[i][j][e + u]);
        __builtin_memcpy(__builtin_assume_aligned(lds + (wm + 32 * i + r) * OP + (wn + 32 * j + 8 * (e >> 2) + 4 * h) * 2, 8), v, 8);
      }
  __syncthreads();
  T *o = out + (int64_t)z * g.M * g.N + (int64_t)m0 * g.N + n0;
#pragma unroll 4
  for (int i = threadIdx.x; i < BT * BT / 8; i += 256) {
    const int row = i / (BT / 8), col = i % (BT / 8) * 8;
    if (row >= rows || col >= cols) continue;
    const mm_chunk v = *reinterpret_cast<const mm_chunk *>(lds + row * OP + col * 2);
    T *dst = o + (int64_t)row * g.N + col;
    if (col + 8 <= cols) {
      __builtin_memcpy(dst, &v, 16);
    } else {
      T w[8];
      __builtin_memcpy(w, &v, 16);
#pragma unroll
      for (int u = 0; u < 7; ++u)
        if (col + u < cols) dst[u] = w[u];
    }
  }
}

template <typename T, bool AKC, bool BKC>
static int launch_mm(hipStream_t st, void *out, const void *A, const void *B, const MatmulArgs &g, int64_t batch) {
  // 64 x 64 tiles; 16-bit operands take 128 x 128 (half the operand traffic per product) once those give every CU two and K
  // is long enough to pay for the larger prologue (64 x 1024 x 1024 x 1024: 200 to 227 against 290 us; 32 x 512 x 80 x 512:
  // 12.1 against 11.2).  Up to 256 bytes of K a tile needs no second stage: one load phase, and less LDS, so more blocks to
  // a CU (us, two stages of 128 bytes, one of 256, one of 192: bf16 32 x 512 x 80 x 512 14.0, 12.0, 10.9; 32 x 512 x 96 x 512 13.5, 11.3,
  // 10.3; 12 x 333 x 96 x 333 5.7, 5.4, 5.0; 64 x 128 x 80 x 128 4.9, 4.8, 4.6; f32 12 x 333 x 40 x 333 7.3, 6.5, 6.2; two stages and one
  // of 256: bf16 32 x 512 x 128 x 512 13.1, 11.5; f32 32 x 512 x 64 x 512 18.4, 18.8).
  const int64_t t64 = batch * ((g.M + 63) / 64) * ((g.N + 63) / 64), tm128 = (g.M + 127) / 128, tn128 = (g.N + 127) / 128;
  const int kb = (int)(g.K * (int64_t)sizeof(T) < 512 ? g.K * sizeof(T) : 512);
  const int tm = (int)((g.M + 63) / 64), tn = (int)((g.N + 63) / 64);
  auto wide = [&](const void *p, int64_t stride, const int64_t *bs) {
    bool ok = (uintptr_t)p % 16 == 0 && stride % 8 == 0;
    for (int d = 0; d < g.batch_rank; ++d) ok = ok && (bs[d] % 8 == 0 || g.batch_shape[d] == 1);
    return ok;
  };
  const bool aligned = wide(A, g.a_rs, g.a_bs) && wide(B, g.b_cs, g.b_bs);
  auto go = [&](auto kernel, int64_t blocks, int tiles_m, int tiles_n) -> int {
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(256), 0, st, (T *)out, (const T *)A, (const T *)B, g, tiles_m, tiles_n);
    return launch_check("matmul_mfma");
  };
  if constexpr (sizeof(T) == 2 && AKC && BKC) {
    if (g.K <= 128 && g.K % 8 == 0 && aligned) {
      // (tiles half of which lie past an end: 50 x 874 x 40 x 41 5.4 us in the form above, 6.3 by large ones)
      const int64_t t128 = batch * tm128 * tn128;
      const bool large = t128 >= kNumCU && 8 * t128 <= 3 * t64;
      auto with = [&](auto bytes) -> int {
        constexpr int KB = decltype(bytes)::value;
        return large ? go(k_matmul_short<T, 2, KB>, batch * tm128 * tn128, (int)tm128, (int)tn128) : go(k_matmul_short<T, 1, (KB + 63) / 64 * 64>, t64, tm, tn);
      };
      switch ((kb + 31) / 32) {
        case 1: return with(std::integral_constant<int, 32>{});
        case 2: return with(std::integral_constant<int, 64>{});
        case 3: return with(std::integral_constant<int, 96>{});
        case 4: return with(std::integral_constant<int, 128>{});
        case 5: return with(std::integral_constant<int, 160>{});
        case 6: return with(std::integral_constant<int, 192>{});
        case 7: return with(std::integral_constant<int, 224>{});
        default: return with(std::integral_constant<int, 256>{});
      }
    }
  }
  if (kb <= 128) return go(k_matmul_mfma<T, AKC, BKC, 1, 128, true>, t64, tm, tn);
  if (kb <= 192) return go(k_matmul_mfma<T, AKC, BKC, 1, 192, true>, t64, tm, tn);
  if (kb <= 256) return go(k_matmul_mfma<T, AKC, BKC, 1, 256, true>, t64, tm, tn);
  auto stages = [&](auto off) -> int {   // two and more
    constexpr bool OFF = decltype(off)::value;
    if constexpr (sizeof(T) == 2) {
      if (batch * tm128 * tn128 >= 2 * kNumCU && g.K >= 256) return go(k_matmul_mfma<T, AKC, BKC, 2, 128, false, OFF>, batch * tm128 * tn128, (int)tm128, (int)tn128);
    }
    return go(k_matmul_mfma<T, AKC, BKC, 1, 128, false, OFF>, t64, tm, tn);
  };
  if constexpr (sizeof(T) == 2 && AKC && BKC) {
    if (!aligned) return stages(std::integral_constant<bool, true>{});
  }
  return stages(std::integral_constant<bool, false>{});
}

bool matmul_mfma_serves(int dtype, const MatmulArgs &g, int64_t batch) {
  const bool a = g.a_cs == 1 || g.a_rs == 1 || g.K == 1 || g.M == 1, b = g.b_rs == 1 || g.b_cs == 1 || g.K == 1 || g.N == 1;
  return (dtype == RAI_F32 || dtype == RAI_BF16 || dtype == RAI_F16) && a && b && g.K < (1 << 30) && g.M < (1LL << 30) && g.N < (1LL << 30) &&
         batch * ((g.M + 63) / 64) * ((g.N + 63) / 64) < (1LL << 31);
}

int launch_matmul_mfma(hipStream_t st, int dtype, void *out, const void *A, const void *B, const MatmulArgs &g0, int64_t batch) {
  MatmulArgs g = g0;
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
