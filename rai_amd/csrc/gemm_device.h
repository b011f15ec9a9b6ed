// What the bf16 tile kernels (gemm_mfma.hip, gemm_persist.hip) share: tile order, activations of bf16 outputs, the
// shares of stream-K.
#pragma once
#include <type_traits>

#include "gemm.h"

namespace rai {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
typedef __attribute__((ext_vector_type(4))) float f32x4;

constexpr int kXcds = 8;

// Tile order inside an XCD's run: bands of kGroupM tile rows swept across all tile columns, so the
// ~100 tiles that are resident on an XCD at any moment form a block of about kGroupM x 12 tiles and
// share their A and B panels through that XCD's L2 (a column-by-column order re-reads all of A from
// memory for every tile column).
constexpr int kGroupM = 8;
__device__ __forceinline__ void tile_coords(int tile, int tiles_m, int tiles_n, int *tile_m, int *tile_n) {
  const int band = tile / (kGroupM * tiles_n);
  const int first_m = band * kGroupM;
  const int height = tiles_m - first_m < kGroupM ? tiles_m - first_m : kGroupM;
  const int in_band = tile - band * kGroupM * tiles_n;
  *tile_m = first_m + in_band % height;
  *tile_n = in_band / height;
}

__device__ __forceinline__ int xcd_remap(int bid, int total) {
  // blocks bid, bid+8, bid+16, ... run on the same XCD; give them consecutive tiles
  const int per = (total + kXcds - 1) / kXcds;
  return (bid % kXcds) * per + bid / kXcds;
}

// Applies activation `act` to the elements of x[8] whose column n + e is >= from.  The switch on the
// (block-uniform) activation sits outside the element loop, so only one activation's code runs.
// The results are rounded to bf16 (relative step 2^-8), so tanh-GELU and SiLU are evaluated through the hardware
// exponential and reciprocal (relative error ~1e-6) instead of the library tanhf / expf and a division:
// 0.5 x (1 + tanh u) = x / (1 + exp(-2u)).  The f32 Linear keeps the library functions (act_eval).
__device__ __forceinline__ float act_eval_bf16_out(int act, float x) {
  if (act == RAI_UN_NEW_GELU) {
    const float u = 0.7978845608028654f * (x + 0.044715f * x * x * x);
    return x * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-2.0f * 1.4426950408889634f * u));
  }
  if (act == RAI_UN_SILU) return x * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * x));
  return act_eval(act, x);
}
template <int N>
__device__ __forceinline__ void act_n(int act, float (&x)[N], int n, int from) {
#define RAI_ACT_CASE(K)                                     \
  case K:                                                   \
    _Pragma("unroll") for (int e = 0; e < N; ++e)           \
      if (n + e >= from) x[e] = act_eval_bf16_out(K, x[e]); \
    break;
  switch (act) {
    RAI_ACT_CASE(RAI_UN_GELU)
    RAI_ACT_CASE(RAI_UN_NEW_GELU)
    RAI_ACT_CASE(RAI_UN_SILU)
    RAI_ACT_CASE(RAI_UN_RELU)
    RAI_ACT_CASE(RAI_UN_TANH)
    default: break;
  }
#undef RAI_ACT_CASE
}
__device__ __forceinline__ void act8(int act, float (&x)[8], int n, int from) { act_n<8>(act, x, n, from); }
// The same by the library's functions.
template <int N>
__device__ __forceinline__ void act_exact(int act, float (&x)[N], int n, int from) {
#define RAI_ACT_CASE(K)                            \
  case K:                                          \
    _Pragma("unroll") for (int e = 0; e < N; ++e)  \
      if (n + e >= from) x[e] = act_eval(K, x[e]); \
    break;
  switch (act) {
    RAI_ACT_CASE(RAI_UN_GELU)
    RAI_ACT_CASE(RAI_UN_NEW_GELU)
    RAI_ACT_CASE(RAI_UN_SILU)
    RAI_ACT_CASE(RAI_UN_RELU)
    RAI_ACT_CASE(RAI_UN_TANH)
    default: break;
  }
#undef RAI_ACT_CASE
}
__device__ __forceinline__ void unpack8(const u32x4 &p, float (&f)[8]) {
#pragma unroll
  for (int e = 0; e < 8; ++e) f[e] = bf16_bits_to_f32((uint16_t)(p[e >> 1] >> (16 * (e & 1))));
}

// Whether a row's 8 columns can be stored, and a residual's read, as one 16-byte word each.
__host__ __device__ __forceinline__ bool rows_store_16(const LinearArgs &a) {
  return (a.ld1 % 8 == 0) && (a.n_split % 8 == 0) && (a.n_split == a.N || a.ld2 % 8 == 0) && ((uintptr_t)a.out1 % 16 == 0) &&
         (a.n_split == a.N || (uintptr_t)a.out2 % 16 == 0) && (!a.residual || (a.ldr % 8 == 0 && (uintptr_t)a.residual % 16 == 0)) && a.N % 8 == 0;
}
// The summed biases of columns n .. n + 7 (zero beyond N).
__device__ __forceinline__ void load_bias8(const LinearArgs &a, int n, float (&bv)[8]) {
  const bool whole = n + 8 <= a.N;
#pragma unroll
  for (int e = 0; e < 8; ++e) bv[e] = 0.f;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const uint16_t *bias = (const uint16_t *)(i ? a.bias2 : a.bias);
    if (!bias || n >= a.N) continue;
    float b[8];
    if (whole && ((uintptr_t)(bias + n) & 15) == 0) unpack8(*reinterpret_cast<const u32x4 *>(bias + n), b);
    else {
#pragma unroll
      for (int e = 0; e < 8; ++e) b[e] = n + e < a.N ? bf16_bits_to_f32(bias[n + e]) : 0.f;
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) bv[e] = i ? bv[e] + b[e] : b[e];
  }
}
// Bias, activation, residual and store of columns n .. n + 7 of row m (both inside the output; whole: n + 8 <= N).  The sums come as
// values: eight floats by reference stay apart from the activation's own, which then copies them there and back (64 x 64 tiles: 160
// moves more; with gelu 67 x 5592 x 832 9.11 us, so 8.99, 68 x 256 x 256 7.20, 6.97).
__device__ __forceinline__ void store_row8(const LinearArgs &a, const f32x4 v0, const f32x4 v1, const float (&bv)[8], int m, int n, bool whole, bool vec_out) {
  float v[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
  const uint16_t *res = (const uint16_t *)a.residual;
  if (a.glu) {  // columns n..n+7 are four (gate, up) pairs -> four outputs at column n/2
    uint16_t *dst = (uint16_t *)a.out1 + (int64_t)m * a.ld1 + (n >> 1);
    float gr[8], ga[4], gl[4];
    if (a.act == kActClampedGlu) {
#pragma unroll
      for (int e = 0; e < 4; ++e) gl[e] = glu_clamped_bf16_out(v[2 * e] + bv[2 * e], v[2 * e + 1] + bv[2 * e + 1], a.act_limit, a.act_alpha);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) gr[e] = bf16_bits_to_f32(f32_to_bf16_bits(v[e] + bv[e]));  // gate / up rounded to bf16 as the reference does
#pragma unroll
      for (int e = 0; e < 4; ++e) ga[e] = gr[2 * e];
      act_n<4>(a.act, ga, 0, 0);   // the four gates
#pragma unroll
      for (int e = 0; e < 4; ++e) gl[e] = bf16_bits_to_f32(f32_to_bf16_bits(ga[e])) * gr[2 * e + 1];
    }
    if (whole && a.ld1 % 4 == 0 && (uintptr_t)a.out1 % 8 == 0) {
      typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;
      u32x2 o = {pack_bf16x2(gl[0], gl[1]), pack_bf16x2(gl[2], gl[3])};
      *reinterpret_cast<u32x2 *>(dst) = o;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (n + 2 * e + 1 < a.N) dst[e] = f32_to_bf16_bits(gl[e]);
    }
    return;
  }
  // compile-time element indices throughout: a loop bounded by a run-time count would index v[]
  // dynamically, which the compiler lowers to a chain of selects per access
  const int lim = a.N - n < 8 ? a.N - n : 8;
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] += bv[e];
  if (a.act >= 0) act8(a.act, v, n, a.act_from);
  if (a.f32_out) {
    float *dst = (float *)a.out1 + (int64_t)m * a.ld1 + n;
    const float *rsrc = res ? (const float *)a.residual + (int64_t)m * a.ldr + n : nullptr;
    if (whole && a.ld1 % 4 == 0 && (!res || a.ldr % 4 == 0) && (((uintptr_t)a.out1 | (uintptr_t)a.residual) & 15) == 0) {
      f32x4 r0 = {0.f, 0.f, 0.f, 0.f}, r1 = r0;
      if (rsrc) {
        r0 = *reinterpret_cast<const f32x4 *>(rsrc);
        r1 = *reinterpret_cast<const f32x4 *>(rsrc + 4);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        r0[e] = fmaf(a.out_scale, v[e], r0[e]);
        r1[e] = fmaf(a.out_scale, v[4 + e], r1[e]);
      }
      *reinterpret_cast<f32x4 *>(dst) = r0;
      *reinterpret_cast<f32x4 *>(dst + 4) = r1;
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (e < lim) dst[e] = fmaf(a.out_scale, v[e], rsrc ? rsrc[e] : 0.f);
    }
    return;
  }
  if (res) {
    if (vec_out) {
      float rv[8];
      unpack8(*reinterpret_cast<const u32x4 *>(res + (int64_t)m * a.ldr + n), rv);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] += rv[e];
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (e < lim) v[e] += bf16_bits_to_f32(res[(int64_t)m * a.ldr + n + e]);
    }
  }
  if (vec_out) {
    const u32x4 o = {pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7])};
    uint16_t *dst = n < a.n_split ? (uint16_t *)a.out1 + (int64_t)m * a.ld1 + n
                                  : (uint16_t *)a.out2 + (int64_t)m * a.ld2 + (n - a.n_split);
    *reinterpret_cast<u32x4 *>(dst) = o;
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      if (e < lim) {
        const int nn = n + e;
        if (nn < a.n_split) ((uint16_t *)a.out1)[(int64_t)m * a.ld1 + nn] = f32_to_bf16_bits(v[e]);
        else ((uint16_t *)a.out2)[(int64_t)m * a.ld2 + (nn - a.n_split)] = f32_to_bf16_bits(v[e]);
      }
    }
  }
}

// 16 bytes to or from memory past the (per-XCD, mutually incoherent) L2s: for data that another block of the same
// launch reads or wrote (p is 16-byte aligned)
__device__ __forceinline__ void store_f32x4_device(float *p, f32x4 v) {
  unsigned long long *q = reinterpret_cast<unsigned long long *>(p);
  __hip_atomic_store(q, (unsigned long long)__float_as_uint(v.x) | ((unsigned long long)__float_as_uint(v.y) << 32), __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(q + 1, (unsigned long long)__float_as_uint(v.z) | ((unsigned long long)__float_as_uint(v.w) << 32), __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ f32x4 load_f32x4_device(const float *p) {
  const unsigned long long *q = reinterpret_cast<const unsigned long long *>(p);
  const unsigned long long lo = __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const unsigned long long hi = __hip_atomic_load(q + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return f32x4{__uint_as_float((uint32_t)lo), __uint_as_float((uint32_t)(lo >> 32)), __uint_as_float((uint32_t)hi),
               __uint_as_float((uint32_t)(hi >> 32))};
}

struct StreamKArgs {
  int sk_tiles;   // tiles 0 .. sk_tiles-1 are shared out by K tile; the rest run whole
  int q, rem;     // units per block: blocks 0 .. rem-1 take q + 1, the others q
  int max_parts;  // slots per tile in the workspace
  float *ws;      // [sk_tiles][max_parts][BM * BN] f32
  int *counters;  // [sk_tiles][2] (tickets, stored shares), zero between launches
  int *fault;     // host-visible word: RAI_FAULT_STREAMK is stored here when a wait for shares expires
  int spin_limit; // polls of the stored-shares counter before the wait is given up
  int drop_tile;  // test hook: the stored shares of this tile are never counted (-1: none), so its wait must expire
};

__device__ __forceinline__ int sk_start(const StreamKArgs &k, int p) { return p * k.q + (p < k.rem ? p : k.rem); }
__device__ __forceinline__ int sk_block_of(const StreamKArgs &k, int u) {
  const int big = k.rem * (k.q + 1);
  return u < big ? u / (k.q + 1) : k.rem + (u - big) / k.q;
}

// A tile that two or three blocks share; acc is this wave's part of block p's share.  Slot layout [wave][accumulator register][lane]: one
// store or load instruction covers 256 consecutive bytes.  The shares cross XCDs, whose L2s are not coherent with each other: they
// are written and read with device-scope accesses (write-through stores, loads that miss L2) instead of a release /
// acquire fence pair, which would write back and invalidate a whole L2 each and, issued by every block of an XCD at about
// the same time, queue up behind one another (measured: +130 us per launch).
// Two counters per tile: `arrived` hands out tickets when a share has been computed, `stored` counts the shares that have
// reached memory.  The block with the last ticket keeps its share in registers and sums, in slot order, so that the result
// does not depend on who was last; the others store theirs.  Its wait is for blocks that already hold a ticket, i.e. are
// running and have nothing left to do but their stores, and it is bounded all the same.  True: this block writes the tile.
// `ticket` is a word of LDS that may hold something else before and after.
template <typename V, int MT, int NT>
__device__ __forceinline__ bool sum_shares(const StreamKArgs &sk, V (&acc)[MT][NT], int *ticket, int tile, int stages, int p, int wave, int lane) {
  constexpr int R = sizeof(V) / sizeof(float), TILE = 256 * 256;
  const int first = sk_block_of(sk, tile * stages), last = sk_block_of(sk, tile * stages + stages - 1);
  const int parts = last - first + 1, slot = p - first;
  float *tile_ws = sk.ws + (int64_t)tile * sk.max_parts * TILE + wave * (MT * NT * R * 64) + lane;
  int *arrived = sk.counters + 2 * tile, *stored = arrived + 1;
  __syncthreads();   // the LDS that holds the ticket is free
  if (threadIdx.x == 0) *ticket = __hip_atomic_fetch_add(arrived, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  if (*ticket != parts - 1) {
    float *mine = tile_ws + (int64_t)slot * TILE;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int r = 0; r < R; ++r)
          __hip_atomic_store(mine + ((i * NT + j) * R + r) * 64, acc[i][j][r], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this wave's share has left for memory
    __syncthreads();
    if (threadIdx.x == 0 && tile != sk.drop_tile) __hip_atomic_fetch_add(stored, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return false;
  }
  __syncthreads();   // every wave has read the ticket
  if (threadIdx.x == 0) {
    bool complete = false;
    for (int spin = 0; spin < sk.spin_limit && !complete; ++spin) {
      complete = __hip_atomic_load(stored, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == parts - 1;
      if (!complete) __builtin_amdgcn_s_sleep(2);
    }
    if (complete) {
      __hip_atomic_store(arrived, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(stored, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else {
      // A share is missing.  Nothing is summed and nothing written for this tile, the counters stay as they are (a late
      // block may still count itself in; the host zeroes them all before the next launch), and the host learns of it at
      // its next synchronisation.
      __hip_atomic_store(sk.fault, (int)RAI_FAULT_STREAMK, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    *ticket = complete;
  }
  __syncthreads();
  const bool complete = *ticket != 0;
  __syncthreads();   // before the ticket's LDS is written
  if (!complete) return false;
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      V sum = acc[i][j];
      for (int s = 0; s < parts; ++s) {
        if (s == slot) {
          if (s > 0) {
#pragma unroll
            for (int r = 0; r < R; ++r) sum[r] += acc[i][j][r];
          }
          continue;
        }
        const float *src = tile_ws + (int64_t)s * TILE + ((i * NT + j) * R) * 64;
        V v;
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = __hip_atomic_load(src + r * 64, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (s == 0) sum = v;
        else {
#pragma unroll
          for (int r = 0; r < R; ++r) sum[r] += v[r];
        }
      }
      acc[i][j] = sum;
    }
  return true;
}

// The 256 x 256 tiles of a product on one block per CU, the next tile's loads under way while the last one's outputs are
// written (gemm_persist.hip); sk: which of them are shared out by K tile (sk_tiles == 0: none).
// It addresses the rows of a tile by 32-bit offsets: of bytes in the operands, 256 rows, and of elements in the outputs, 16 rows.
inline bool gemm_persist_serves(const LinearArgs &a) { return a.lda < (1 << 22) && a.ldw < (1 << 22) && a.ld1 < (1 << 28) && a.ld2 < (1 << 28); }
// What its fast way out needs of the product as a whole (a wave has 64 columns of a tile).
constexpr int kPersistColumns = 64;
inline bool gemm_persist_plain(const LinearArgs &a) {
  return rows_store_16(a) && !a.f32_out && !a.bias2 && !(a.residual && (a.bias || a.act >= 0)) && ((uintptr_t)a.bias & 3) == 0 &&
         (a.n_split == a.N || a.n_split % kPersistColumns == 0) && a.act_from % kPersistColumns == 0 && (!a.glu || (a.N % 16 == 0 && a.act != kActClampedGlu));
}
int launch_gemm_bf16_persist(hipStream_t st, const LinearArgs &a, const StreamKArgs &sk);

// The arrival counters of a device's K splits, zero between launches (null: device unknown).
constexpr int kSplitTickets = 16384;
int *splitk_tickets(const LinearArgs &a);

}  // namespace rai
