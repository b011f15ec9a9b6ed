// Internal helpers shared by the HIP translation units of librai_hip.so.
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>

#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <type_traits>

#include "rai_hip.h"

namespace rai {

// ---------------------------------------------------------------- errors
void set_error(const char *fmt, ...);
int fail(int code, const char *fmt, ...);

#define RAI_HIP_TRY(expr)                                                                     \
  do {                                                                                        \
    hipError_t _e = (expr);                                                                   \
    if (_e != hipSuccess)                                                                     \
      return ::rai::fail(RAI_ERR_HIP, "%s:%d %s -> %s", __FILE__, __LINE__, #expr,            \
                         hipGetErrorString(_e));                                              \
  } while (0)

#define RAI_TRY(expr)        \
  do {                       \
    int _s = (expr);         \
    if (_s != RAI_OK) return _s; \
  } while (0)

#define RAI_REQUIRE(cond, code, ...)                  \
  do {                                                \
    if (!(cond)) return ::rai::fail(code, __VA_ARGS__); \
  } while (0)

// ---------------------------------------------------------------- device ctx
struct DeviceCtx;
// Returns nullptr (and sets the error) when dev is out of range or init fails.
DeviceCtx *ctx(int dev);
hipStream_t stream_of(int dev);
// The stream of an already initialised device; never creates a context (no allocation): nullptr + error otherwise.
hipStream_t stream_if_ready(int dev);
// Compute units of the device, asked of it once when its context is created (0 when the device cannot be set up).
int device_cu_count(int dev);
// Kernels that wait for other blocks bound their wait; one that gives up stores a RAI_FAULT_* code (system scope) to
// this word, which lives in pinned host memory, and every wave still exits normally.  The host looks at the word after
// each synchronisation of the device's stream (rai_hip_sync, rai_hip_d2h, the decoder's generate) and turns a
// non-zero code into RAI_ERR_HIP, clears it and resets the counters those kernels share.
int *kernel_fault_word(int dev);
int check_kernel_fault(int dev);
enum { RAI_FAULT_STREAMK = 1, RAI_FAULT_CHAIN = 2 };
// Zeroes the stream-K tile kernel's arrival counters on `st` (gemm_mfma.hip).
int streamk_counters_reset(int dev, hipStream_t st);
// Looks up this device's address of the fixed scratch array of the allocation-free argmax (reduce.hip); called once
// per device, with that device current, while its context is created.
int arg_static_scratch_init(int dev);
// The device's scratch block, which lives as long as the device context (grown on demand, never shrinks), for kernels
// that need partial results.  A call keeps its hold on the block until it has enqueued the last kernel or copy that uses
// it: another thread's work then comes behind it on the device's one stream, and nobody replaces the block between the
// call's launches.  (Without the hold two threads' kernels could be enqueued in turn and read each other's partial sums.)
// A thread holds it once at a time.
struct WorkspaceHold {
  std::unique_lock<std::mutex> lock;
};
int workspace(int dev, size_t bytes, void **out, WorkspaceHold *hold);
// The same for work that can do with less: up to `bytes` of the block, as many as it has where it cannot grow.  Returns
// how many.
size_t workspace_if_room(int dev, size_t bytes, void **out, WorkspaceHold *hold);
// Device counter bumped by gather kernels on an out-of-range index.
unsigned long long *index_error_counter(int dev);
int launch_check(const char *what);

// ---------------------------------------------------------------- dtypes
inline size_t dtype_size(int dt) {
  switch (dt) {
    case RAI_U8: return 1;
    case RAI_U32: return 4;
    case RAI_I64: return 8;
    case RAI_F16: return 2;
    case RAI_BF16: return 2;
    case RAI_F32: return 4;
    case RAI_F64: return 8;
    default: return 0;
  }
}
inline bool is_float(int dt) { return dt == RAI_F16 || dt == RAI_BF16 || dt == RAI_F32 || dt == RAI_F64; }
inline const char *dtype_name(int dt) {
  static const char *n[] = {"u8", "u32", "i64", "f16", "bf16", "f32", "f64"};
  return (dt >= 0 && dt <= 6) ? n[dt] : "?";
}

inline int64_t numel(const rai_hip_tensor *t) {
  int64_t n = 1;
  for (int i = 0; i < t->rank; ++i) n *= t->shape[i];
  return n;
}
inline bool is_contiguous(const rai_hip_tensor *t) {
  int64_t expect = 1;
  for (int i = t->rank - 1; i >= 0; --i) {
    if (t->shape[i] == 1) continue;
    if (t->stride[i] != expect) return false;
    expect *= t->shape[i];
  }
  return true;
}
inline bool same_shape(const rai_hip_tensor *a, const rai_hip_tensor *b) {
  if (a->rank != b->rank) return false;
  for (int i = 0; i < a->rank; ++i)
    if (a->shape[i] != b->shape[i]) return false;
  return true;
}
int validate(const rai_hip_tensor *t, const char *name);
inline char *base_ptr(const rai_hip_tensor *t) {
  return static_cast<char *>(t->data) + t->offset * (int64_t)dtype_size(t->dtype);
}

// A tensor view with dims merged where strides allow, for index decomposition on
// the device.  Up to three operands share one iteration space.
struct StridedArgs {
  int rank;
  int64_t shape[RAI_HIP_MAX_RANK];
  int64_t stride[3][RAI_HIP_MAX_RANK];
};
// Collapses the common iteration space of n (<=3) same-shape views.
void coalesce(int n, const rai_hip_tensor *const *ts, StridedArgs *out);

// ---------------------------------------------------------------- device-side scalar conversion
typedef __hip_bfloat16 bf16_t;
typedef __half f16_t;

__device__ __forceinline__ float bf16_bits_to_f32(uint16_t b) { return __uint_as_float(((uint32_t)b) << 16); }
// round-to-nearest-even through the gfx950 conversion instruction (v_cvt_pk_bf16_f32)
__device__ __forceinline__ uint16_t f32_to_bf16_bits(float f) {
  return __builtin_bit_cast(uint16_t, (__bf16)f);
}
// two floats -> packed bf16 pair (lo in bits 0..15)
__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
  typedef __attribute__((ext_vector_type(2))) float f32x2_t;
  typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_t;
  f32x2_t v = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
}

template <typename T> struct Scalar;  // load/store through a compute type
template <> struct Scalar<float> {
  typedef float compute;
  static __device__ __forceinline__ float load(const float *p) { return *p; }
  static __device__ __forceinline__ void store(float *p, float v) { *p = v; }
};
template <> struct Scalar<double> {
  typedef double compute;
  static __device__ __forceinline__ double load(const double *p) { return *p; }
  static __device__ __forceinline__ void store(double *p, double v) { *p = v; }
};
struct bf16_raw { uint16_t bits; };
struct f16_raw { uint16_t bits; };
template <> struct Scalar<bf16_raw> {
  typedef float compute;
  static __device__ __forceinline__ float load(const bf16_raw *p) { return bf16_bits_to_f32(p->bits); }
  static __device__ __forceinline__ void store(bf16_raw *p, float v) { p->bits = f32_to_bf16_bits(v); }
};
template <> struct Scalar<f16_raw> {
  typedef float compute;
  static __device__ __forceinline__ float load(const f16_raw *p) {
    return __half2float(__ushort_as_half(p->bits));
  }
  static __device__ __forceinline__ void store(f16_raw *p, float v) {
    p->bits = __half_as_ushort(__float2half_rn(v));
  }
};
template <> struct Scalar<uint8_t> {
  typedef uint8_t compute;
  static __device__ __forceinline__ uint8_t load(const uint8_t *p) { return *p; }
  static __device__ __forceinline__ void store(uint8_t *p, uint8_t v) { *p = v; }
};
template <> struct Scalar<uint32_t> {
  typedef uint32_t compute;
  static __device__ __forceinline__ uint32_t load(const uint32_t *p) { return *p; }
  static __device__ __forceinline__ void store(uint32_t *p, uint32_t v) { *p = v; }
};
template <> struct Scalar<int64_t> {
  typedef int64_t compute;
  static __device__ __forceinline__ int64_t load(const int64_t *p) { return *p; }
  static __device__ __forceinline__ void store(int64_t *p, int64_t v) { *p = v; }
};

// Calls f(T{}) with the storage type matching a runtime dtype.
#define RAI_DISPATCH_ALL(dt, T, ...)                         \
  switch (dt) {                                              \
    case RAI_U8: { typedef uint8_t T; __VA_ARGS__; break; }   \
    case RAI_U32: { typedef uint32_t T; __VA_ARGS__; break; } \
    case RAI_I64: { typedef int64_t T; __VA_ARGS__; break; }  \
    case RAI_F16: { typedef ::rai::f16_raw T; __VA_ARGS__; break; }  \
    case RAI_BF16: { typedef ::rai::bf16_raw T; __VA_ARGS__; break; } \
    case RAI_F32: { typedef float T; __VA_ARGS__; break; }    \
    case RAI_F64: { typedef double T; __VA_ARGS__; break; }   \
    default: return ::rai::fail(RAI_ERR_BAD_DTYPE, "bad dtype %d", (int)(dt)); \
  }
#define RAI_DISPATCH_FLOAT(dt, T, ...)                       \
  switch (dt) {                                              \
    case RAI_F16: { typedef ::rai::f16_raw T; __VA_ARGS__; break; }  \
    case RAI_BF16: { typedef ::rai::bf16_raw T; __VA_ARGS__; break; } \
    case RAI_F32: { typedef float T; __VA_ARGS__; break; }    \
    case RAI_F64: { typedef double T; __VA_ARGS__; break; }   \
    default: return ::rai::fail(RAI_ERR_BAD_DTYPE, "float dtype required, got %s", ::rai::dtype_name(dt)); \
  }

// ---------------------------------------------------------------- wave helpers (wave64)
// op(v of lane l, v of lane l ^ 8), then ^ 4, 2, 1, in every lane, by DPP: over the 16 lanes of a row.
template <typename Op> __device__ __forceinline__ float row_fold(float v, Op op) {
  const auto dpp = [](int old, float x, auto ctrl, auto banks) { return __builtin_amdgcn_update_dpp(old, __float_as_int(x), decltype(ctrl)::value, 0xf, decltype(banks)::value, false); };
  using std::integral_constant;
  typedef integral_constant<int, 0xf> all;
  v = op(v, __int_as_float(dpp(0, v, integral_constant<int, 0x128>{}, all{})));   // row_ror:8
  int four = dpp(0, v, integral_constant<int, 0x104>{}, integral_constant<int, 0x5>{});   // row_shl:4 into lanes 0-3, 8-11 of a row
  four = dpp(four, v, integral_constant<int, 0x114>{}, integral_constant<int, 0xa>{});    // row_shr:4 into the others
  v = op(v, __int_as_float(four));
  v = op(v, __int_as_float(dpp(0, v, integral_constant<int, 0x4e>{}, all{})));   // quad_perm [2, 3, 0, 1]
  return op(v, __int_as_float(dpp(0, v, integral_constant<int, 0xb1>{}, all{})));   // quad_perm [1, 0, 3, 2]
}
__device__ __forceinline__ float row_sum(float v) { return row_fold(v, [](float a, float b) { return a + b; }); }
// ^ 32 and ^ 16 before that: swaps of half and quarter waves.  Some twenty vector instructions in all, where each of the six __shfl_xor
// is a trip through the LDS pipeline (bits as with those).
template <typename Op> __device__ __forceinline__ float wave_fold(float v, Op op) {
  typedef __attribute__((ext_vector_type(2))) unsigned pair;
  auto swap32 = [](float x) { return __builtin_bit_cast(pair, __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false)); };
  auto swap16 = [](float x) { return __builtin_bit_cast(pair, __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false)); };
  pair p = swap32(v);
  v = op(__uint_as_float(p.x), __uint_as_float(p.y));
  p = swap16(v);
  return row_fold(op(__uint_as_float(p.x), __uint_as_float(p.y)), op);
}
__device__ __forceinline__ float wave_sum(float v) { return wave_fold(v, [](float a, float b) { return a + b; }); }
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
__device__ __forceinline__ float wave_max(float v) { return wave_fold(v, [](float a, float b) { return fmaxf(a, b); }); }

constexpr int kWave = 64;
constexpr int kNumCU = 256;

// A grid of at least `blocks` blocks: HIP launches no dimension of 2^32 threads or more, so blocks beyond 2^31 threads go to a second
// one.  A kernel's block is blockIdx.y * gridDim.x + blockIdx.x (blocks go to the XCDs in that order, as gridDim.x is a multiple
// of 8 there), and those past the last one leave.
inline int grid_of_blocks(int64_t blocks, int threads, dim3 *grid) {
  const int64_t most = (1ll << 31) / threads / 8 * 8, x = blocks < most ? blocks : most, y = (blocks + x - 1) / x;
  RAI_REQUIRE(y <= 65535, RAI_ERR_UNSUPPORTED, "%lld blocks in one launch", (long long)blocks);
  *grid = dim3((unsigned)x, (unsigned)y);
  return RAI_OK;
}

}  // namespace rai
