// Scaled-dot-product attention.
//   k_attn_row: one 256-thread block per (query row, head, batch).  K and V of the
//   head are streamed once per block with 16-byte loads; scores live in LDS as
//   f32.  This is the decode kernel (S == 1: HBM-bound on the KV cache) and the
//   dtype-generic fallback for short prefills.
//
// Reference semantics: rai-models/src/llm/phi2.rs:244-262 (f32 scores, -inf mask,
// f32 softmax, P cast to V's dtype), qwen2.rs:205-221 and gemma.rs:238-254
// (scores, scale and softmax rounded to the model dtype), repeat_kv
// gemma.rs:191-201 (query head h reads kv head h / (Hq/Hkv)).
#include <cstdlib>
#include <type_traits>

#include "attention.h"

namespace rai {

template <typename T> struct AttnVec;
template <> struct AttnVec<float> { static constexpr int V = 4; };
template <> struct AttnVec<bf16_raw> { static constexpr int V = 8; };
template <> struct AttnVec<f16_raw> { static constexpr int V = 8; };
template <typename T, int V> struct alignas(sizeof(T) * V) APack { T v[V]; };

template <typename T> __device__ __forceinline__ float round_to(float x) {
  T t;
  Scalar<T>::store(&t, x);
  return (float)Scalar<T>::load(&t);
}
template <> __device__ __forceinline__ float round_to<float>(float x) { return x; }

__device__ __forceinline__ float gate_sigmoid(float z) { return 1.0f / (1.0f + expf(-z)); }
__device__ __forceinline__ float cap_score(float s, float cap) { return cap > 0.f ? cap * tanhf(s / cap) : s; }
template <typename T> __device__ __forceinline__ float sink_of(const void *sink, int h) {
  return sink ? (float)Scalar<T>::load((const T *)sink + h) : -INFINITY;
}

template <typename T>
__global__ void __launch_bounds__(256) k_attn_row(AttnArgs a) {
  constexpr int V = AttnVec<T>::V;
  extern __shared__ __attribute__((aligned(16))) float smem[];
  // layout: q[D] | red[groups*D] | scores[T]
  const int D = a.D, ncol = D / V;
  const int groups = 256 / ncol;
  float *qf = smem;
  float *red = qf + D;
  float *scores = red + groups * D;
  __shared__ float sh[8];

  const int s = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int hk = h / (a.Hq / a.Hkv);
  int n_keys = a.T;
  if (a.t_dev) {
    n_keys = *a.t_dev + a.t_add;
    if (n_keys > a.T) n_keys = a.T;
  }
  int t_end = a.causal ? (n_keys - a.S + s + 1) : n_keys;
  if (t_end > n_keys) t_end = n_keys;
  if (t_end < 0) t_end = 0;
  const int t_begin = a.window > 0 && t_end > a.window ? t_end - a.window : 0;   // oldest key of the sliding window

  const T *q = (const T *)a.q + b * a.qs[0] + h * a.qs[1] + s * a.qs[2];
  const T *K = (const T *)a.k + b * a.ks[0] + hk * a.ks[1];
  const T *Vp = (const T *)a.v + b * a.vs[0] + hk * a.vs[1];
  for (int d = tid; d < D; d += 256) qf[d] = (float)Scalar<T>::load(q + d);
  __syncthreads();

  // A pass over the keys is a chain of trips to memory, so U rows of each group are on their way together, every load whole (past the
  // last key, that one again): a load under a mask is waited for where the mask ends.  Measured (us, one row of a group at a time before):
  // 2 x 32 heads x 4 x 256 on 689 keys in bf16 74 -> 31, 8 x 15 x 128 on 1500 84 -> 34, 8 x 32 x 12 x 64 on 64 14.6 -> 12.9, f32 32 x 2 x 128 on 900
  // 78 -> 26; eight rows: 31.5, 34, 16.8, 25.
  // kAll: every group has U keys; kSome: some have; kFew: none has, and what no group needs is not asked for.
  constexpr int U = 4;
  enum { kAll, kSome, kFew };
  // ---- scores: 16 lanes cooperate on one key row
  {
    const int g = tid >> 4, gl = tid & 15;
    auto round = [&](int base, auto keys) __attribute__((always_inline)) {
      float acc[U];
#pragma unroll
      for (int u = 0; u < U; ++u) acc[u] = 0.f;
      for (int c0 = 0; c0 < ncol; c0 += 16) {
        const int c = min(c0 + gl, ncol - 1);
        APack<T, V> pk[U];
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (keys() != kFew || base + 16 * u < t_end)
            pk[u] = *reinterpret_cast<const APack<T, V> *>(K + (int64_t)(keys() == kAll ? base + g + 16 * u : min(base + g + 16 * u, t_end - 1)) * a.ks[2] + c * V);
        const bool mine = c0 + gl < ncol;
        float qv[V];
#pragma unroll
        for (int j = 0; j < V; ++j) qv[j] = qf[c * V + j];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          if (keys() == kFew && base + 16 * u >= t_end) break;
          float sum = acc[u];
#pragma unroll
          for (int j = 0; j < V; ++j) sum = fmaf(qv[j], (float)Scalar<T>::load(&pk[u].v[j]), sum);
          acc[u] = mine ? sum : acc[u];
        }
      }
      float sum = 0.f;   // lane gl finishes the group's key gl
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (keys() == kFew && base + 16 * u >= t_end) break;
        const float all = row_sum(acc[u]);
        sum = gl == u ? all : sum;
      }
      const int t = base + g + 16 * gl;
      if (gl < U && (keys() == kAll || t < t_end)) {
        float sc;
        if (a.f32_scores) sc = cap_score(sum * a.scale, a.softcap);
        else sc = round_to<T>(round_to<T>(sum) * round_to<T>(a.scale));
        scores[t - t_begin] = sc;
      }
    };
    int base = t_begin;
    for (; base + 16 * U <= t_end; base += 16 * U) round(base, std::integral_constant<int, kAll>());
    if (base + 16 * (U - 1) < t_end) round(base, std::integral_constant<int, kSome>());
    else if (base < t_end) round(base, std::integral_constant<int, kFew>());
  }
  __syncthreads();

  // ---- softmax over the scores of keys [t_begin, t_end)
  const int n_seen = t_end - t_begin;
  const float sink = sink_of<T>(a.sink, h);
  float m = -INFINITY;
  for (int t = tid; t < n_seen; t += 256) m = fmaxf(m, scores[t]);
  m = wave_max(m);
  if (lane == 0) sh[wave] = m;
  __syncthreads();
  m = fmaxf(fmaxf(fmaxf(sh[0], sh[1]), fmaxf(sh[2], sh[3])), sink);
  float sum = 0.f;
  for (int t = tid; t < n_seen; t += 256) {
    float e = expf(scores[t] - m);
    if (!a.f32_scores) e = round_to<T>(e);
    scores[t] = e;
    sum += e;
  }
  sum = wave_sum(sum);
  if (lane == 0) sh[4 + wave] = sum;
  __syncthreads();
  sum = sh[4] + sh[5] + sh[6] + sh[7];
  if (a.sink) sum += expf(sink - m);
  if (!a.f32_scores) sum = round_to<T>(sum);
  const float inv = 1.0f / sum;

  // ---- P.V: thread (grp, col) accumulates keys grp, grp+groups, ... for V
  //      consecutive output features
  {
    const int col = tid % ncol, grp = tid / ncol;
    float acc[V];
#pragma unroll
    for (int j = 0; j < V; ++j) acc[j] = 0.f;
    auto round = [&](int base, auto keys) __attribute__((always_inline)) {
      APack<T, V> pk[U];
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (keys() != kFew || base + groups * u < n_seen)
          pk[u] = *reinterpret_cast<const APack<T, V> *>(Vp + (int64_t)(t_begin + min(base + grp + groups * u, n_seen - 1)) * a.vs[2] + col * V);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (keys() == kFew && base + groups * u >= n_seen) break;
        const int t = base + grp + groups * u;
        const float e = scores[min(t, n_seen - 1)];
        // the reference rounds the normalised probabilities to V's dtype
        const float p = a.f32_scores ? round_to<T>(e * inv) : round_to<T>(e / sum);
#pragma unroll
        for (int j = 0; j < V; ++j) {
          const float with = fmaf(p, (float)Scalar<T>::load(&pk[u].v[j]), acc[j]);
          acc[j] = keys() == kAll || t < n_seen ? with : acc[j];
        }
      }
    };
    int base = 0;
    for (; base + groups * U <= n_seen; base += groups * U) round(base, std::integral_constant<int, kAll>());
    if (base + groups * (U - 1) < n_seen) round(base, std::integral_constant<int, kSome>());
    else if (base < n_seen) round(base, std::integral_constant<int, kFew>());
    if (grp < groups) {
#pragma unroll
      for (int j = 0; j < V; ++j) red[grp * D + col * V + j] = acc[j];
    }
  }
  __syncthreads();
  T *o = (T *)a.out + ((int64_t)b * a.S + s) * a.out_row_stride + (int64_t)h * D;
  for (int d = tid; d < D; d += 256) {
    float r = 0.f;
    for (int g = 0; g < groups; ++g) r += red[g * D + d];
    if (a.gate)
      r *= gate_sigmoid((float)Scalar<T>::load((const T *)a.gate + ((int64_t)b * a.S + s) * a.gate_row_stride + (int64_t)h * D + d));
    Scalar<T>::store(o + d, (typename Scalar<T>::compute)r);
  }
}

// Rotary embedding of feature d of one head for position pos, with the
// reference's three roundings (x*cos, rotate_half(x)*sin, their sum:
// rai-models/src/llm/phi2.rs:75).
template <typename T>
__device__ __forceinline__ float rope_feature(const T *head, int d, int rot, const T *cos_t, const T *sin_t, int pos, int tab_f32) {
  float v = (float)Scalar<T>::load(head + d);
  if (d >= rot) return v;
  const int half = rot >> 1;
  float other = d < half ? -(float)Scalar<T>::load(head + d + half) : (float)Scalar<T>::load(head + d - half);
  if (tab_f32) {   // f32 tables: products and sum in f32, one rounding
    const int64_t e = (int64_t)pos * rot + d;
    return round_to<T>(fmaf(v, ((const float *)cos_t)[e], other * ((const float *)sin_t)[e]));
  }
  float c = (float)Scalar<T>::load(cos_t + (int64_t)pos * rot + d);
  float s = (float)Scalar<T>::load(sin_t + (int64_t)pos * rot + d);
  return round_to<T>(round_to<T>(v * c) + round_to<T>(other * s));
}

// The same in two steps, so that what it reads is asked for before anything waits: no request stands under a condition (what
// such a load returns is waited for where the condition ends).  A table's element is read as the aligned word around it.
template <typename T> struct RopeRaw {
  T v, other;
  uint32_t c, s, half_c, half_s;
};
template <typename T> __device__ __forceinline__ void rope_request_row(RopeRaw<T> &x, const T *head, int d, int rot) {
  const int half = rot >> 1;
  x.v = head[d];
  x.other = head[d < half ? d + half : d < rot ? d - half : d];
}
template <typename T>
__device__ __forceinline__ void rope_request_tables(RopeRaw<T> &x, int d, int rot, const void *cos_t, const void *sin_t, const void *any, int pos, int tab_f32) {
  const uint32_t size = tab_f32 ? 4 : sizeof(T);
  const int64_t at = rot ? ((int64_t)pos * rot + (d < rot ? d : 0)) * size : 0;   // (rot 0: no tables)
  const uintptr_t c = (uintptr_t)(rot ? cos_t : any) + at, s = (uintptr_t)(rot ? sin_t : any) + at;
  typedef const __attribute__((address_space(1))) uint32_t *word;
  x.c = *(word)(c & ~(uintptr_t)3);
  x.s = *(word)(s & ~(uintptr_t)3);
  x.half_c = (uint32_t)(c & 2) * 8;
  x.half_s = (uint32_t)(s & 2) * 8;
}
template <typename T> __device__ __forceinline__ float table_value(uint32_t word, uint32_t shift) {
  if constexpr (sizeof(T) == 4) return __uint_as_float(word);
  else {
    const T t = {(uint16_t)(word >> shift)};
    return (float)Scalar<T>::load(&t);
  }
}
template <typename T> __device__ __forceinline__ float rope_finish(const RopeRaw<T> &x, int d, int rot, int tab_f32) {
  const float v = (float)Scalar<T>::load(&x.v), o = (float)Scalar<T>::load(&x.other), other = d < (rot >> 1) ? -o : o;
  const float f = round_to<T>(fmaf(v, __uint_as_float(x.c), other * __uint_as_float(x.s)));
  const float t = round_to<T>(round_to<T>(v * table_value<T>(x.c, x.half_c)) + round_to<T>(other * table_value<T>(x.s, x.half_s)));
  return d >= rot ? v : tab_f32 ? f : t;
}

// Decode attention, split over the context ("flash decoding"): block
// (split, kv-head group, batch) handles ceil((pos+1)/NS) consecutive keys for
// the R query heads that share one KV head, so the cached K and V are read once
// per KV head (repeat_kv is never materialised) and NS * Hkv * B blocks keep
// every CU busy even at batch 1.  All of a block's first K and V loads are
// issued before anything is computed: a short context costs one HBM round trip.
// Each block writes an unnormalised partial (running max m, sum l, o[D]) per
// query head; the last block of a head group to finish (device-scope counter)
// merges the NS partials and writes the output row.  The new token's rotated
// key and value are appended to the cache by the block that owns position pos
// and are used from LDS.  Probabilities stay in f32 until the product with V.
//   What bounds it is the chain of trips: the position, everything that is read, the partials, the counter, the merge.  So nothing is
// asked for under a condition, and the tables come before the keys, whose arrival the rotation need not wait for: one head of 128
// a block, 777 keys over 33 splits 16.3 -> 10.8 us (masked loads: seven trips before the first score), the form below with 24 blocks of
// 96 keys x 256 features 11.7 -> 10.4.
constexpr int kDecodeThreads = 256;
constexpr int kDecodeMaxSplits = 64;
constexpr int kDecodeCounterStride = 32;

// Device-scope accesses for data handed from one block to another inside a
// kernel.  The L2 of each XCD is not coherent with the others for ordinary
// accesses, and a device-scope fence writes back and invalidates a whole L2;
// relaxed device-scope atomics instead write through / read around the L2 for
// just the words involved.
__device__ __forceinline__ void store_device(float *p, float v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float load_device(const float *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Tail of a decode-attention block: once its partials are written, the block
// counts itself in; the last block of the head group to arrive merges the NS
// partials of the R query heads starting at hq0 and writes their output rows.
// wbuf is block-shared scratch of 2 * R * NS floats that no wave uses any more.
// The merge is a chain of dependent memory round trips, so it is kept short: one for the (m, l) statistics, the sinks, the gate and
// the first SB splits' outputs alike (EU features a thread; up to 64 loads in flight), then the per-split weights
// exp(m_s - M) / L are computed once per head.  EU R: the features of a block's heads for up to 256 of them a head.
template <typename T, int EU>
__device__ __forceinline__ void decode_merge_last(const AttnDecodeArgs &a, int b, int hq0, int R, int *sh_last,
                                                  float *wbuf) {
  constexpr int NT = kDecodeThreads, SB = EU == 1 ? 32 : 64 / EU;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, NS = a.ns, D = a.D, PW = D + 2;
  // every thread's write-through stores have completed before the block's arrival is counted
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  int *counter = a.counters + ((int64_t)b * a.Hq + hq0) * kDecodeCounterStride;  // one 128-byte line each
  if (tid == 0) *sh_last = atomicAdd(counter, 1) == NS - 1;
  __syncthreads();
  if (!*sh_last) return;
  const float *all = a.ws + ((int64_t)b * a.Hq + hq0) * NS * PW;
  float *wm = wbuf, *wl = wbuf + R * NS;
  const float *po[EU];
  int hr[EU], hd[EU];
  float ov[EU][SB], gate[EU];
  auto features = [&](int e0) {   // this thread's features from e0 on
#pragma unroll
    for (int i = 0; i < EU; ++i) {
      const int e = e0 + i * NT < R * D ? e0 + i * NT : R * D - 1;
      hr[i] = e / D;
      hd[i] = e - hr[i] * D;
      po[i] = all + (int64_t)hr[i] * NS * PW + 2 + hd[i];
    }
  };
  auto outputs = [&](int s0) {
#pragma unroll
    for (int i = 0; i < EU; ++i)
#pragma unroll
      for (int j = 0; j < SB; ++j) ov[i][j] = load_device(po[i] + (s0 + j < NS ? s0 + j : NS - 1) * PW);
  };
  const float first_m = load_device(all + (int64_t)min(tid, R * NS - 1) * PW), first_l = load_device(all + (int64_t)min(tid, R * NS - 1) * PW + 1);
  const float sink0 = sink_of<T>(a.sink, hq0 + min(wave, R - 1));
  features(tid);
  if (a.gate) {
#pragma unroll
    for (int i = 0; i < EU; ++i)
      gate[i] = (float)Scalar<T>::load((const T *)a.gate + (int64_t)b * a.gate_row_stride + (int64_t)(hq0 + hr[i]) * D + hd[i]);
  }
  outputs(0);
  if (tid < R * NS) {   // (head r, split s) at index r*NS + s
    wm[tid] = first_m;
    wl[tid] = first_l;
  }
  for (int i = tid + NT; i < R * NS; i += NT) {
    const float *st = all + (int64_t)i * PW;
    wm[i] = load_device(st);
    wl[i] = load_device(st + 1);
  }
  __syncthreads();
  for (int r = wave; r < R; r += NT / 64) {      // NS <= 64: one split per lane
    const float m = lane < NS ? wm[r * NS + lane] : -INFINITY;
    const float sink = r == wave ? sink0 : sink_of<T>(a.sink, hq0 + r);
    const float M = fmaxf(wave_max(m), sink);    // split 0 always holds a key, so M is finite
    const float e = lane < NS ? expf(m - M) : 0.f;  // an empty split has m = -inf: weight 0
    const float L = wave_sum(lane < NS ? e * wl[r * NS + lane] : 0.f) + (a.sink ? expf(sink - M) : 0.f);
    if (lane < NS) wm[r * NS + lane] = e / L;
  }
  __syncthreads();
  for (int e0 = tid; e0 - tid < R * D; e0 += NT * EU) {
    if (e0 != tid) {   // (more than 256 features a head)
      features(e0);
#pragma unroll
      for (int i = 0; i < EU; ++i)
        if (a.gate) gate[i] = (float)Scalar<T>::load((const T *)a.gate + (int64_t)b * a.gate_row_stride + (int64_t)(hq0 + hr[i]) * D + hd[i]);
      outputs(0);
    }
    float O[EU];
#pragma unroll
    for (int i = 0; i < EU; ++i) O[i] = 0.f;
    for (int s0 = 0;;) {
#pragma unroll
      for (int i = 0; i < EU; ++i)
#pragma unroll
        for (int j = 0; j < SB; ++j)
          if (s0 + j < NS) O[i] = fmaf(wm[hr[i] * NS + s0 + j], ov[i][j], O[i]);
      s0 += SB;
      if (s0 >= NS) break;
      outputs(s0);
    }
#pragma unroll
    for (int i = 0; i < EU; ++i)
      if (e0 + i * NT < R * D) {
        if (a.gate) O[i] *= gate_sigmoid(gate[i]);
        Scalar<T>::store((T *)a.out + (int64_t)b * a.out_row_stride + (int64_t)(hq0 + hr[i]) * D + hd[i],
                         (typename Scalar<T>::compute)O[i]);
      }
  }
  if (tid == 0) *counter = 0;  // ready for the next launch (stream order)
}

template <typename T, int R, int CC, int UK, int UV>
__global__ void __launch_bounds__(kDecodeThreads) k_attn_decode_split(AttnDecodeArgs a) {
  constexpr int V = AttnVec<T>::V;
  constexpr int NT = kDecodeThreads, NW = NT / 64;
  extern __shared__ __attribute__((aligned(16))) float smem[];
  const int D = a.D, ncol = D / V, groups = NT / ncol;
  const int NS = a.ns, CH = a.chunk_cap;
  // layout: q[R*D] | knew[D] | vnew[D] | scores[R*CH] | red[groups*R*D]
  float *qf = smem;
  float *knew = qf + R * D;
  float *vnew = knew + D;
  float *scores = vnew + D;
  float *red = scores + R * CH;
  __shared__ float sh_m[R], sh_l[R];
  __shared__ int sh_last;

  const int s = blockIdx.x, b = blockIdx.z;
  const int hq0 = blockIdx.y * R;           // first query head of this block
  const int n_rep = a.Hq / a.Hkv, hk = hq0 / n_rep;
  const bool writer = hq0 % n_rep == 0;     // one block per KV head appends the new token
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int QD = a.Hq * D, KD = a.Hkv * D;
  // the new token's rows: one packed [q | k | v] row per sequence, or three separate ones
  const T *qrow = (const T *)a.qkv + (int64_t)b * (a.k_new ? a.q_row_stride : (int64_t)(QD + 2 * KD));
  const T *krow = (a.k_new ? (const T *)a.k_new + (int64_t)b * a.k_row_stride : qrow + QD) + hk * D;
  const T *vrow = (a.k_new ? (const T *)a.v_new + (int64_t)b * a.v_row_stride : qrow + QD + KD) + hk * D;
  // asked for before the position is here: the query rows (up to 256 features a head; what is beyond, further down), the new key and value
  RopeRaw<T> qx[R], kx;
  int qd[R];
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int e = min(tid + i * NT, R * D - 1), r = e / D;
    qd[i] = e - r * D;
    rope_request_row(qx[i], qrow + (hq0 + r) * D, qd[i], a.rot);
  }
  const int kd = min(tid, D - 1);
  rope_request_row(kx, krow, kd, a.rot);
  const T v_new = vrow[kd];
  int pos = a.pos_dev ? *a.pos_dev : a.pos_host;
  if (pos > a.Tmax - 1) pos = a.Tmax - 1;   // capacity is checked on the host; never write past the cache
  const int cnt = pos + 1;
  int chunk = (cnt + NS - 1) / NS;
  if (chunk > CH) chunk = CH;
  const int t0 = s * chunk;
  const int t1 = t0 + chunk < cnt ? t0 + chunk : cnt;
  const int n = t1 > t0 ? t1 - t0 : 0;      // keys of this split (the new token included when it falls inside)
  const bool has_new = pos >= t0 && pos < t1;
  const int t1c = has_new ? pos : t1;       // cached keys are [t0, t1c)

  T *Kc = (T *)a.kcache + ((int64_t)b * a.Hkv + hk) * a.Tmax * D;
  T *Vc = (T *)a.vcache + ((int64_t)b * a.Hkv + hk) * a.Tmax * D;
  const T *cos_t = (const T *)a.cos_t, *sin_t = (const T *)a.sin_t;
  const int g = tid >> 4, gl = tid & 15;
  const int col = tid % ncol, grp = tid / ncol;

  // ---- tables, then the first round of K and V: every load whole (keys past the end: the last one, never used)
#pragma unroll
  for (int i = 0; i < R; ++i) rope_request_tables(qx[i], qd[i], a.rot, cos_t, sin_t, qrow, pos, a.tab_f32);
  rope_request_tables(kx, kd, a.rot, cos_t, sin_t, qrow, pos, a.tab_f32);
  APack<T, V> kreg[UK][CC], vreg[UV];
  const int last = max(t1c - 1, 0);
  auto ask_k = [&](int tb) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < UK; ++u)
#pragma unroll
      for (int cc = 0; cc < CC; ++cc)
        kreg[u][cc] = *reinterpret_cast<const APack<T, V> *>(Kc + (int64_t)min(tb + 16 * u, last) * D + min(gl + 16 * cc, ncol - 1) * V);
  };
  auto ask_v = [&](int tb) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < UV; ++u) vreg[u] = *reinterpret_cast<const APack<T, V> *>(Vc + (int64_t)min(tb + u * groups, last) * D + col * V);
  };
  ask_k(t0 + g);
  ask_v(t0 + grp);
  // ---- rotary embedding of the R query rows (and of the new key where it is needed)
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const float x = rope_finish(qx[i], qd[i], a.rot, a.tab_f32);
    if (tid + i * NT < R * D) qf[tid + i * NT] = x;
  }
  for (int e = tid + R * NT; e < R * D; e += NT) {
    const int r = e / D, d = e - r * D;
    qf[e] = rope_feature<T>(qrow + (hq0 + r) * D, d, a.rot, cos_t, sin_t, pos, a.tab_f32);
  }
  if (has_new) {
    for (int d = tid; d < D; d += NT) {
      const float kr = d == tid ? rope_finish(kx, kd, a.rot, a.tab_f32) : rope_feature<T>(krow, d, a.rot, cos_t, sin_t, pos, a.tab_f32);
      const T vt = d == tid ? v_new : vrow[d];
      const float vr = (float)Scalar<T>::load(&vt);
      knew[d] = kr;
      vnew[d] = vr;
      if (writer) {
        Scalar<T>::store(Kc + (int64_t)pos * D + d, (typename Scalar<T>::compute)kr);
        Scalar<T>::store(Vc + (int64_t)pos * D + d, (typename Scalar<T>::compute)vr);
      }
    }
  }
  __syncthreads();

  auto finish_score = [&](float acc) -> float {
    if (a.f32_scores) return cap_score(acc * a.scale, a.softcap);
    return round_to<T>(round_to<T>(acc) * round_to<T>(a.scale));
  };
  // ---- scores against the cached keys: 16 lanes per key row, each round's keys asked for a round ahead
  for (int base = t0; base < t1c; base += 16 * UK) {
    const int tb = base + g;
    float kf[UK][CC][V];
#pragma unroll
    for (int u = 0; u < UK; ++u)
#pragma unroll
      for (int cc = 0; cc < CC; ++cc)
#pragma unroll
        for (int j = 0; j < V; ++j) kf[u][cc][j] = (float)Scalar<T>::load(&kreg[u][cc].v[j]);
    if (base + 16 * UK < t1c) ask_k(tb + 16 * UK);
#pragma unroll
    for (int u = 0; u < UK; ++u) {
      const int t = tb + 16 * u;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        float acc = 0.f;
#pragma unroll
        for (int cc = 0; cc < CC; ++cc) {
          const int c = gl + 16 * cc;
          if (t < t1c && c < ncol) {
#pragma unroll
            for (int j = 0; j < V; ++j) acc = fmaf(qf[r * D + c * V + j], kf[u][cc][j], acc);
          }
        }
        acc = row_sum(acc);
        if (gl == 0 && t < t1c) scores[r * CH + (t - t0)] = finish_score(acc);
      }
    }
  }
  if (has_new && wave == NW - 1) {  // the new token's own key, still in LDS
    for (int r = 0; r < R; ++r) {
      float acc = 0.f;
      for (int d = lane; d < D; d += 64) acc = fmaf(qf[r * D + d], knew[d], acc);
      acc = wave_sum(acc);
      if (lane == 0) scores[r * CH + (pos - t0)] = finish_score(acc);
    }
  }
  __syncthreads();
  // ---- partial softmax statistics, one wave per query head
  for (int r = wave; r < R; r += NW) {
    float m = -INFINITY;
    for (int t = lane; t < n; t += 64) m = fmaxf(m, scores[r * CH + t]);
    m = wave_max(m);
    float l = 0.f;
    for (int t = lane; t < n; t += 64) {
      const float e = expf(scores[r * CH + t] - m);
      scores[r * CH + t] = e;
      l += e;
    }
    l = wave_sum(l);
    if (lane == 0) { sh_m[r] = m; sh_l[r] = l; }
  }
  __syncthreads();
  // ---- unnormalised P.V over the cached values: round 0 from the prefetched registers
  {
    float acc[R][V];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int j = 0; j < V; ++j) acc[r][j] = 0.f;
    {
      for (int base = t0; base < t1c; base += UV * groups) {
        const int tb = base + grp;
        if (base != t0) ask_v(tb);
#pragma unroll
        for (int u = 0; u < UV; ++u) {
          const int t = tb + u * groups;
          if (t < t1c && grp < groups) {
            float vf[V];
#pragma unroll
            for (int j = 0; j < V; ++j) vf[j] = (float)Scalar<T>::load(&vreg[u].v[j]);
#pragma unroll
            for (int r = 0; r < R; ++r) {
              const float p = scores[r * CH + (t - t0)];
#pragma unroll
              for (int j = 0; j < V; ++j) acc[r][j] = fmaf(p, vf[j], acc[r][j]);
            }
          }
        }
      }
      if (grp < groups) {
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
          for (int j = 0; j < V; ++j) red[(grp * R + r) * D + col * V + j] = acc[r][j];
      }
    }
  }
  __syncthreads();
  // ---- partial (m, l, o[D]) of every query head of the block
  const int PW = D + 2;
  float *part = a.ws + (((int64_t)b * a.Hq + hq0) * NS + s) * PW;  // head r at part + r*NS*PW
  for (int e = tid; e < R * D; e += NT) {
    const int r = e / D, d = e - r * D;
    float o = has_new ? scores[r * CH + (pos - t0)] * vnew[d] : 0.f;
    for (int gg = 0; gg < groups; ++gg) o += red[(gg * R + r) * D + d];
    store_device(part + (int64_t)r * NS * PW + 2 + d, o);
  }
  if (tid < R) {
    store_device(part + (int64_t)tid * NS * PW, sh_m[tid]);
    store_device(part + (int64_t)tid * NS * PW + 1, sh_l[tid]);
  }
  decode_merge_last<T, R>(a, b, hq0, R, &sh_last, smem);
}

// Number of context splits: enough blocks to fill the chip, bounded so that a
// block's share of the longest context fits the LDS score buffer.
static int decode_splits(const AttnDecodeArgs &a, int head_groups) {
  const char *knob = getenv("RAI_HIP_ATTN_SPLITS");  // tuning and test aid, read at every launch
  const int forced = knob ? atoi(knob) : 0;
  int ns = forced > 0 ? forced : (2 * kNumCU + head_groups * a.B - 1) / (head_groups * a.B);
  // not more blocks than there are runs of 64 keys: below that a block's share no longer pays for its part of the
  // merge (a 530-key context of 32 heads: 8 splits 1.89 ms per Phi-2 token through the graph path, 16 splits 1.96,
  // 32 splits 2.34).  The length is the host's when it knows it, the cache's capacity otherwise.
  const int len = a.pos_dev ? a.Tmax : a.pos_host + 1;
  if (forced <= 0 && ns > (len + 63) / 64) ns = (len + 63) / 64;
  const int need = (a.Tmax + 1023) / 1024;
  if (ns < need) ns = need;
  if (ns > kDecodeMaxSplits) ns = kDecodeMaxSplits;
  if (ns > a.Tmax) ns = a.Tmax;
  return ns < 1 ? 1 : ns;
}

size_t attention_decode_ws_bytes(int B, int Hq, int D) {
  return sizeof(float) * (size_t)B * Hq * kDecodeMaxSplits * (D + 2);
}
size_t attention_decode_counter_bytes(int B, int Hq) { return sizeof(int) * (size_t)B * Hq * kDecodeCounterStride; }

// Decode attention for grouped-query models in bf16, both products on
// v_mfma_f32_16x16x32_bf16.  Block (split, kv head, batch) serves all R <= 16 query
// heads of one KV head over at most CH (64 or 128) consecutive keys:
//   - every K and V load of the block is issued before anything is computed.  K goes
//     straight from global memory into MFMA A fragments (lane l: key l%16 of a 16-key
//     tile, features 32*step + 8*(l/16) ..), one or two tiles per wave; V goes through LDS;
//   - scores^T[key, head] = K . Q^T per tile; accumulator register r of lane l is key
//     4*(l/16)+r, head l%16.  The rotated queries are the B fragments, held in registers;
//   - per-head max / exp / sum over the block's keys (one wave per head), exp values
//     rounded to bf16 for the second product (the reference rounds P to V's dtype);
//   - O[head, feature] = P . V: wave w of NW owns features [w*D/NW, (w+1)*D/NW), P fragments are
//     16-byte LDS reads, V fragments are gathered from LDS two bytes at a time (the
//     transposition costs LDS reads, of which there are few: the kernel is bound by
//     the K/V stream);
//   - partial (m, l, o[D]) per head, merged by the last block as in the split kernel.
typedef __attribute__((ext_vector_type(8))) __bf16 ad_bf16x8;
typedef __attribute__((ext_vector_type(4))) float ad_f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t ad_u32x4;

template <int D, int CH, int NT>
__global__ void __launch_bounds__(NT) k_attn_decode_mfma(AttnDecodeArgs a) {
  typedef bf16_raw T;
  constexpr int NW = NT / 64;
  constexpr int KS = D / 32, KT = (CH / 16 + NW - 1) / NW;  // 16-key tiles per wave (the last may be empty)
  constexpr int VP = D + 8, PP = CH + 8;           // LDS pitches (bf16 elements)
  constexpr int CPR = D / 8;                        // 16-byte chunks per K/V row
  constexpr int VL = CH * CPR / NT;                  // V chunks per thread
  constexpr int DT = D / 16 / NW;                    // 16-feature tiles per wave in P.V
  extern __shared__ __attribute__((aligned(16))) float smem[];
  uint16_t *Vs = reinterpret_cast<uint16_t *>(smem);          // [CH][VP]; the first 16 rows hold Q until the scores are done
  const int R = a.Hq / a.Hkv;
  float *scores = reinterpret_cast<float *>(Vs + CH * VP);    // [R][CH]
  uint16_t *ps = reinterpret_cast<uint16_t *>(scores + R * CH);   // [16][PP]
  uint16_t *knew = ps + 16 * PP;                              // [D]
  uint16_t *vnew = knew + D;                                  // [D]
  __shared__ float sh_m[16], sh_l[16];

  const int s = blockIdx.x, hk = blockIdx.y, b = blockIdx.z;
  const int hq0 = hk * R;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lrow = lane & 15, lq = lane >> 4;
  const int NS = a.ns;
  const int QD = a.Hq * D, KD = a.Hkv * D;
  // the new token's rows: one packed [q | k | v] row per sequence, or three separate ones
  const T *qrow = (const T *)a.qkv + (int64_t)b * (a.k_new ? a.q_row_stride : (int64_t)(QD + 2 * KD));
  const T *krow = (a.k_new ? (const T *)a.k_new + (int64_t)b * a.k_row_stride : qrow + QD) + hk * D;
  const T *vrow = (a.k_new ? (const T *)a.v_new + (int64_t)b * a.v_row_stride : qrow + QD + KD) + hk * D;
  // ---- asked for before the position is here, every load whole: feature tid of the new token's key and value, the query rows
  // (eight features per item; `by8`: a rotary half is whole items)
  static_assert(D <= NT && CH * CPR % NT == 0 && D % (16 * NW) == 0, "a thread per feature, whole rounds of V, whole tiles of features");
  constexpr int QI = (16 * CPR + NT - 1) / NT;
  const bool by8 = a.rot % 16 == 0;
  const int rot8 = by8 ? a.rot : 0, half = rot8 >> 1, kd = tid < D ? tid : D - 1;
  RopeRaw<T> kx;
  rope_request_row(kx, krow, kd, a.rot);
  const T new_v = vrow[kd];
  ad_u32x4 qx[QI], qo[QI], qc[QI][2], qn[QI][2];
#pragma unroll
  for (int i = 0; i < QI; ++i) {
    const int item = tid + i * NT, r = item / CPR, d = (item - r * CPR) * 8;
    const T *row = qrow + (hq0 + min(r, R - 1)) * D;
    qx[i] = *reinterpret_cast<const ad_u32x4 *>(row + d);
    qo[i] = *reinterpret_cast<const ad_u32x4 *>(row + (d < half ? d + half : d < rot8 ? d - half : d));
  }
  int pos = a.pos_dev ? *a.pos_dev : a.pos_host;
  if (pos > a.Tmax - 1) pos = a.Tmax - 1;   // capacity is checked on the host; never write past the cache
  const int cnt = pos + 1;
  int chunk = (cnt + NS - 1) / NS;
  if (chunk > CH) chunk = CH;
  const int t0 = s * chunk;
  const int t1 = t0 + chunk < cnt ? t0 + chunk : cnt;
  const int n = t1 > t0 ? t1 - t0 : 0;
  const bool has_new = pos >= t0 && pos < t1;
  const int t1c = has_new ? pos : t1;       // cached keys are [t0, t1c)
  const int new_row = pos - t0;

  T *Kc = (T *)a.kcache + ((int64_t)b * a.Hkv + hk) * a.Tmax * D;
  T *Vc = (T *)a.vcache + ((int64_t)b * a.Hkv + hk) * a.Tmax * D;
  const T *cos_t = (const T *)a.cos_t, *sin_t = (const T *)a.sin_t;

  // ---- the tables (eight values are 16 or 32 bytes), then all K and V loads of the block (past the end: the last key once more)
#pragma unroll
  for (int i = 0; i < QI; ++i) {
    const int item = tid + i * NT, d = item % CPR * 8, size = a.tab_f32 ? 4 : 2;
    const int64_t at = ((int64_t)pos * rot8 + (d < rot8 ? d : 0)) * size;
    const char *c = by8 && rot8 ? (const char *)a.cos_t + at : (const char *)qrow, *sn = by8 && rot8 ? (const char *)a.sin_t + at : (const char *)qrow;
    const int second = a.tab_f32 && by8 && rot8 ? 16 : 0;
    __builtin_memcpy(&qc[i][0], c, 16);
    __builtin_memcpy(&qc[i][1], c + second, 16);
    __builtin_memcpy(&qn[i][0], sn, 16);
    __builtin_memcpy(&qn[i][1], sn + second, 16);
  }
  rope_request_tables(kx, kd, a.rot, cos_t, sin_t, qrow, pos, a.tab_f32);
  const int last = max(t1c - 1, 0);
  ad_bf16x8 kreg[KT][KS];
#pragma unroll
  for (int i = 0; i < KT; ++i)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      kreg[i][ks] = *reinterpret_cast<const ad_bf16x8 *>(Kc + (int64_t)min(t0 + (wave + NW * i) * 16 + lrow, last) * D + ks * 32 + lq * 8);
  ad_u32x4 vreg[VL];
#pragma unroll
  for (int j = 0; j < VL; ++j) {
    const int c = tid + j * NT, r = c / CPR, c8 = c - r * CPR;
    vreg[j] = *reinterpret_cast<const ad_u32x4 *>(Vc + (int64_t)min(t0 + r, last) * D + c8 * 8);
  }
  // ---- rotated queries (rows >= R are zero)
  if (by8) {
#pragma unroll
    for (int i = 0; i < QI; ++i) {
      const int item = tid + i * NT, r = item / CPR, d = (item - r * CPR) * 8;
      if (item >= 16 * CPR) continue;
      ad_u32x4 out = r < R ? qx[i] : ad_u32x4{0u, 0u, 0u, 0u};
      if (r < R && d < a.rot && a.tab_f32) {   // f32 tables: products and sum in f32, one rounding
        const float sign = d < half ? -1.f : 1.f;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          float res[2];
#pragma unroll
          for (int hbit = 0; hbit < 2; ++hbit) {
            const int sh = 16 * hbit;
            const float x = bf16_bits_to_f32((uint16_t)(qx[i][w] >> sh)), o = sign * bf16_bits_to_f32((uint16_t)(qo[i][w] >> sh));
            res[hbit] = fmaf(x, __uint_as_float(qc[i][w >> 1][(2 * w + hbit) & 3]), o * __uint_as_float(qn[i][w >> 1][(2 * w + hbit) & 3]));
          }
          out[w] = pack_bf16x2(res[0], res[1]);
        }
      } else if (r < R && d < a.rot) {
        const float sign = d < half ? -1.f : 1.f;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          uint32_t packed = 0;
#pragma unroll
          for (int hbit = 0; hbit < 2; ++hbit) {
            const int sh = 16 * hbit;
            const float x = bf16_bits_to_f32((uint16_t)(qx[i][w] >> sh)), o = sign * bf16_bits_to_f32((uint16_t)(qo[i][w] >> sh));
            const float c = bf16_bits_to_f32((uint16_t)(qc[i][0][w] >> sh)), sn = bf16_bits_to_f32((uint16_t)(qn[i][0][w] >> sh));
            // three roundings, as rope_feature
            const float res = round_to<T>(round_to<T>(x * c) + round_to<T>(o * sn));
            packed |= (uint32_t)f32_to_bf16_bits(res) << sh;
          }
          out[w] = packed;
        }
      }
      *reinterpret_cast<ad_u32x4 *>(Vs + r * VP + d) = out;
    }
  } else {
    for (int e = tid; e < 16 * D; e += NT) {
      const int r = e / D, d = e - r * D;
      const float q = r < R ? rope_feature<T>(qrow + (hq0 + r) * D, d, a.rot, cos_t, sin_t, pos, a.tab_f32) : 0.f;
      Vs[r * VP + d] = f32_to_bf16_bits(q);
    }
  }
  for (int e = tid; e < 16 * PP; e += NT) ps[e] = 0;
  if (has_new && tid < D) {
    const uint16_t kr = f32_to_bf16_bits(rope_finish(kx, kd, a.rot, a.tab_f32));
    knew[tid] = kr;
    vnew[tid] = new_v.bits;
    (Kc + (int64_t)pos * D + tid)->bits = kr;
    (Vc + (int64_t)pos * D + tid)->bits = new_v.bits;
  }
  __syncthreads();

  // ---- scores
  {
    ad_bf16x8 qf[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = *reinterpret_cast<const ad_bf16x8 *>(Vs + lrow * VP + ks * 32 + lq * 8);
#pragma unroll
    for (int i = 0; i < KT; ++i) {
      const int tile = wave + NW * i;
      if (tile * 16 >= CH) continue;
      if (has_new && new_row == tile * 16 + lrow) {   // the lanes that hold the new token's key row
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) kreg[i][ks] = *reinterpret_cast<const ad_bf16x8 *>(knew + ks * 32 + lq * 8);
      }
      ad_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kreg[i][ks], qf[ks], acc, 0, 0, 0);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int tl = tile * 16 + 4 * lq + r;
        float sc = a.f32_scores ? cap_score(acc[r] * a.scale, a.softcap) : round_to<T>(round_to<T>(acc[r]) * round_to<T>(a.scale));
        if (lrow < R) scores[lrow * CH + tl] = tl < n ? sc : -INFINITY;
      }
    }
  }
  __syncthreads();

  // ---- V into LDS (the new token's row from the activations), softmax statistics
#pragma unroll
  for (int j = 0; j < VL; ++j) {
    const int c = tid + j * NT, r = c / CPR, c8 = c - r * CPR;
    ad_u32x4 v = t0 + r < t1c ? vreg[j] : ad_u32x4{0u, 0u, 0u, 0u};
    if (has_new && r == new_row) v = *reinterpret_cast<const ad_u32x4 *>(vnew + c8 * 8);
    *reinterpret_cast<ad_u32x4 *>(Vs + r * VP + c8 * 8) = v;
  }
  for (int r = wave; r < R; r += NW) {
    float m = -INFINITY;
    for (int t = lane; t < n; t += 64) m = fmaxf(m, scores[r * CH + t]);
    m = wave_max(m);
    float l = 0.f;
    for (int t = lane; t < n; t += 64) {
      const float e = expf(scores[r * CH + t] - m);
      ps[r * PP + t] = f32_to_bf16_bits(e);
      l += e;
    }
    l = wave_sum(l);
    if (lane == 0) { sh_m[r] = m; sh_l[r] = l; }
  }
  __syncthreads();

  // ---- O = P . V for this wave's features
  const int PW = D + 2;
  float *part = a.ws + (((int64_t)b * a.Hq + hq0) * NS + s) * PW;  // head r at part + r*NS*PW
  {
    ad_f32x4 o[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) o[dt] = ad_f32x4{0.f, 0.f, 0.f, 0.f};
    const int d0 = wave * (D / NW);
    for (int k0 = 0; k0 < n; k0 += 32) {
      const ad_bf16x8 pf = *reinterpret_cast<const ad_bf16x8 *>(ps + lrow * PP + k0 + lq * 8);
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        typedef __attribute__((ext_vector_type(8))) uint16_t u16x8;
        u16x8 vb;
#pragma unroll
        for (int j = 0; j < 8; ++j) vb[j] = Vs[(k0 + lq * 8 + j) * VP + d0 + dt * 16 + lrow];
        o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pf, __builtin_bit_cast(ad_bf16x8, vb), o[dt], 0, 0, 0);
      }
    }
    // accumulator register r of lane l is head 4*(l/16)+r, feature l%16 of the tile
    if (NS == 1) {   // nothing to merge
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int h = 4 * lq + r;
        if (h >= R) continue;
        const float sink = sink_of<T>(a.sink, hq0 + h), M = fmaxf(sh_m[h], sink), e = expf(sh_m[h] - M);
        const float w = e / (e * sh_l[h] + (a.sink ? expf(sink - M) : 0.f));
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
          const int64_t f = (int64_t)(hq0 + h) * D + d0 + dt * 16 + lrow;
          float y = w * o[dt][r];
          if (a.gate) y *= gate_sigmoid((float)Scalar<T>::load((const T *)a.gate + (int64_t)b * a.gate_row_stride + f));
          Scalar<T>::store((T *)a.out + (int64_t)b * a.out_row_stride + f, y);
        }
      }
      return;
    }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int h = 4 * lq + r;
        if (h < R) part[(int64_t)h * NS * PW + 2 + d0 + dt * 16 + lrow] = o[dt][r];
      }
  }
  if (tid < R) {
    part[(int64_t)tid * NS * PW] = sh_m[tid];
    part[(int64_t)tid * NS * PW + 1] = sh_l[tid];
  }
}

// Merges the NS partials of one (batch, query head): block (head, batch), one
// thread per output feature.  Every wave computes the split weights
// exp(m_s - M) / L with one split per lane (NS <= 64), then each thread has all
// its partial-output loads in flight at once: two memory round trips in all.
__global__ void __launch_bounds__(256) k_attn_decode_merge_bf16(AttnDecodeArgs a) {
  const int h = blockIdx.x, b = blockIdx.y, d = threadIdx.x, lane = threadIdx.x & 63;
  const int NS = a.ns, D = a.D, PW = D + 2;
  const float *pr = a.ws + ((int64_t)b * a.Hq + h) * NS * PW;
  const float m = lane < NS ? pr[lane * PW] : -INFINITY;
  const float l = lane < NS ? pr[lane * PW + 1] : 0.f;
  const float sink = sink_of<bf16_raw>(a.sink, h);
  float gate = 1.f;
  if (a.gate) gate = gate_sigmoid((float)Scalar<bf16_raw>::load((const bf16_raw *)a.gate + (int64_t)b * a.gate_row_stride + (int64_t)h * D + d));
  const float M = fmaxf(wave_max(m), sink);       // split 0 always holds a key, so M is finite
  const float e = lane < NS ? expf(m - M) : 0.f;  // an empty split has m = -inf: weight 0
  const float L = wave_sum(e * l) + (a.sink ? expf(sink - M) : 0.f);
  const float w = e / L;
  float O = 0.f;
  constexpr int SB = 16;
  for (int s0 = 0; s0 < NS; s0 += SB) {
    float ov[SB];
#pragma unroll
    for (int j = 0; j < SB; ++j) ov[j] = pr[(s0 + j < NS ? s0 + j : NS - 1) * PW + 2 + d];
#pragma unroll
    for (int j = 0; j < SB; ++j)
      if (s0 + j < NS) O = fmaf(__shfl(w, s0 + j, 64), ov[j], O);
  }
  ((bf16_raw *)a.out + (int64_t)b * a.out_row_stride + (int64_t)h * D + d)->bits = f32_to_bf16_bits(O * gate);
}

// Splits of the context over blocks of `ch` keys.  A block that holds the longest context the cache has room for (the context itself is the
// device's to know) writes the result itself, without the launch that merges: 24 sequences on 51 to 83 keys (8 heads of 256 on one) 10.4 us
// for 7.2 + 4.7 in two blocks a sequence (four waves each).  One to 32 sequences of 52 to 122 keys decoded so, against two blocks each: 128 features 0.2 to
// 3 % sooner, 256 features 0.3 to 2 % up to 96 keys and within 1 % either way beyond.
static int mfma_decode_splits(const AttnDecodeArgs &a, int ch) {
  if (a.Tmax <= ch && !getenv("RAI_HIP_ATTN_SPLITS")) return 1;
  const int ns = decode_splits(a, a.Hkv), need = (a.Tmax + ch - 1) / ch;
  return ns < need ? need : ns;
}

template <int D, int CH, int NT> static int launch_decode_mfma_cfg(hipStream_t st, AttnDecodeArgs a) {
  const int R = a.Hq / a.Hkv;
  a.chunk_cap = CH;
  const size_t lds = (size_t)CH * (D + 8) * 2 + (size_t)R * CH * 4 + 16 * (CH + 8) * 2 + 2 * D * 2;
  static bool attr_set = false;
  if (lds > 64 * 1024 && !attr_set) {
    RAI_HIP_TRY(hipFuncSetAttribute((const void *)k_attn_decode_mfma<D, CH, NT>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                    (int)((size_t)CH * (D + 8) * 2 + 16 * CH * 4 + 16 * (CH + 8) * 2 + 2 * D * 2)));
    attr_set = true;
  }
  RAI_REQUIRE(a.Hkv <= 65535 && a.B <= 65535, RAI_ERR_UNSUPPORTED, "attention decode: grid too large");
  hipLaunchKernelGGL((k_attn_decode_mfma<D, CH, NT>), dim3(a.ns, a.Hkv, a.B), dim3(NT), lds, st, a);
  RAI_TRY(launch_check("attention_decode_mfma"));
  if (a.ns == 1) return RAI_OK;
  hipLaunchKernelGGL(k_attn_decode_merge_bf16, dim3(a.Hq, a.B), dim3(D), 0, st, a);
  return launch_check("attention_decode_merge");
}

// Eight waves to a block where all blocks are on the chip with them, four beyond, where more blocks share a CU and its registers.  A block is a chain
// of a few trips to memory and of its own steps, which eight waves halve.  Measured (us, four waves, eight): 256 features, 24 blocks
// of 96 keys 10.3, 7.7, 16 of 64 7.1, 6.1, 240 8.4, 7.6, 512 12.0, 10.9; 128 features, 32 blocks 5.6, 5.1, 256 6.3, 5.6, 320 7.2, 7.1, 1024
// 11.9, 13.5.  (128 keys of 256 features take more registers than two blocks of eight waves have.)
template <int D, int CH> static int launch_decode_mfma_waves(hipStream_t st, AttnDecodeArgs a) {
  a.ns = mfma_decode_splits(a, CH);
  if constexpr (D >= 128) {
    if ((int64_t)a.ns * a.Hkv * a.B <= (D == 256 && CH < 128 ? 2 : 1) * kNumCU) return launch_decode_mfma_cfg<D, CH, 512>(st, a);
  }
  return launch_decode_mfma_cfg<D, CH, 256>(st, a);
}

// Keys per block: 64, 96 or 128.  Every block issues all its loads up front and a CU holds as many blocks as their LDS
// allows, so what counts is the number of rounds the blocks need on the chip: a few blocks more than one round (1056
// blocks of 64 keys on 1024 places, Gemma-2B at batch 32 just past 2048 tokens) cost a whole block time.  Fewest
// rounds wins, then the smaller block.
constexpr int kMfmaDecodeKeysMax = 128;
template <int D> static size_t decode_mfma_lds(int CH, int R) {
  return (size_t)CH * (D + 8) * 2 + (size_t)R * CH * 4 + 16 * (CH + 8) * 2 + 2 * D * 2;
}
template <int D> static int launch_decode_mfma(hipStream_t st, const AttnDecodeArgs &a) {
  const char *knob = getenv("RAI_HIP_ATTN_KEYS");  // tuning and test aid: 64, 96 or 128 keys per block
  const int forced = knob ? atoi(knob) : 0;
  const int R = a.Hq / a.Hkv;
  int best = 0, best_rounds = 0;
  for (int ch : {64, 96, 128}) {
    if ((a.Tmax + ch - 1) / ch > kDecodeMaxSplits) continue;
    const int ns = mfma_decode_splits(a, ch);
    const long long blocks = (long long)ns * a.Hkv * a.B;
    const long long per_cu = (long long)((160 * 1024) / (decode_mfma_lds<D>(ch, R) + 256));
    const long long places = (per_cu < 1 ? 1 : per_cu) * kNumCU;
    const int rounds = (int)((blocks + places - 1) / places);
    if (forced == ch) { best = ch; break; }
    if (!best || rounds < best_rounds) { best = ch; best_rounds = rounds; }
    if (ns == 1 && !forced) { best = ch; break; }   // the smallest block that holds every key
  }
  if (best == 64) return launch_decode_mfma_waves<D, 64>(st, a);
  if (best == 96) return launch_decode_mfma_waves<D, 96>(st, a);
  return launch_decode_mfma_waves<D, 128>(st, a);
}

// The MFMA kernel serves bf16 grouped-query shapes whose longest context fits
// kDecodeMaxSplits blocks of kMfmaDecodeKeysMax keys.
static bool decode_mfma_eligible(const AttnDecodeArgs &a) {
  const bool off = getenv("RAI_HIP_NO_MFMA_DECODE") != nullptr;   // per call: a test compares both kernels in one process
  const int rep = a.Hq / a.Hkv;
  return !off && a.dtype == RAI_BF16 && rep >= 4 && rep <= 16 && (a.D == 64 || a.D == 128 || a.D == 256) &&
         (a.Tmax + kMfmaDecodeKeysMax - 1) / kMfmaDecodeKeysMax <= kDecodeMaxSplits;
}

template <typename T, int R, int CC, int UK, int UV> static int launch_decode_cfg(hipStream_t st, AttnDecodeArgs a) {
  constexpr int V = AttnVec<T>::V;
  const int ncol = a.D / V, groups = kDecodeThreads / ncol;
  const int head_groups = a.Hq / R;
  a.ns = decode_splits(a, head_groups);
  a.chunk_cap = (a.Tmax + a.ns - 1) / a.ns;
  const size_t lds = sizeof(float) * ((size_t)R * a.D + 2 * (size_t)a.D + (size_t)R * a.chunk_cap + (size_t)groups * R * a.D);
  RAI_REQUIRE(lds <= 150 * 1024, RAI_ERR_UNSUPPORTED, "attention: context %d too long for the decode kernel", a.Tmax);
  static size_t attr_bytes = 0;
  if (lds > 64 * 1024 && lds > attr_bytes) {
    RAI_HIP_TRY(hipFuncSetAttribute((const void *)k_attn_decode_split<T, R, CC, UK, UV>,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, 150 * 1024));
    attr_bytes = 150 * 1024;
  }
  RAI_REQUIRE(head_groups <= 65535 && a.B <= 65535, RAI_ERR_UNSUPPORTED, "attention decode: grid too large");
  hipLaunchKernelGGL((k_attn_decode_split<T, R, CC, UK, UV>), dim3(a.ns, head_groups, a.B), dim3(kDecodeThreads), lds, st, a);
  return launch_check("attention_decode");
}

template <typename T, int R> static int launch_decode_r(hipStream_t st, const AttnDecodeArgs &a) {
  constexpr int V = AttnVec<T>::V;
  const int ncol = a.D / V;
  if (ncol <= 16) return launch_decode_cfg<T, R, 1, 3, 3>(st, a);
  if (ncol <= 32) return launch_decode_cfg<T, R, 2, 2, 4>(st, a);
  return launch_decode_cfg<T, R, 4, 1, 2>(st, a);
}

template <typename T> static int launch_decode(hipStream_t st, const AttnDecodeArgs &a) {
  constexpr int V = AttnVec<T>::V;
  RAI_REQUIRE(a.D % V == 0 && a.D / V <= 64, RAI_ERR_BAD_SHAPE, "attention: head_dim %d unsupported", a.D);
  // the query heads of one KV head share a block when their count has an instantiation
  switch (a.Hq / a.Hkv) {
    case 2: return launch_decode_r<T, 2>(st, a);
    case 4: return launch_decode_r<T, 4>(st, a);
    case 6: return launch_decode_r<T, 6>(st, a);
    case 8: return launch_decode_r<T, 8>(st, a);
    default: return launch_decode_r<T, 1>(st, a);
  }
}

int launch_attention_decode(hipStream_t st, const AttnDecodeArgs &a) {
  RAI_REQUIRE(a.B > 0 && a.Hq > 0 && a.Hkv > 0 && a.D > 0 && a.Tmax > 0 && a.Hq % a.Hkv == 0, RAI_ERR_BAD_SHAPE,
              "attention decode: bad problem");
  RAI_REQUIRE(a.rot >= (a.tab_f32 ? 0 : 2) && a.rot % 2 == 0 && a.rot <= a.D, RAI_ERR_BAD_ARG, "attention decode: rot %d", a.rot);
  RAI_REQUIRE(a.f32_scores || (!a.sink && a.softcap <= 0.f), RAI_ERR_BAD_ARG, "attention decode: a cap or a sink needs the f32-score form");
  RAI_REQUIRE(a.ws && a.counters, RAI_ERR_BAD_ARG, "attention decode: partial-result workspace missing");
  if (decode_mfma_eligible(a)) {
    if (a.D == 64) return launch_decode_mfma<64>(st, a);
    if (a.D == 128) return launch_decode_mfma<128>(st, a);
    return launch_decode_mfma<256>(st, a);
  }
  switch (a.dtype) {
    case RAI_F32: return launch_decode<float>(st, a);
    case RAI_BF16: return launch_decode<bf16_raw>(st, a);
    default: return fail(RAI_ERR_BAD_DTYPE, "attention decode: dtype %s unsupported", dtype_name(a.dtype));
  }
}

template <typename T> static int launch_row(hipStream_t st, const AttnArgs &a) {
  constexpr int V = AttnVec<T>::V;
  RAI_REQUIRE(a.D % V == 0 && a.D / V <= 256, RAI_ERR_BAD_SHAPE, "attention: head_dim %d unsupported", a.D);
  const int ncol = a.D / V, groups = 256 / ncol;
  const size_t lds = sizeof(float) * ((size_t)a.D + (size_t)groups * a.D + (size_t)(a.window > 0 && a.window < a.T ? a.window : a.T));
  RAI_REQUIRE(lds <= 150 * 1024, RAI_ERR_UNSUPPORTED, "attention: context %d too long for the row kernel", a.T);
  static size_t attr_bytes = 0;
  if (lds > 64 * 1024 && lds > attr_bytes) {
    RAI_HIP_TRY(hipFuncSetAttribute((const void *)k_attn_row<T>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                    150 * 1024));
    attr_bytes = 150 * 1024;
  }
  RAI_REQUIRE(a.Hq <= 65535 && a.B <= 65535, RAI_ERR_UNSUPPORTED, "attention: grid too large");
  hipLaunchKernelGGL((k_attn_row<T>), dim3(a.S, a.Hq, a.B), dim3(256), lds, st, a);
  return launch_check("attention_row");
}

int launch_attention(hipStream_t st, const AttnArgs &a) {
  RAI_REQUIRE(a.B > 0 && a.Hq > 0 && a.Hkv > 0 && a.S > 0 && a.T > 0 && a.D > 0, RAI_ERR_BAD_SHAPE,
              "attention: empty problem");
  RAI_REQUIRE(a.Hq % a.Hkv == 0, RAI_ERR_BAD_SHAPE, "attention: %d query heads not divisible by %d kv heads", a.Hq,
              a.Hkv);
  RAI_REQUIRE(a.window >= 0 && (!a.window || a.causal) && (a.f32_scores || (!a.gate && !a.sink && a.softcap <= 0.f)), RAI_ERR_BAD_ARG,
              "attention: a window needs the causal form, an output gate, a cap or a sink the f32-score form");
  if (flash_serves(a)) return launch_flash_prefill(st, a);
  if (attention_f32_serves(a)) return launch_attention_f32(st, a);
  switch (a.dtype) {
    case RAI_F32: return launch_row<float>(st, a);
    case RAI_BF16: return launch_row<bf16_raw>(st, a);
    case RAI_F16: return launch_row<f16_raw>(st, a);
    default: return fail(RAI_ERR_BAD_DTYPE, "attention: dtype %s unsupported", dtype_name(a.dtype));
  }
}

}  // namespace rai

using namespace rai;

extern "C" int rai_hip_attention(int dev, const rai_hip_tensor *q, const rai_hip_tensor *k, const rai_hip_tensor *v,
                                 double scale, int32_t causal, int32_t f32_scores, const rai_hip_tensor *out) {
  RAI_TRY(validate(q, "q"));
  RAI_TRY(validate(k, "k"));
  RAI_TRY(validate(v, "v"));
  RAI_TRY(validate(out, "out"));
  RAI_REQUIRE(q->rank == 4 && k->rank == 4 && v->rank == 4 && out->rank == 3, RAI_ERR_BAD_SHAPE,
              "attention: q/k/v must be rank 4 and out rank 3");
  RAI_REQUIRE(q->dtype == k->dtype && q->dtype == v->dtype && q->dtype == out->dtype, RAI_ERR_BAD_DTYPE,
              "attention: dtype mismatch");
  const int64_t B = q->shape[0], Hq = q->shape[1], S = q->shape[2], D = q->shape[3];
  const int64_t Hkv = k->shape[1], T = k->shape[2];
  RAI_REQUIRE(k->shape[0] == B && v->shape[0] == B && k->shape[3] == D && v->shape[3] == D && v->shape[1] == Hkv &&
                  v->shape[2] == T,
              RAI_ERR_BAD_SHAPE, "attention: k/v shapes do not match q");
  RAI_REQUIRE(out->shape[0] == B && out->shape[1] == S && out->shape[2] == Hq * D && is_contiguous(out),
              RAI_ERR_BAD_SHAPE, "attention: out must be contiguous [B, S, Hq*D]");
  RAI_REQUIRE((q->stride[3] == 1 && k->stride[3] == 1 && v->stride[3] == 1) || D == 1, RAI_ERR_BAD_STRIDE,
              "attention: head_dim must have unit stride");
  RAI_REQUIRE(!causal || S <= T, RAI_ERR_BAD_SHAPE, "attention: causal needs S <= T");
  hipStream_t st = stream_of(dev);
  if (!st) return RAI_ERR_HIP;
  if (numel(out) == 0) return RAI_OK;
  const size_t es = dtype_size(q->dtype);
  const int vec = (int)(16 / es);
  auto ok = [&](const rai_hip_tensor *t) {
    if ((uintptr_t)base_ptr(t) % 16) return false;
    for (int i = 0; i < 3; ++i)
      if (t->shape[i] > 1 && t->stride[i] % vec) return false;
    return true;
  };
  RAI_REQUIRE(ok(k) && ok(v) && D % vec == 0, RAI_ERR_BAD_STRIDE, "attention: k/v rows must be 16-byte aligned");
  AttnArgs a;
  memset(&a, 0, sizeof(a));
  a.q = base_ptr(q); a.k = base_ptr(k); a.v = base_ptr(v); a.out = base_ptr(out);
  for (int i = 0; i < 3; ++i) { a.qs[i] = q->stride[i]; a.ks[i] = k->stride[i]; a.vs[i] = v->stride[i]; }
  a.out_row_stride = Hq * D;
  a.B = (int)B; a.Hq = (int)Hq; a.Hkv = (int)Hkv; a.S = (int)S; a.T = (int)T; a.D = (int)D;
  a.scale = (float)scale; a.causal = causal; a.f32_scores = f32_scores; a.dtype = q->dtype;
  return launch_attention(st, a);
}
