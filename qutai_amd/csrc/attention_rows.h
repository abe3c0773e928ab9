// One wave per row: attention for any head dimension up to 256, fp32 or bf16
// storage of any alignment, fp32 math (the reference's warp kernels
// lm_attention / lm_attention_delta / lm_attention_backward_q / _kv,
// src/qutai/backends/cuda/lm.cu:65-87 and :289-343).  One wave computes a
// query row (forward, dq) or key row (dk, dv); lane l owns dimensions l,
// l + 64, l + 128, l + 192; dot products are wave-wide sums.  Bound by the
// cross-lane sums of every score, so it serves the rows that the matrix
// kernels (attention_mma.h) leave: rows that are not 16-byte aligned,
// sequences of a few positions, and waves whose operands hold an infinity or
// a NaN.
#pragma once
#include "attention_common.h"

namespace {

struct AttnGenArgs {
  const void* g;
  const void* q;
  const void* k;
  const void* v;
  const void* o;
  float* lse;
  float* delta;
  void* dq;  // forward: the output
  void* dk;
  void* dv;
  int64_t batch, heads, kv_heads, time, dim;
  int64_t qb, qh, qt, kb, kh, kt, lb, lh, lt;
  float scale;
  float scale_log2, scale_log2_lo;  // scale * log2(e) and its rounding error
  int causal;
  // split: each dK/dV workgroup takes one query head of its kv head's group
  // and writes unscaled fp32 partials to part_k / part_v + head * part_stride
  // (dk's element offsets); dkv_sum adds them up
  int split;
  float* part_k;
  float* part_v;
  int64_t part_stride;
};

template <class T> __device__ __forceinline__ float ld(const void* p, int64_t i);
template <> __device__ __forceinline__ float ld<float>(const void* p, int64_t i) { return ((const float*)p)[i]; }
template <> __device__ __forceinline__ float ld<bf16_t>(const void* p, int64_t i) {
  return bf16_to_f32(((const bf16_t*)p)[i]);
}
template <class T> __device__ __forceinline__ void st(void* p, int64_t i, float x);
template <> __device__ __forceinline__ void st<float>(void* p, int64_t i, float x) { ((float*)p)[i] = x; }
template <> __device__ __forceinline__ void st<bf16_t>(void* p, int64_t i, float x) {
  ((bf16_t*)p)[i] = f32_to_bf16(x);
}

__device__ __forceinline__ float wave_sum(float x) {
#pragma unroll
  for (int off = 32; off; off >>= 1) x += __shfl_xor(x, off);
  return x;
}

constexpr int GEN_WAVES = 4;  // rows per workgroup

// row -> (b, h, t) and its element offset in a q-shaped array
__device__ __forceinline__ void gen_row(const AttnGenArgs& p, int64_t row, int64_t heads, int64_t& b, int64_t& h,
                                        int64_t& t) {
  t = row % p.time;
  h = (row / p.time) % heads;
  b = row / (p.time * heads);
}

// Output and lse of query t of (b, h).
template <class T>
__device__ __forceinline__ void fwd_row(const AttnGenArgs& p, int64_t b, int64_t h, int64_t t, int lane) {
  const int64_t kvh = h / (p.heads / p.kv_heads);
  const int64_t qi = b * p.qb + h * p.qh + t * p.qt, kbase = b * p.kb + kvh * p.kh;
  const int D = (int)p.dim;
  float qv[4], acc[4];
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const int d = lane + 64 * j;
    qv[j] = d < D ? ld<T>(p.q, qi + d) : 0.f;
    acc[j] = 0.f;
  }
  float m = -INFINITY, l = 0.f;
  const int64_t end = p.causal ? t + 1 : p.time;
  for (int64_t s = 0; s < end; s++) {
    const int64_t ki = kbase + s * p.kt;
    float dot = 0.f;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int d = lane + 64 * j;
      if (d < D) dot += qv[j] * ld<T>(p.k, ki + d);
    }
    const float x = wave_sum(dot) * p.scale;
    const float m_new = fmaxf(m, x);
    const float alpha = __expf(m - m_new), pr = __expf(x - m_new);
    l = l * alpha + pr;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int d = lane + 64 * j;
      acc[j] = acc[j] * alpha + (d < D ? pr * ld<T>(p.v, ki + d) : 0.f);
    }
    m = m_new;
  }
  const float inv = l > 0.f ? 1.f / l : 0.f;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const int d = lane + 64 * j;
    if (d < D) st<T>(p.dq, qi + d, acc[j] * inv);
  }
  if (p.lse && lane == 0) p.lse[b * p.lb + h * p.lh + t * p.lt] = m + __logf(l);
}

// dQ and delta of query t of (b, h).
template <class T>
__device__ __forceinline__ void bwd_q_row(const AttnGenArgs& p, int64_t b, int64_t h, int64_t t, int lane) {
  const int64_t kvh = h / (p.heads / p.kv_heads);
  const int64_t qi = b * p.qb + h * p.qh + t * p.qt, kbase = b * p.kb + kvh * p.kh;
  const int64_t li = b * p.lb + h * p.lh + t * p.lt;
  const int D = (int)p.dim;
  float qv[4], gv[4], acc[4], dl = 0.f;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const int d = lane + 64 * j;
    qv[j] = d < D ? ld<T>(p.q, qi + d) : 0.f;
    gv[j] = d < D ? ld<T>(p.g, qi + d) : 0.f;
    dl += d < D ? gv[j] * ld<T>(p.o, qi + d) : 0.f;
    acc[j] = 0.f;
  }
  dl = wave_sum(dl);
  if (lane == 0) p.delta[li] = dl;
  const float lse = p.lse[li];
  const int64_t end = p.causal ? t + 1 : p.time;
  for (int64_t s = 0; s < end; s++) {
    const int64_t ki = kbase + s * p.kt;
    float dot = 0.f, dp = 0.f;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int d = lane + 64 * j;
      if (d < D) {
        dot += qv[j] * ld<T>(p.k, ki + d);
        dp += gv[j] * ld<T>(p.v, ki + d);
      }
    }
    const float pr = __expf(wave_sum(dot) * p.scale - lse);
    const float ds = pr * (wave_sum(dp) - dl) * p.scale;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int d = lane + 64 * j;
      if (d < D) acc[j] += ds * ld<T>(p.k, ki + d);
    }
  }
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const int d = lane + 64 * j;
    if (d < D) st<T>(p.dq, qi + d, acc[j]);
  }
}

// dK and dV of key s of (b, kvh), summed over the query heads [g_lo, g_hi) of
// its group (p.split: head g_lo's unscaled partials).
template <class T>
__device__ __forceinline__ void bwd_kv_row(const AttnGenArgs& p, int64_t b, int64_t kvh, int64_t s, int lane,
                                           int g_lo, int g_hi) {
  const int64_t ki = b * p.kb + kvh * p.kh + s * p.kt;
  const int64_t group = p.heads / p.kv_heads;
  const int D = (int)p.dim;
  const float scale = p.split ? 1.f : p.scale;
  float kv_[4], vv[4], ak[4], av[4];
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const int d = lane + 64 * j;
    kv_[j] = d < D ? ld<T>(p.k, ki + d) : 0.f;
    vv[j] = d < D ? ld<T>(p.v, ki + d) : 0.f;
    ak[j] = av[j] = 0.f;
  }
  for (int64_t h = kvh * group + g_lo; h < kvh * group + g_hi; h++) {
    for (int64_t t = p.causal ? s : 0; t < p.time; t++) {
      const int64_t qi = b * p.qb + h * p.qh + t * p.qt;
      const int64_t li = b * p.lb + h * p.lh + t * p.lt;
      float dot = 0.f, dp = 0.f;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const int d = lane + 64 * j;
        if (d < D) {
          dot += ld<T>(p.q, qi + d) * kv_[j];
          dp += ld<T>(p.g, qi + d) * vv[j];
        }
      }
      const float pr = __expf(wave_sum(dot) * p.scale - p.lse[li]);
      const float ds = pr * (wave_sum(dp) - p.delta[li]) * scale;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const int d = lane + 64 * j;
        if (d < D) {
          ak[j] += ds * ld<T>(p.q, qi + d);
          av[j] += pr * ld<T>(p.g, qi + d);
        }
      }
    }
  }
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const int d = lane + 64 * j;
    if (d < D) {
      if (p.split) {
        p.part_k[g_lo * p.part_stride + ki + d] = ak[j];
        p.part_v[g_lo * p.part_stride + ki + d] = av[j];
      } else {
        st<T>(p.dk, ki + d, ak[j]);
        st<T>(p.dv, ki + d, av[j]);
      }
    }
  }
}

template <class T>
__global__ void __launch_bounds__(GEN_WAVES * 64) attention_fwd_rows(AttnGenArgs p) {
  const int64_t row = (int64_t)blockIdx.x * GEN_WAVES + (threadIdx.x >> 6);
  if (row >= p.batch * p.heads * p.time) return;  // whole wave
  int64_t b, h, t;
  gen_row(p, row, p.heads, b, h, t);
  fwd_row<T>(p, b, h, t, threadIdx.x & 63);
}

template <class T>
__global__ void __launch_bounds__(GEN_WAVES * 64) attention_bwd_q_rows(AttnGenArgs p) {
  const int64_t row = (int64_t)blockIdx.x * GEN_WAVES + (threadIdx.x >> 6);
  if (row >= p.batch * p.heads * p.time) return;
  int64_t b, h, t;
  gen_row(p, row, p.heads, b, h, t);
  bwd_q_row<T>(p, b, h, t, threadIdx.x & 63);
}

template <class T>
__global__ void __launch_bounds__(GEN_WAVES * 64) attention_bwd_kv_rows(AttnGenArgs p) {
  const int64_t row = (int64_t)blockIdx.x * GEN_WAVES + (threadIdx.x >> 6);
  if (row >= p.batch * p.kv_heads * p.time) return;
  int64_t b, kvh, s;
  gen_row(p, row, p.kv_heads, b, kvh, s);
  bwd_kv_row<T>(p, b, kvh, s, threadIdx.x & 63, 0, (int)(p.heads / p.kv_heads));
}

}  // namespace
