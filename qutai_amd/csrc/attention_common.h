// Helpers shared by the attention kernels of attention.hip (bf16, D = 64) and
// attention_general.hip (every other head width and fp32 storage).
#pragma once
#include "common.h"
#include "qutai_amd.h"

#include <initializer_list>

using namespace qa;

namespace {

constexpr float LOG2E = 1.4426950408889634f;
constexpr float LOG2E_LO = (float)(1.4426950408889634 - (double)LOG2E);

// Both halves of the wavefront (lanes l and l ^ 32) hold the same query:
// the gfx950 half swap exchanges them without LDS.
__device__ __forceinline__ float pair_max(float x) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float pair_sum(float x) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// element strides of (batch, head, token) for q-shaped, kv-shaped and lse arrays
template <class Args>
int set_layout(Args& a, int64_t batch, int64_t heads, int64_t kv_heads, int64_t time, int64_t dim, int layout) {
  if (batch < 0 || heads <= 0 || kv_heads <= 0 || heads % kv_heads || time < 0 || dim <= 0) return QA_EINVAL;
  if (layout != 0 && layout != 1) return QA_EINVAL;
  if (time > (1 << 30) / (heads > kv_heads ? heads : kv_heads) / dim) return QA_EINVAL;  // 32-bit element offsets
  a.batch = batch;
  a.heads = heads;
  a.kv_heads = kv_heads;
  a.time = time;
  if (layout == 0) {  // [batch][heads][time][dim]
    a.qb = heads * time * dim, a.qh = time * dim, a.qt = dim;
    a.kb = kv_heads * time * dim, a.kh = time * dim, a.kt = dim;
    a.lb = heads * time, a.lh = time, a.lt = 1;
  } else {            // [batch][time][heads][dim] (the lm layout)
    a.qb = time * heads * dim, a.qh = dim, a.qt = heads * dim;
    a.kb = time * kv_heads * dim, a.kh = dim, a.kt = kv_heads * dim;
    a.lb = time * heads, a.lh = 1, a.lt = heads;
  }
  return QA_OK;
}

int64_t cu_count() {
  static int cached[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (!cached[dev]) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cached[dev] = n;
  }
  return cached[dev];
}

bool aligned16(std::initializer_list<const void*> ptrs) {
  for (const void* ptr : ptrs)
    if (!ptr || (uintptr_t)ptr % 16) return false;
  return true;
}

}  // namespace

// The general path (attention_general.hip); arguments checked by the C entry
// points for null pointers and the scale's range.
int attention_general_fwd(const void* q, const void* k, const void* v, void* out, float* lse, int64_t batch,
                          int64_t heads, int64_t kv_heads, int64_t time, int64_t dim, int dtype, int layout,
                          double scale, int causal, hipStream_t stream);
size_t attention_general_workspace(int64_t batch, int64_t heads, int64_t kv_heads, int64_t time, int64_t dim,
                                   int dtype);
int attention_general_bwd(const void* grad, const void* q, const void* k, const void* v, const void* out,
                          const float* lse, void* dq, void* dk, void* dv, float* delta, void* workspace,
                          size_t workspace_bytes, int64_t batch, int64_t heads, int64_t kv_heads, int64_t time,
                          int64_t dim, int dtype, int layout, double scale, int causal, hipStream_t stream);
