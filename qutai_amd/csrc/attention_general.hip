// Attention forward and backward for every head width and storage type but
// bf16 with D = 64 (attention.hip): on the matrix cores where rows are
// 16-byte aligned (attention_mma.h), one wave per row otherwise
// (attention_rows.h).
#include <algorithm>
#include <type_traits>

#include "attention_rows.h"
#include "attention_mma.h"

namespace {

// dK = scale * sum_g part_k[g], dV = sum_g part_v[g] (g in order), one
// rounding to the storage type; 4 elements per lane and step.
template <bool F32>
__global__ void dkv_sum(AttnGenArgs p, int64_t n4, int group) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n4; i += (int64_t)gridDim.x * blockDim.x) {
    f32x4 sk = global_load<f32x4>(p.part_k + 4 * i), sv = global_load<f32x4>(p.part_v + 4 * i);
    for (int g = 1; g < group; g++) {
      sk += global_load<f32x4>(p.part_k + g * p.part_stride + 4 * i);
      sv += global_load<f32x4>(p.part_v + g * p.part_stride + 4 * i);
    }
    put4<F32>(p.dk, 4 * i, sk * p.scale);
    put4<F32>(p.dv, 4 * i, sv);
  }
}

enum Pass { FORWARD, QUERIES, KEYS };

template <bool F32, int DP>
void launch_pass(Pass pass, const AttnGenArgs& a, unsigned blocks, hipStream_t stream) {
  const dim3 grid(blocks), block(256);
  if (pass == FORWARD) hipLaunchKernelGGL((attention_fwd_mma<F32, DP>), grid, block, 0, stream, a);
  else if (pass == QUERIES) hipLaunchKernelGGL((attention_bwd_dq_mma<F32, DP>), grid, block, 0, stream, a);
  else if constexpr (DP > 128) {
    hipLaunchKernelGGL((attention_bwd_dkv_mma<F32, DP, KEYS_DV>), grid, block, 0, stream, a);
    hipLaunchKernelGGL((attention_bwd_dkv_mma<F32, DP, KEYS_DK>), grid, block, 0, stream, a);
  } else {
    hipLaunchKernelGGL((attention_bwd_dkv_mma<F32, DP, KEYS_BOTH>), grid, block, 0, stream, a);
  }
}

// The kernel width DP is the smallest built one that holds the head
// dimension: the MFMAs work on whole 32-wide d blocks.  fp32 above 128 would
// need more registers than a wave has (three parts of q and dO).
bool mma_fits(int dtype, int64_t dim) { return dtype == BF16 ? dim % 8 == 0 && dim <= 256 : dim % 4 == 0 && dim <= 128; }

// Whether 64 rows of every operand lie within the 2 GiB of a buffer descriptor,
// beyond which the kernels' loads read zeros (rows of 8 million fp32 values).
bool mma_spans(const AttnGenArgs& a, int dtype) {
  return 64 * std::max(a.qt, a.kt) * (dtype == F32 ? 4 : 2) <= 0x7ffffff0;
}

// A scale of the scores with which the factors that take the parts' scaling
// back (2^-48 at most) keep their bits: any in earnest use.
bool mma_scale(double scale) { return scale >= 0x1p-50; }

hipError_t launch_mma(Pass pass, int dtype, const AttnGenArgs& a, int64_t blocks, hipStream_t stream) {
  const unsigned n = (unsigned)blocks;
  if (dtype == BF16) {
    if (a.dim <= 32) launch_pass<false, 32>(pass, a, n, stream);
    else if (a.dim <= 96) launch_pass<false, 96>(pass, a, n, stream);
    else if (a.dim <= 128) launch_pass<false, 128>(pass, a, n, stream);
    else launch_pass<false, 256>(pass, a, n, stream);
  } else {
    if (a.dim <= 32) launch_pass<true, 32>(pass, a, n, stream);
    else if (a.dim <= 64) launch_pass<true, 64>(pass, a, n, stream);
    else if (a.dim <= 96) launch_pass<true, 96>(pass, a, n, stream);
    else launch_pass<true, 128>(pass, a, n, stream);
  }
  return hipGetLastError();
}

template <class Kernel>
hipError_t launch_rows(Kernel bf16, Kernel fp32, int dtype, const AttnGenArgs& a, int64_t rows, hipStream_t stream) {
  hipLaunchKernelGGL((dtype == BF16 ? bf16 : fp32), dim3((unsigned)((rows + GEN_WAVES - 1) / GEN_WAVES)),
                     dim3(GEN_WAVES * 64), 0, stream, a);
  return hipGetLastError();
}

// scale_log2 takes the scores of the matrix kernels, products of two stored
// values as they are scaled (AttnTile::STORED)
void set_scale(AttnGenArgs& a, double scale, int dtype) {
  a.scale = (float)scale;
  const double log2 = scale * 1.4426950408889634 * (dtype == F32 ? 0x1p-48 : 1.0);
  a.scale_log2 = (float)log2;
  a.scale_log2_lo = (float)(log2 - (double)a.scale_log2);
}

constexpr int64_t OWNED = 128;  // queries or keys of a workgroup

// Whether a call takes one wave per row although the matrix kernels could hold
// it: the tiles of a sequence of a few positions are mostly empty, and sums of
// one or two terms round best on their own.  Measured with 8000 and 16000 heads
// (us; rows, tiles), the lines lie at the crossings: forward bf16 D 32, T 6 72
// and 75; bf16 D 128, T 6 103 and 178, T 8 191 and 180; bf16 D 136, T 10 154 and
// 209, T 13 236 and 209; fp32 D 64, T 8 128 and 148, T 13 121 and 80 (8000); fp32
// D 96, T 10 116 and 181, T 13 179 and 182; fp32 D 128, T 13 181 and 218, T 16 357
// and 216.  Backward bf16 D 32, T 6 153 and 168, T 8 279 and 168; fp32 D 32, T 8
// 270 and 312; bf16 D 128, T 2 45 and 723, T 13 390 and 469 (8000); fp32 D 64,
// T 13 251 and 354; fp32 D 128, T 13 433 and 1021, T 20 885 and 1061.  Grids of
// fewer heads than the GPU holds at once take the tiles earlier (32 heads of
// 128, bf16: forward, T 3, 10 and 7.6; backward, T 4, 20 and 22, T 5 24 and 22).
bool few_positions(int dtype, int64_t batch, int64_t heads, int64_t kv_heads, int64_t time, int64_t dim,
                   bool backward) {
  const bool f32 = dtype == F32;
  int64_t most;
  if (dim <= 32) most = f32 ? (backward ? 8 : 7) : 6;
  else if (backward) most = f32 && dim > 96 && heads == kv_heads ? 20 : 13;
  else most = f32 ? (dim <= 64 ? 8 : 13) : dim <= 128 ? 8 : 10;
  return time <= (backward ? 4 : 2) || (time <= most && batch * heads >= 2 * cu_count());
}

// Partial dK/dV of the query heads of each kv head's group, for grids of
// fewer workgroups than the GPU holds at once (two per CU).
size_t split_bytes(int64_t batch, int64_t heads, int64_t kv_heads, int64_t time, int64_t dim) {
  if (kv_heads <= 0 || heads <= kv_heads || heads % kv_heads) return 0;
  if (batch * kv_heads * ((time + OWNED - 1) / OWNED) >= 2 * cu_count()) return 0;
  return (size_t)2 * (heads / kv_heads) * batch * time * kv_heads * dim * sizeof(float);
}

}  // namespace

int attention_general_fwd(const void* q, const void* k, const void* v, void* out, float* lse, int64_t batch,
                          int64_t heads, int64_t kv_heads, int64_t time, int64_t dim, int dtype, int layout,
                          double scale, int causal, hipStream_t stream) {
  if ((dtype != BF16 && dtype != F32) || dim > 256) return QA_EINVAL;
  AttnGenArgs a = {};
  if (set_layout(a, batch, heads, kv_heads, time, dim, layout) != QA_OK) return QA_EINVAL;
  if (batch * time == 0) return QA_OK;
  a.q = q;
  a.k = k;
  a.v = v;
  a.dq = out;
  a.lse = lse;
  a.dim = dim;
  set_scale(a, scale, dtype);
  a.causal = causal ? 1 : 0;
  const int64_t rows = batch * heads * time;
  if ((rows + GEN_WAVES - 1) / GEN_WAVES > 0x7fffffff) return QA_EINVAL;
  if (mma_fits(dtype, dim) && mma_scale(scale) && mma_spans(a, dtype) && aligned16({q, k, v, out}) &&
      !few_positions(dtype, batch, heads, kv_heads, time, dim, false))
    return (int)launch_mma(FORWARD, dtype, a, batch * heads * ((time + OWNED - 1) / OWNED), stream);
  return (int)launch_rows(attention_fwd_rows<bf16_t>, attention_fwd_rows<float>, dtype, a, rows, stream);
}

size_t attention_general_workspace(int64_t batch, int64_t heads, int64_t kv_heads, int64_t time, int64_t dim,
                                   int dtype) {
  if ((dtype != BF16 && dtype != F32) || dim <= 0 || batch < 0 || time < 0 || !mma_fits(dtype, dim)) return 0;
  if (few_positions(dtype, batch, heads, kv_heads, time, dim, true)) return 0;
  return split_bytes(batch, heads, kv_heads, time, dim);
}

int attention_general_bwd(const void* grad, const void* q, const void* k, const void* v, const void* out,
                          const float* lse, void* dq, void* dk, void* dv, float* delta, void* workspace,
                          size_t workspace_bytes, int64_t batch, int64_t heads, int64_t kv_heads, int64_t time,
                          int64_t dim, int dtype, int layout, double scale, int causal, hipStream_t stream) {
  if ((dtype != BF16 && dtype != F32) || dim > 256) return QA_EINVAL;
  AttnGenArgs a = {};
  if (set_layout(a, batch, heads, kv_heads, time, dim, layout) != QA_OK) return QA_EINVAL;
  if (batch * time == 0) return QA_OK;
  a.g = grad;
  a.q = q;
  a.k = k;
  a.v = v;
  a.o = out;
  a.lse = const_cast<float*>(lse);
  a.delta = delta;
  a.dq = dq;
  a.dk = dk;
  a.dv = dv;
  a.dim = dim;
  set_scale(a, scale, dtype);
  a.causal = causal ? 1 : 0;
  const int64_t q_rows = batch * heads * time, k_rows = batch * kv_heads * time;
  if ((q_rows + GEN_WAVES - 1) / GEN_WAVES > 0x7fffffff) return QA_EINVAL;
  // the q pass writes delta, which the kv pass reads
  if (!mma_fits(dtype, dim) || !mma_scale(scale) || !mma_spans(a, dtype) ||
      !aligned16({grad, q, k, v, out, dq, dk, dv}) ||
      few_positions(dtype, batch, heads, kv_heads, time, dim, true)) {
    const hipError_t e =
        launch_rows(attention_bwd_q_rows<bf16_t>, attention_bwd_q_rows<float>, dtype, a, q_rows, stream);
    if (e != hipSuccess) return (int)e;
    return (int)launch_rows(attention_bwd_kv_rows<bf16_t>, attention_bwd_kv_rows<float>, dtype, a, k_rows, stream);
  }
  const int64_t blocks = (time + OWNED - 1) / OWNED, group = heads / kv_heads;
  const size_t need = split_bytes(batch, heads, kv_heads, time, dim);
  if (need && workspace && workspace_bytes >= need && (uintptr_t)workspace % 16 == 0) {
    a.split = 1;
    a.part_stride = batch * time * kv_heads * dim;
    a.part_k = (float*)workspace;
    a.part_v = a.part_k + group * a.part_stride;
  }
  hipError_t e = launch_mma(QUERIES, dtype, a, batch * heads * blocks, stream);
  if (e != hipSuccess) return (int)e;
  e = launch_mma(KEYS, dtype, a, batch * kv_heads * blocks * (a.split ? group : 1), stream);
  if (e != hipSuccess || !a.split) return (int)e;
  const int64_t n4 = a.part_stride / 4;
  const unsigned grid = (unsigned)std::min<int64_t>((n4 + 255) / 256, 1 << 20);
  if (dtype == BF16) hipLaunchKernelGGL(dkv_sum<false>, dim3(grid), dim3(256), 0, stream, a, n4, (int)group);
  else hipLaunchKernelGGL(dkv_sum<true>, dim3(grid), dim3(256), 0, stream, a, n4, (int)group);
  return (int)hipGetLastError();
}
