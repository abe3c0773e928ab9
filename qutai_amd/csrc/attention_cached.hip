// Attention of a few new positions over a key/value cache (generation step):
// C ABI `qutai_amd_attention_cached`.  The products of
// MultiHeadAttention's cache path (scores, offset causal mask, softmax, values;
// src/qutai/nn/layers.py:345-355) in one launch, with the scores, the
// probabilities and all sums in fp32.
//
// A workgroup of 16 waves owns one query of one (batch, head).  A row of K or V
// is read by G lanes of 16 bytes, so a wave reads 64 / G rows at a time and has
// four such reads in flight:
//  1. scores of the visible keys into LDS (a lane's 16-byte share of the dot
//     product, summed over the G lanes of a row);
//  2. their maximum and the sum of exponentials;
//  3. every row group sums its keys' probability times V in registers, and the
//     groups and waves are added up through LDS in a fixed order.
// Bound by latency and by the K and V reads of its CU.  One query, bf16, eight
// batches of 16 heads of 64, 1001 keys (33 MB): 8.9 us a call, against 102 us for
// the transposed copy of the keys, two products, mask and softmax (52 us of it in
// kernels).  A CU alone draws 67 GB/s with 16 waves, 35 with eight (12000 keys of
// 128: 92 against 172 us); eight reads in flight give 3 % there and cost 25 % at
// eight queries.
#include "attention_common.h"

namespace {

constexpr int CW = 16;                   // waves
constexpr int64_t CACHED_KEYS = 12000;  // their scores fit beside the partial sums (at most 16 KiB) in 64 KiB of LDS

struct CachedArgs {
  const void* q;
  const void* k;
  const void* v;
  void* out;
  int64_t pairs, heads, length, total, dim;  // pairs: (batch, head)
  float scale;
};

// E elements of one 16-byte chunk as floats
template <bool F32>
__device__ __forceinline__ void chunk_values(const u32x4& w, float (&v)[F32 ? 4 : 8]) {
#pragma unroll
  for (int e = 0; e < (F32 ? 4 : 8); e++) {
    if constexpr (F32) v[e] = __uint_as_float(w[e]);
    else v[e] = __uint_as_float((e & 1) ? (w[e >> 1] & 0xffff0000u) : (w[e >> 1] << 16));
  }
}

// G lanes per row, the smallest power of two whose 16-byte chunks hold a row.
template <bool F32, int G>
__global__ void __launch_bounds__(CW * 64) attention_cached(CachedArgs p) {
  constexpr int E = F32 ? 4 : 8, ES = F32 ? 4 : 2, ROWS = 64 / G, DEEP = 4;
  extern __shared__ __attribute__((aligned(16))) float lds[];
  float* scores = lds;                                  // [total rounded up to 64]
  float* sums = lds + (p.total + 63) / 64 * 64;          // [CW][G * E], and CW values of the reductions
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, part = lane % G, row = lane / G;
  // the queries of a head sit eight workgroups apart, on one XCD, whose L2 then holds the head's keys and
  // values (eight queries of the shape above 38 -> 18 us with eight waves)
  const int64_t group = blockIdx.x / (8 * p.length), rest = blockIdx.x % (8 * p.length);
  const int64_t width = p.pairs - 8 * group < 8 ? p.pairs - 8 * group : 8;
  const int64_t query = rest / width, bh = 8 * group + rest % width, b = bh / p.heads, h = bh % p.heads;
  const int visible = (int)(p.total - p.length + query + 1);
  const bool in = part * E < p.dim;
  const int64_t q_at = ((b * p.length + query) * p.heads + h) * p.dim;
  const char* K = (const char*)p.k + bh * p.total * p.dim * ES + part * 16;
  const char* V = (const char*)p.v + bh * p.total * p.dim * ES + part * 16;
  const int64_t stride = p.dim * ES;

  float qv[E];
  {
    u32x4 w = {0u, 0u, 0u, 0u};
    if (in) w = global_load<u32x4>((const char*)p.q + q_at * ES + part * 16);
    chunk_values<F32>(w, qv);
  }
  // ---- scores
  float top = -INFINITY;
  for (int s0 = wave * ROWS; s0 < visible; s0 += CW * ROWS * DEEP) {
    u32x4 w[DEEP];
#pragma unroll
    for (int u = 0; u < DEEP; u++) {
      const int s = s0 + u * CW * ROWS + row;
      w[u] = u32x4{0u, 0u, 0u, 0u};
      if (in && s < visible) w[u] = global_load<u32x4>(K + s * stride);
    }
#pragma unroll
    for (int u = 0; u < DEEP; u++) {
      const int s = s0 + u * CW * ROWS + row;
      float kv[E], dot = 0.f;
      chunk_values<F32>(w[u], kv);
#pragma unroll
      for (int e = 0; e < E; e++) dot = __builtin_fmaf(qv[e], kv[e], dot);
#pragma unroll
      for (int o = G / 2; o; o >>= 1) dot += __shfl_xor(dot, o);
      dot *= p.scale;
      if (s < visible) {
        if (part == 0) scores[s] = dot;
        top = fmaxf(top, dot);
      }
    }
  }
  // ---- maximum over the workgroup, then the exponentials and their sum
#pragma unroll
  for (int o = 32; o; o >>= 1) top = fmaxf(top, __shfl_xor(top, o));
  float* shared = sums + CW * G * E;
  if (lane == 0) shared[wave] = top;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < CW; w++) top = fmaxf(top, shared[w]);
  float total = 0.f;
  for (int s = tid; s < visible; s += CW * 64) {
    const float x = __expf(scores[s] - top);
    scores[s] = x;
    total += x;
  }
#pragma unroll
  for (int o = 32; o; o >>= 1) total += __shfl_xor(total, o);
  __syncthreads();  // every wave has read the maxima; the exponentials are written
  if (lane == 0) shared[wave] = total;
  // ---- values
  float acc[E];
#pragma unroll
  for (int e = 0; e < E; e++) acc[e] = 0.f;
  for (int s0 = wave * ROWS; s0 < visible; s0 += CW * ROWS * DEEP) {
    u32x4 w[DEEP];
#pragma unroll
    for (int u = 0; u < DEEP; u++) {
      const int s = s0 + u * CW * ROWS + row;
      w[u] = u32x4{0u, 0u, 0u, 0u};
      if (in && s < visible) w[u] = global_load<u32x4>(V + s * stride);
    }
#pragma unroll
    for (int u = 0; u < DEEP; u++) {
      const int s = s0 + u * CW * ROWS + row;
      const float x = s < visible ? scores[s] : 0.f;
      float vv[E];
      chunk_values<F32>(w[u], vv);
#pragma unroll
      for (int e = 0; e < E; e++) acc[e] = __builtin_fmaf(x, vv[e], acc[e]);
    }
  }
#pragma unroll
  for (int e = 0; e < E; e++)
#pragma unroll
    for (int o = G; o < 64; o <<= 1) acc[e] += __shfl_xor(acc[e], o);
  if (row == 0) {
#pragma unroll
    for (int e = 0; e < E; e++) sums[(wave * G + part) * E + e] = acc[e];
  }
  __syncthreads();
  if (tid < p.dim) {
    float y = 0.f, n = 0.f;
#pragma unroll
    for (int w = 0; w < CW; w++) {
      y += sums[w * G * E + tid];
      n += shared[w];
    }
    y /= n;
    if constexpr (F32) ((float*)p.out)[q_at + tid] = y;
    else ((bf16_t*)p.out)[q_at + tid] = f32_to_bf16(y);
  }
}

// Keys and values of earlier positions and of new ones joined along the length
// axis, both caches in one launch.  A workgroup moves up to 4 KiB x 4 of one
// (batch, head)'s row of 16-byte chunks, four loads in flight per lane, with all
// divisions on scalars.  HBM-bound; a generation step's cache is small enough
// that its launches cost more: four strided copies before (two per cache).  8
// sequences, 16 heads of 64, 1000 cached positions, bf16 (66 MB moved): a layer
// call 160 -> 138 us.
constexpr int JOIN_THREADS = 256, JOIN_DEEP = 4;

struct JoinArgs {
  const u32x4* past[2];
  const u32x4* fresh[2];
  u32x4* out[2];
  uint32_t rows, segments, past_chunks, new_chunks;  // chunks of 16 bytes per row
};

__global__ void __launch_bounds__(JOIN_THREADS) cache_join(JoinArgs p) {
  const uint32_t line = blockIdx.x / p.segments, segment = blockIdx.x - line * p.segments;
  const uint32_t which = line >= p.rows ? 1 : 0;
  const int64_t row = line - which * p.rows;
  const uint32_t chunks = p.past_chunks + p.new_chunks;
  const u32x4* past = p.past[which] + row * p.past_chunks;
  const u32x4* fresh = p.fresh[which] + row * p.new_chunks;
  u32x4* out = p.out[which] + row * chunks;
  const uint32_t first = segment * (JOIN_THREADS * JOIN_DEEP) + threadIdx.x;
  u32x4 v[JOIN_DEEP];
#pragma unroll
  for (int u = 0; u < JOIN_DEEP; u++) {
    const uint32_t c = first + u * JOIN_THREADS;
    if (c < chunks) v[u] = global_load<u32x4>(c < p.past_chunks ? past + c : fresh + (c - p.past_chunks));
  }
#pragma unroll
  for (int u = 0; u < JOIN_DEEP; u++) {
    const uint32_t c = first + u * JOIN_THREADS;
    if (c < chunks) global_store(out + c, v[u]);
  }
}

template <bool F32, int G>
void launch(const CachedArgs& a, unsigned blocks, hipStream_t stream) {
  const size_t bytes = ((a.total + 63) / 64 * 64 + CW * G * (F32 ? 4 : 8) + CW) * sizeof(float);
  hipLaunchKernelGGL((attention_cached<F32, G>), dim3(blocks), dim3(CW * 64), bytes, stream, a);
}

}  // namespace

extern "C" int qutai_amd_attention_cached(const void* q, const void* k, const void* v, void* out, int64_t batch,
                                          int64_t heads, int64_t length, int64_t total, int64_t dim, int dtype,
                                          double scale, void* stream_) {
  if (batch < 0 || heads <= 0 || length <= 0 || total < length || dim <= 0 || dim > 256) return QA_EINVAL;
  if ((dtype != BF16 && dtype != F32) || dim % (dtype == F32 ? 4 : 8)) return QA_EINVAL;
  // a launch holds fewer than 2^32 threads: 2^22 workgroups of 16 waves are too many
  if (total > CACHED_KEYS || heads > 65536 || batch > 0x3fffff / heads / length || !(scale > 0.0) || scale > 1e30)
    return QA_EINVAL;
  if (batch == 0) return QA_OK;
  if (!aligned16({q, k, v, out})) return QA_EINVAL;
  const CachedArgs a = {q, k, v, out, batch * heads, heads, length, total, dim, (float)scale};
  const unsigned blocks = (unsigned)(batch * heads * length);
  hipStream_t stream = (hipStream_t)stream_;
  if (dtype == F32) {
    if (dim <= 32) launch<true, 8>(a, blocks, stream);
    else if (dim <= 64) launch<true, 16>(a, blocks, stream);
    else if (dim <= 128) launch<true, 32>(a, blocks, stream);
    else launch<true, 64>(a, blocks, stream);
  } else {
    if (dim <= 32) launch<false, 4>(a, blocks, stream);
    else if (dim <= 64) launch<false, 8>(a, blocks, stream);
    else if (dim <= 128) launch<false, 16>(a, blocks, stream);
    else launch<false, 32>(a, blocks, stream);
  }
  return (int)hipGetLastError();
}

extern "C" int qutai_amd_cache_join(const void* past_k, const void* past_v, const void* new_k, const void* new_v,
                                    void* out_k, void* out_v, int64_t rows, int64_t past_bytes, int64_t new_bytes,
                                    void* stream_) {
  if (rows < 0 || past_bytes < 0 || new_bytes < 0 || past_bytes % 16 || new_bytes % 16) return QA_EINVAL;
  if (past_bytes > (1ll << 34) || new_bytes > (1ll << 34)) return QA_EINVAL;  // a row's chunks stay below 2^31
  const int64_t chunks = (past_bytes + new_bytes) / 16, segments = (chunks + JOIN_THREADS * JOIN_DEEP - 1) / (JOIN_THREADS * JOIN_DEEP);
  if (rows == 0 || chunks == 0) return QA_OK;
  if (rows > 0x7fffff / segments) return QA_EINVAL;  // 2 x rows x segments workgroups of 256 threads, below 2^32 threads
  if ((past_bytes && !aligned16({past_k, past_v})) || (new_bytes && !aligned16({new_k, new_v})) ||
      !aligned16({out_k, out_v}))
    return QA_EINVAL;
  const JoinArgs a = {{(const u32x4*)past_k, (const u32x4*)past_v}, {(const u32x4*)new_k, (const u32x4*)new_v},
                      {(u32x4*)out_k, (u32x4*)out_v}, (uint32_t)rows, (uint32_t)segments,
                      (uint32_t)(past_bytes / 16), (uint32_t)(new_bytes / 16)};
  hipLaunchKernelGGL(cache_join, dim3((unsigned)(2 * rows * segments)), dim3(JOIN_THREADS), 0, (hipStream_t)stream_, a);
  return (int)hipGetLastError();
}
