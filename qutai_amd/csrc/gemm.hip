// GEMM entry points of libqutai_amd (C ABI).  The argument meaning, the
// dtype rules and the validation follow the reference GEMM boundary
// `cuda.gemm` (src/qutai/backends/cuda.py:305-362) and its kernel signature
// (src/qutai/backends/cuda/gemm.cu:35, `(a, b, out, M, K, N, sa, sb, ta, tb,
// accumulate)`); kernel choice is MI355X-specific.
#include <cstdlib>
#include <string>

#include "gemm_kernel.h"
#include "gemm_pingpong.h"
#include "gemm_short.h"

#include <algorithm>
#include "qutai_amd.h"

using namespace qa;

namespace {

template <class Kern>
__global__ void __launch_bounds__(Kern::NT) gemm_entry(GemmArgs p) {
  __shared__ __attribute__((aligned(16))) char smem[Kern::LDS_BYTES];
  Kern::run(p, smem);
}

// fp32 on 128x128 tiles and thin ones: two workgroups per CU, 256 registers
template <class Kern>
__global__ void __launch_bounds__(Kern::NT, 2) gemm_entry_two(GemmArgs p) {
  __shared__ __attribute__((aligned(16))) char smem[Kern::LDS_BYTES];
  Kern::run(p, smem);
}

template <class Kern>
__global__ void __launch_bounds__(Kern::NT) pingpong_entry(GemmArgs p) {
  __shared__ __attribute__((aligned(16))) char smem[Kern::LDS_BYTES];
  Kern::run(p, smem);
}

template <class Kern>
__global__ void __launch_bounds__(Kern::NT, Kern::MIN_BLOCKS) short_entry(ShortArgs p) {
  __shared__ __attribute__((aligned(16))) char smem[Kern::LDS_BYTES];
  Kern::run(p, smem);
}

// fp64 GEMM: plain 32x32 SIMT tiles, 2x2 outputs per thread (not an MFMA
// target; kept for the float64 storage contract of the boundary).
__global__ void __launch_bounds__(256) gemm_f64(const double* a, const double* b, double* out, int64_t M,
                                                int64_t K, int64_t N, int64_t sa, int64_t sb, int ta, int tb,
                                                int accumulate, int64_t tiles_n, int64_t tiles_m) {
  __shared__ double As[32][33], Bs[32][33];
  int x = threadIdx.x & 15, y = threadIdx.x >> 4;
  int64_t id = blockIdx.x;
  int64_t z = id / (tiles_m * tiles_n), t = id % (tiles_m * tiles_n);
  int64_t tm = t / tiles_n, tn = t % tiles_n;
  a += z * sa;
  b += z * sb;
  out += z * M * N;
  double c[2][2] = {{0, 0}, {0, 0}};
  for (int64_t k0 = 0; k0 < K; k0 += 32) {
    for (int dy = 0; dy < 2; dy++)
      for (int dx = 0; dx < 2; dx++) {
        int64_t r = tm * 32 + y + dy * 16, k = k0 + x + dx * 16;
        As[y + dy * 16][x + dx * 16] = (r < M && k < K) ? a[ta ? k * M + r : r * K + k] : 0.0;
        int64_t kk = k0 + y + dy * 16, cc = tn * 32 + x + dx * 16;
        Bs[y + dy * 16][x + dx * 16] = (kk < K && cc < N) ? b[tb ? cc * K + kk : kk * N + cc] : 0.0;
      }
    __syncthreads();
    for (int k = 0; k < 32; k++) {
      double a0 = As[y][k], a1 = As[y + 16][k], b0 = Bs[k][x], b1 = Bs[k][x + 16];
      c[0][0] = __dadd_rn(c[0][0], __dmul_rn(a0, b0));
      c[0][1] = __dadd_rn(c[0][1], __dmul_rn(a0, b1));
      c[1][0] = __dadd_rn(c[1][0], __dmul_rn(a1, b0));
      c[1][1] = __dadd_rn(c[1][1], __dmul_rn(a1, b1));
    }
    __syncthreads();
  }
  for (int dy = 0; dy < 2; dy++)
    for (int dx = 0; dx < 2; dx++) {
      int64_t r = tm * 32 + y + dy * 16, cc = tn * 32 + x + dx * 16;
      if (r < M && cc < N) {
        double v = c[dy][dx];
        if (accumulate) v += out[r * N + cc];
        out[r * N + cc] = v;
      }
    }
}

// Operand re-layout into the workspace: dst[z][o][i] = src[z*stride + o*inner + i]
// for i < inner (converted to the compute type; fp32 -> bf16 rounds to
// nearest even) and 0 in the padding up to `pitch`.  Used when an fp32
// operand feeds the bf16 MFMA path (mixed inputs, autocast) or when the
// operand's rows are not 16-byte aligned.  Each thread fills PREP_CHUNKS
// 16-byte chunks of the destination (E = 8 bf16 or 4 fp32 values; pitch is
// a multiple of E) with loads that are contiguous across a wavefront, all in
// flight before the 16-byte stores (one per thread measured fastest: the
// grid then keeps every CU's wave slots busy).  One launch covers the rows [row_base, row_base + rows) with
// 32-bit chunk indices (rows * pitch / E < 2^31; the host splits larger
// operands into several launches), the row's (batch, row) pair in 64 bits.
struct PrepareArgs {
  const void* src;
  void* dst;
  int64_t row_base, outer, stride;
  uint32_t rows, inner, pitch;
};

// One destination chunk i (16 bytes) of the re-layout, loaded and packed.
template <bool SRC_BF16, bool DST_BF16>
__device__ __forceinline__ u32x4 prepare_load(const PrepareArgs& a, uint32_t i) {
  constexpr int E = DST_BF16 ? 8 : 4;
  const uint32_t per_row = a.pitch / E;
  const uint32_t r = i / per_row, c0 = (i - r * per_row) * E;
  const int64_t row = a.row_base + r, z = row / a.outer, o = row - z * a.outer;
  const int64_t at = z * a.stride + o * a.inner + c0;
  if constexpr (SRC_BF16 && DST_BF16) {
    if (c0 + E <= a.inner) {
      // a whole chunk inside the row: one 16-byte load at the element's own
      // (2-byte) alignment -- unaligned global loads are enabled on this
      // platform, and the compiler emits the same for an unaligned memcpy
      u32x4 w;
      __builtin_memcpy(&w, (const char*)a.src + at * 2, 16);
      return w;
    }
  }
  float v[E];
#pragma unroll
  for (int t = 0; t < E; t++) {
    v[t] = 0.f;
    if (c0 + t < a.inner)
      v[t] = SRC_BF16 ? bf16_to_f32(((const bf16_t*)a.src)[at + t]) : ((const float*)a.src)[at + t];
  }
  if constexpr (DST_BF16)
    return u32x4{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7])};
  else
    return u32x4{__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3])};
}

// PREP_CHUNKS chunks per thread, 256 apart (a wavefront's loads stay
// contiguous).
constexpr int PREP_CHUNKS = 1;
template <bool SRC_BF16, bool DST_BF16>
__device__ __forceinline__ void prepare_chunks(const PrepareArgs& a, uint32_t block) {
  constexpr int E = DST_BF16 ? 8 : 4;
  const uint32_t total = a.rows * (a.pitch / E);
  u32x4 w[PREP_CHUNKS];
#pragma unroll
  for (int q = 0; q < PREP_CHUNKS; q++) {
    const uint32_t i = (block * PREP_CHUNKS + q) * 256u + threadIdx.x;
    if (i < total) w[q] = prepare_load<SRC_BF16, DST_BF16>(a, i);
  }
#pragma unroll
  for (int q = 0; q < PREP_CHUNKS; q++) {
    const uint32_t i = (block * PREP_CHUNKS + q) * 256u + threadIdx.x;
    if (i < total) global_store((char*)a.dst + (a.row_base * (a.pitch / E) + i) * 16, w[q]);
  }
}

template <bool SRC_BF16, bool DST_BF16>
__global__ void __launch_bounds__(256) prepare_operand(PrepareArgs a) {
  prepare_chunks<SRC_BF16, DST_BF16>(a, blockIdx.x);
}

// Split-K reduction: out[b][e] = sum over s of part[b * splits + s][e] in
// order s = 0, 1, ... (fp32), plus the old output when accumulating, one
// rounding to the output type.  The partials hold rows of `cols` elements;
// out's rows are `ldc` apart (a column window of a wider output).
__global__ void splitk_reduce(const float* part, void* out, int64_t n, int64_t total, int splits, int accumulate,
                              int out_bf16, int64_t cols, int64_t ldc) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t b = i / n, e = i - b * n;
    const float* src = part + b * splits * n + e;
    float acc = 0.f;
    for (int s = 0; s < splits; s++) acc += src[s * n];
    const int64_t row = e / cols, at = (b * (n / cols) + row) * ldc + (e - row * cols);
    if (accumulate) acc += out_bf16 ? bf16_to_f32(((const bf16_t*)out)[at]) : ((const float*)out)[at];
    if (out_bf16) ((bf16_t*)out)[at] = f32_to_bf16(acc);
    else ((float*)out)[at] = acc;
  }
}

// The same for columns, row pitch, product size and output start that are
// multiples of four elements: 16 bytes of each partial per thread, 32-bit
// indices (total / 4 below 2^32).  3584 x 1024 outputs in 2 chunks: 15 -> 8 us.
__global__ void __launch_bounds__(256) splitk_reduce4(const float* part, void* out, uint32_t n4, uint32_t total4,
                                                      int splits, int accumulate, int out_bf16, uint32_t cols4,
                                                      int64_t ldc) {
  for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < total4; i += gridDim.x * 256) {
    const uint32_t b = i / n4, e = i - b * n4;
    const float* src = part + ((int64_t)b * splits * n4 + e) * 4;
    f32x4 acc = {};
    for (int s = 0; s < splits; s++) acc += global_load<f32x4>(src + (int64_t)s * n4 * 4);
    const uint32_t row = e / cols4;
    const int64_t at = ((int64_t)b * (n4 / cols4) + row) * ldc + (int64_t)(e - row * cols4) * 4;
    if (out_bf16) {
      bf16_t* q = (bf16_t*)out + at;
      if (accumulate) {
        const u32x2 old = global_load<u32x2>(q);
        acc += f32x4{__uint_as_float(old[0] << 16), __uint_as_float(old[0] & 0xffff0000u),
                     __uint_as_float(old[1] << 16), __uint_as_float(old[1] & 0xffff0000u)};
      }
      global_store(q, u32x2{pack_bf16x2(acc[0], acc[1]), pack_bf16x2(acc[2], acc[3])});
    } else {
      float* q = (float*)out + at;
      if (accumulate) acc += global_load<f32x4>(q);
      global_store(q, acc);
    }
  }
}

// Column remainder of at most 8 columns with a K-major A (the last r
// columns of a 256 q + r wide product): a workgroup of RWAVES waves computes
// RWAVES * RROWS output rows.  It stages B's r columns for KC values of k at
// a time in LDS as fp32 (zero beyond K; each element rounded to the compute
// type first, so an fp32 B read in place gives what its re-laid-out bf16
// copy would), while every wave's 16-byte loads of its rows of A for the
// same KC values are in flight:
// lane l sums the 16-byte chunks l, l + 64, ... of its row in K order
// (KC is a multiple of 64 chunks, so the staging does not change that
// order), then a fixed xor tree over the lanes, then the GEMM epilogue's
// accumulate and rounding.  A is a planned operand: rows 16-byte aligned and
// zero-padded to its pitch, so no 16-byte chunk crosses the allocation.  B is
// read at its source dtype and pitch (b_bf16, kb: K-major), r columns from
// column `col`.
constexpr int RWAVES = 4, RROWS = 4, RBLOCK = RWAVES * RROWS, RKC = 1024;
struct RemainderArgs {
  const void* a;
  const void* b;
  void* out;
  int64_t M, K, lda, ldb, ldc, col;
  int r, out_bf16, accumulate;
};

template <bool BF16, bool B_BF16, bool KB>
__device__ __forceinline__ void remainder_block(const RemainderArgs& p, int64_t block, float* cols) {
  constexpr int E = BF16 ? 8 : 4;
  constexpr int NC = RKC / E / 64;  // 16-byte chunks per lane and row in one staged block
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t row0 = block * RBLOCK + wave * RROWS;
  const int r = p.r;
  float acc[RROWS][8];
#pragma unroll
  for (int i = 0; i < RROWS; i++)
#pragma unroll
    for (int j = 0; j < 8; j++) acc[i][j] = 0.f;
  for (int64_t kc = 0; kc < p.K; kc += RKC) {
    // this block's A chunks first (in flight while B's columns are staged)
    const int64_t chunks = (std::min<int64_t>(p.K - kc, RKC) + E - 1) / E;
    u32x4 w[RROWS][NC];
#pragma unroll
    for (int i = 0; i < RROWS; i++)
#pragma unroll
      for (int q = 0; q < NC; q++) {
        const int64_t m = row0 + i, c = lane + 64 * q;
        w[i][q] = u32x4{0u, 0u, 0u, 0u};
        if (m < p.M && c < chunks) w[i][q] = *(const u32x4*)((const char*)p.a + (m * p.lda + kc + c * E) * (BF16 ? 2 : 4));
      }
    __syncthreads();  // the previous block's columns are no longer read
    // cols[j][k - kc] = B(k, col + j) in the compute type; MN-major B: the
    // r columns of one k are neighbours, so a wave reads whole row segments
    // (four loads in flight per thread: the elements of an MN-major B sit
    // in as many rows, one cache line each)
    for (int t0 = 0; t0 < r * RKC; t0 += 4 * 64 * RWAVES) {
      float v[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int t = t0 + u * 64 * RWAVES + tid;
        const int j = KB ? t / RKC : t % r, kk = KB ? t % RKC : t / r;
        const int64_t k = kc + kk;
        v[u] = 0.f;
        if (t < r * RKC && k < p.K) {
          const int64_t at = KB ? (p.col + j) * p.ldb + k : k * p.ldb + p.col + j;
          v[u] = B_BF16 ? bf16_to_f32(((const bf16_t*)p.b)[at]) : ((const float*)p.b)[at];
          if (BF16 && !B_BF16) v[u] = bf16_to_f32(f32_to_bf16(v[u]));
        }
      }
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int t = t0 + u * 64 * RWAVES + tid;
        const int j = KB ? t / RKC : t % r, kk = KB ? t % RKC : t / r;
        if (t < r * RKC) cols[j * RKC + kk] = v[u];
      }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NC; q++) {
      const int64_t c = lane + 64 * q;
      if (c >= chunks) break;
      // one column's values at a time (few registers, so the re-layout
      // workgroups that share this kernel keep their occupancy); every
      // (row, column) sum still runs over its chunk's elements in order
#pragma unroll
      for (int j = 0; j < 8; j++) {
        if (j >= r) break;
        float bv[E];
#pragma unroll
        for (int e = 0; e < E; e += 4) {
          const f32x4 v = *(const f32x4*)(cols + j * RKC + c * E + e);
          bv[e] = v[0];
          bv[e + 1] = v[1];
          bv[e + 2] = v[2];
          bv[e + 3] = v[3];
        }
#pragma unroll
        for (int i = 0; i < RROWS; i++) {
#pragma unroll
          for (int e = 0; e < E; e++) {
            const uint32_t h = w[i][q][BF16 ? e >> 1 : e];
            const float x = BF16 ? __uint_as_float((e & 1) ? (h & 0xffff0000u) : (h << 16)) : __uint_as_float(h);
            acc[i][j] = __builtin_fmaf(x, bv[e], acc[i][j]);
          }
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < RROWS; i++) {
    const int64_t m = row0 + i;
#pragma unroll
    for (int j = 0; j < 8; j++) {
      if (j >= r) break;
      float v = acc[i][j];
      for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
      if (lane == j && m < p.M) {
        const int64_t at = m * p.ldc + j;
        if (p.accumulate) v += p.out_bf16 ? bf16_to_f32(((const bf16_t*)p.out)[at]) : ((const float*)p.out)[at];
        if (p.out_bf16) ((bf16_t*)p.out)[at] = f32_to_bf16(v);
        else ((float*)p.out)[at] = v;
      }
    }
  }
}

template <bool BF16, bool B_BF16, bool KB>
__global__ void __launch_bounds__(64 * RWAVES, 3) remainder_columns(RemainderArgs p) {
  __shared__ __attribute__((aligned(16))) float cols[8 * RKC];
  remainder_block<BF16, B_BF16, KB>(p, blockIdx.x, cols);
}

// B's re-layout and the column remainder in one launch: they are
// independent (the remainder reads B at its source pitch), so the first
// `rem_blocks` workgroups compute remainder rows while the others copy B;
// the large-tile launch that reads the re-laid-out B follows on the stream.
template <bool SRC_BF16, bool BF16, bool KB>
__global__ void __launch_bounds__(256, 3) prepare_remainder(PrepareArgs a, RemainderArgs p, unsigned rem_blocks) {
  __shared__ __attribute__((aligned(16))) float cols[8 * RKC];
  if (blockIdx.x < rem_blocks) remainder_block<BF16, SRC_BF16, KB>(p, blockIdx.x, cols);
  else prepare_chunks<SRC_BF16, BF16>(a, blockIdx.x - rem_blocks);
}

// Kernel configurations: (BM x BN, WM x WN waves, BK, LDS stages, staging).
//   L8D2: 256x256, 8 waves (2 per SIMD), BK 64 (bf16) / 32 (fp32), two-stage
//         direct-to-LDS ring, the next stage's copies spread over the k-steps
//   L8R : 256x256, 8 waves, same K step, register staging
//   L4D2: 256x256, 4 waves (one per SIMD, 128x128 per wave), two-stage ring
//   S   : 128x128, 4 waves, BK 32 / 16, four-stage ring (small grids, short K)
//   S2  : 128x128, 4 waves, BK 32 / 16, two-stage ring (bf16, K <= 64: four per CU)
//   N   : 256x64, 4 waves (N <= 64), BK 64 / 32, two-stage ring, A's copies
//         streamed (nontemporal: one column tile reads every A row once)
//         when A's rows start on 128-byte lines and A exceeds 256 MiB
//   W   : 64x256, 4 waves (M <= 64), BK 32 / 16, four-stage ring
//   H   : 256x128, 8 waves 4x2 (64x64 per wave), BK 64, three-stage ring
//         (grids of 256x256 tiles that would leave half the CUs idle)
//   T, U: 192x256 (8 waves 2x4, 96x64 per wave) and 256x192 (4x2, 64x96),
//         BK 64, two-stage ring, bf16 only (a grid of 256x256 tiles just
//         short of the CU count, e.g. 5632 x 2048: 176 tiles -> 240)
//   R   : short-K row strips (gemm_short.h): bf16 NT with K <= 64, a 128-row
//         block of A held in registers, 128-column chunks of B through a
//         two-slot LDS ring, 128-byte row segments staged through LDS
//   X   : 128x128, 8 waves 2x4 (64x32 per wave), BK 64 / 32, three- / two-stage
//         ring: two waves per SIMD where a grid has one such tile per CU
//   Y, Z: 128x64 and 64x64, 4 waves 2x2, BK 64 / 16, three-stage ring, for
//         grids that larger tiles would leave to a part of the CUs
enum Tile { TILE_L8D2, TILE_L8R, TILE_L4D2, TILE_S, TILE_N, TILE_W, TILE_H, TILE_T, TILE_U, TILE_S2, TILE_R, TILE_P,
            TILE_X, TILE_Y, TILE_Z, TILE_COUNT };

template <bool F32, bool TA, bool TB, int BM, int BN, int WM, int WN, int BK, int ST, bool DMA, bool SWIGLU = false,
          bool GATHER_B = false, bool STREAM_A = false>
hipError_t launch_cfg(GemmArgs p, hipStream_t stream) {
  typedef GemmKernel<F32, TA, TB, BM, BN, WM, WN, BK, ST, DMA, SWIGLU, GATHER_B, STREAM_A> Kern;
  int64_t tiles_n = (p.N + Kern::BNO - 1) / Kern::BNO;
  if (p.groups == 0) p.tiles_m = (int)((p.M + BM - 1) / BM);
  int64_t blocks = (int64_t)p.tiles_m * tiles_n * (p.groups ? 1 : p.batch);
  if (blocks <= 0) return hipSuccess;
  if (blocks > 0x7fffffff) return hipErrorInvalidValue;
  if constexpr (F32 && WM * WN == 4 && BM * BN <= 256 * 64)
    hipLaunchKernelGGL(gemm_entry_two<Kern>, dim3((unsigned)blocks), dim3(Kern::NT), 0, stream, p);
  else hipLaunchKernelGGL(gemm_entry<Kern>, dim3((unsigned)blocks), dim3(Kern::NT), 0, stream, p);
  return hipGetLastError();
}

int forced_tile();

// Tile P: the ping-pong kernel (gemm_pingpong.h) for plain bf16 products
// with K a multiple of 64; other calls take L8D2, whose results it matches
// bit for bit.  Unforced, a 256x256 choice in the NN, NT and TT forms runs
// it (1-3% faster on 4096^3 and 8192-class shapes; TN is equal or 1% slower
// and keeps GemmKernel).
bool pingpong_fits(const GemmArgs& p) {
  return p.K > 0 && p.K % 64 == 0 && p.groups == 0 && p.k_split <= 1 && p.k_head == 0 && !p.group_k;
}
template <bool TA, bool TB>
hipError_t launch_pingpong(GemmArgs p, hipStream_t stream) {
  typedef PingPong<TA, TB> Kern;
  p.tiles_m = (int)((p.M + 255) / 256);
  const int64_t blocks = (int64_t)p.tiles_m * ((p.N + 255) / 256) * p.batch;
  if (blocks <= 0) return hipSuccess;
  if (blocks > 0x7fffffff) return hipErrorInvalidValue;
  hipLaunchKernelGGL(pingpong_entry<Kern>, dim3((unsigned)blocks), dim3(Kern::NT), 0, stream, p);
  return hipGetLastError();
}

// Streamed A copies for the thin tile: A's rows (K-major) or k-rows
// (MN-major), in every batch entry and second K segment, start on 128-byte
// lines, and A spans at least the 256 MiB of the memory-side cache (an
// operand that fits there is cheaper to read with plain loads, which find
// the lines a previous kernel or call left there: a 16384 x 1408 A of a
// 32-column product ran 19.5 us plain against 21.6 us streamed).
bool stream_a(const GemmArgs& p, int64_t es) {
  auto line = [](int64_t bytes) { return bytes % 128 == 0; };
  const int64_t span = p.a_bytes > 0 ? p.a_bytes
                       : (p.batch > 1 && p.sa > 0 ? p.batch * p.sa : (p.groups ? 0 : p.M * p.lda)) * es;
  return span >= (int64_t(256) << 20) && (uintptr_t)p.a % 128 == 0 && line(p.lda * es) && line(p.sa * es) &&
         (p.k_head == 0 || (uintptr_t)p.a_tail % 128 == 0);
}

template <bool F32, bool TA, bool TB>
hipError_t launch_tile(Tile tile, GemmArgs p, hipStream_t stream) {
  constexpr int KB = F32 ? 16 : 32;  // K per stage of the four-stage rings
  constexpr int KR = F32 ? 32 : 64;  // K per stage of the two-stage rings
  switch (tile) {
    case TILE_P:
      if constexpr (!F32)
        if (pingpong_fits(p)) return launch_pingpong<TA, TB>(p, stream);
      return launch_cfg<F32, TA, TB, 256, 256, 2, 4, KR, 2, true>(p, stream);
    case TILE_L8R: return launch_cfg<F32, TA, TB, 256, 256, 2, 4, KR, 2, false>(p, stream);
    case TILE_L4D2: return launch_cfg<F32, TA, TB, 256, 256, 2, 2, KR, 2, true>(p, stream);
    case TILE_S: return launch_cfg<F32, TA, TB, 128, 128, 2, 2, KB, 4, true>(p, stream);
    case TILE_S2: return launch_cfg<F32, TA, TB, 128, 128, 2, 2, KB, 2, true>(p, stream);
    case TILE_X: return launch_cfg<F32, TA, TB, 128, 128, 2, 4, KR, F32 ? 2 : 3, true>(p, stream);
    case TILE_Y: return launch_cfg<F32, TA, TB, 128, 64, 2, 2, F32 ? 16 : KR, 3, true>(p, stream);
    case TILE_Z: return launch_cfg<F32, TA, TB, 64, 64, 2, 2, F32 ? 16 : KR, 3, true>(p, stream);
    case TILE_N:
      // one column tile: every A row is read by one workgroup, streamed
      // (nontemporal copies, K per stage 64 bf16 / 32 fp32 = 128 bytes of a
      // K-major row) where A's rows start on 128-byte lines, so that every
      // copy reads whole lines, and A is larger than the memory-side cache;
      // otherwise the same tile with plain copies
      if (stream_a(p, F32 ? 4 : 2))
        return launch_cfg<F32, TA, TB, 256, 64, 4, 1, KR, 2, true, false, false, true>(p, stream);
      return launch_cfg<F32, TA, TB, 256, 64, 4, 1, KR, 2, true>(p, stream);
    case TILE_W: return launch_cfg<F32, TA, TB, 64, 256, 1, 4, KB, 4, true>(p, stream);
    case TILE_H: return launch_cfg<F32, TA, TB, 256, 128, 4, 2, KR, 3, true>(p, stream);
    case TILE_T:
      if constexpr (F32) return launch_cfg<F32, TA, TB, 256, 256, 2, 4, KR, 2, true>(p, stream);
      else return launch_cfg<F32, TA, TB, 192, 256, 2, 4, KR, 2, true>(p, stream);
    case TILE_U:
      if constexpr (F32) return launch_cfg<F32, TA, TB, 256, 256, 2, 4, KR, 2, true>(p, stream);
      else return launch_cfg<F32, TA, TB, 256, 192, 4, 2, KR, 2, true>(p, stream);
    default:
      // the ping-pong kernel where it measured faster (bit-identical results)
      if constexpr (!F32 && !(TA && !TB))
        if (forced_tile() < 0 && pingpong_fits(p)) return launch_pingpong<TA, TB>(p, stream);
      return launch_cfg<F32, TA, TB, 256, 256, 2, 4, KR, 2, true>(p, stream);
  }
}

// Grouped-K products whose B K rows are read through GemmArgs::b_rows: the
// two-stage direct-to-LDS tiles (192x256 and 256x192 for bf16, else 256x256).
template <bool F32>
hipError_t launch_gathered_k(Tile tile, const GemmArgs& p, hipStream_t stream) {
  constexpr int KR = F32 ? 32 : 64;
  if constexpr (!F32) {
    if (tile == TILE_T) return launch_cfg<F32, true, false, 192, 256, 2, 4, KR, 2, true, false, true>(p, stream);
    if (tile == TILE_U) return launch_cfg<F32, true, false, 256, 192, 4, 2, KR, 2, true, false, true>(p, stream);
  }
  return launch_cfg<F32, true, false, 256, 256, 2, 4, KR, 2, true, false, true>(p, stream);
}

template <bool F32>
hipError_t launch_mma(Tile tile, bool ta, bool tb, const GemmArgs& p, hipStream_t stream) {
  if (ta) return tb ? launch_tile<F32, true, true>(tile, p, stream) : launch_tile<F32, true, false>(tile, p, stream);
  return tb ? launch_tile<F32, false, true>(tile, p, stream) : launch_tile<F32, false, false>(tile, p, stream);
}

// compute units of the current device (cached per device)
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

// QUTAI_AMD_GEMM_TILE=<L8D2|L8R|L4D2|S|N|W|H|T|U|S2|R|P|X|Y|Z> overrides the
// tile choice (tuning and tests; R applies only where the short-K strip kernel
// does, other calls then take L8D2).
int forced_tile() {
  static int forced = [] {
    const char* v = getenv("QUTAI_AMD_GEMM_TILE");
    if (!v) return -1;
    const char* names[TILE_COUNT] = {"L8D2", "L8R", "L4D2", "S", "N", "W", "H", "T", "U", "S2", "R", "P", "X", "Y", "Z"};
    for (int i = 0; i < TILE_COUNT; i++)
      if (std::string(v) == names[i]) return i;
    return -1;
  }();
  return forced;
}

// What a launch of `units` tiles over K costs, in us: K / 64 steps of the
// time that the most loaded CU takes for its tiles, plus the first copies and
// the epilogue of each round.  Measured on this GPU with every tile forced over
// 25 (bf16) and 19 (fp32) shapes from 8 x 1024 x 1024 to 4096^3, whole and
// partial rounds; the choice is the fastest tile or within 5% of it on all but
// two of them.  A CU holds one 256x256, 256x128, 192x256, 256x192 or (bf16)
// eight-wave 128x128 tile, two four-wave 128x128 or 128x64, three or more
// 64x64: small tiles cost more per output and win where large ones would leave
// CUs idle (bf16, 1024^3: 128x128 16.8 us, 64x64 11.1; 2048 x 1024 x 2048 with
// fp32 output: 29.6 and, 128x64, 23.9; fp32, 512^3: 41 and 21).
double launch_cost(Tile tile, int64_t units, int64_t K, bool bf16, bool ta) {
  const int64_t cus = cu_count();
  const int64_t r = (units + cus - 1) / cus;  // tiles of the most loaded CU
  const double n = (double)r, pairs = (double)(r / 2), odd = (double)(r % 2);
  double step, round;
  int64_t held = 1;
  switch (tile) {
    case TILE_H: step = (bf16 ? 1.04 : 6.0) * n, round = 5; break;
    case TILE_T:
    case TILE_U: step = bf16 ? 1.40 * n : 10.4 * n, round = 6; break;
    case TILE_S: step = bf16 ? 1.09 * pairs + 0.78 * odd : 6.2 * pairs + 4.2 * odd, round = 4, held = 2; break;
    // eight waves: bf16 with an MN-major A pays for its transpose reads
    case TILE_X: step = bf16 ? (ta ? 0.83 : 0.67) * n : 6.1 * pairs + 3.5 * odd, round = 4, held = bf16 ? 1 : 2; break;
    case TILE_Y: step = bf16 ? 0.80 * pairs + 0.55 * odd : 4.6 * pairs + 3.2 * odd, round = 3, held = 2; break;
    case TILE_Z: {
      const double b[] = {0.39, 0.55, 0.70, 0.97}, f[] = {2.0, 2.35, 3.3, 4.35};
      step = r <= 4 ? (bf16 ? b : f)[r - 1] : (bf16 ? 0.243 : 1.1) * n;
      round = 2.5, held = 3;
      break;
    }
    default: step = (bf16 ? 1.56 : 10.4) * n, round = 7; break;
  }
  return step * (double)K / 64 + round * (double)((r + held - 1) / held);
}

int64_t tile_count(Tile tile, int64_t rows, int64_t cols, int64_t batch) {
  int64_t bm = 256, bn = 256;
  if (tile == TILE_S || tile == TILE_X) bm = bn = 128;
  else if (tile == TILE_Y) bm = 128, bn = 64;
  else if (tile == TILE_Z) bm = bn = 64;
  else if (tile == TILE_H) bn = 128;
  else if (tile == TILE_T) bm = 192;
  else if (tile == TILE_U) bn = 192;
  else if (tile == TILE_N) bn = 64;
  else if (tile == TILE_W) bm = 64;
  return ((rows + bm - 1) / bm) * ((cols + bn - 1) / bn) * batch;
}

// The cheapest tile of an M x N output (batch of them) over K; the first of
// this order (large to small: less traffic per product) within 3% of the best.
Tile pick_tile(int64_t M, int64_t N, int64_t K, int64_t batch, bool bf16, bool ta, double* cost) {
  static const Tile wide[] = {TILE_H, TILE_U, TILE_T, TILE_L8D2, TILE_X, TILE_S, TILE_Y, TILE_Z};
  static const Tile narrow[] = {TILE_L8D2, TILE_X, TILE_Z};  // fp32: the others never win
  const Tile* tiles = bf16 ? wide : narrow;
  const int count = bf16 ? 8 : 3;
  double best = 1e30, each[8];
  for (int i = 0; i < count; i++) {
    each[i] = launch_cost(tiles[i], tile_count(tiles[i], M, N, batch), K, bf16, ta);
    best = std::min(best, each[i]);
  }
  int pick = 0;
  while (each[pick] > best * 1.03) pick++;
  if (cost) *cost = each[pick];
  return tiles[pick];
}

// The cheapest tile that launch_gathered_k has, for `groups` products.
Tile gathered_k_tile(int64_t rows, int64_t cols, int64_t inner, int groups, bool bf16) {
  if (forced_tile() >= 0) return (Tile)forced_tile();
  Tile pick = TILE_L8D2;
  if (!bf16) return pick;
  double best = launch_cost(pick, tile_count(pick, rows, cols, groups), inner, true, true);
  for (Tile t : {TILE_U, TILE_T}) {
    const double cost = launch_cost(t, tile_count(t, rows, cols, groups), inner, true, true);
    if (cost < 0.97 * best) best = cost, pick = t;
  }
  return pick;
}

Tile choose_tile(int64_t M, int64_t N, int64_t K, int64_t batch, bool bf16, bool ta) {
  if (forced_tile() >= 0) return (Tile)forced_tile();
  const int64_t cus = cu_count();
  // Thin outputs whose 256-wide tiles fill the CUs twice: the tile that reads
  // each row of the long operand once.  Fewer: 64x64, four times the
  // workgroups (4096 x 1024 x 8 logits: 15.5 us in K chunks, 9.8 whole).
  if (N <= 64 && tile_count(TILE_N, M, N, batch) >= 2 * cus) return TILE_N;
  if (M <= 64 && N > 64 && tile_count(TILE_W, M, N, batch) >= 2 * cus) return TILE_W;
  if (N <= 64 || M <= 64) return TILE_Z;
  // Short K is bound by writing the output.  K <= 64 (bf16; the attention
  // score product S = Q K^T with K = the head size): a two-stage ring halves
  // the LDS of the four-stage one, so four workgroups fit per CU instead of
  // two (config 3's S product 336 -> 291 us).  Grids of less than one 128x128
  // tile per CU, or outputs that such tiles would pad by a third, take 64x64.
  const int64_t small = tile_count(TILE_S, M, N, batch);
  if (K <= 128 && small > cus && 3 * tile_count(TILE_Z, M, N, batch) >= 9 * small)
    return bf16 && K <= 64 ? TILE_S2 : bf16 ? TILE_S : TILE_X;
  if (K <= 128) return TILE_Z;
  return pick_tile(M, N, K, batch, bf16, ta, nullptr);
}

// Column remainder: an output N = 256 q + r wide with 0 < r <= 64, whose last
// r columns cost the large tiles about a round of their own (4095 x 4097:
// 272 tiles of 256x256 or 352 of 256x192 for 256 CUs), runs as two launches:
// the first 256 q columns on the large tiles and the last r on the thin
// 256x64 tile, which splits K when its tiles fill few CUs (priced at 0.3 of a
// round).  Returns the first launch's width, or 0 for one launch.  Each
// output element still sums K through the same MFMA chain (split K sums its
// chunks in order), so results stay bit-repeatable.
int64_t column_split(int64_t M, int64_t N, int64_t K, int64_t batch, bool bf16, bool ta) {
  if (forced_tile() >= 0 || batch != 1 || M <= 64 || K <= 128 || N < 512) return 0;
  const int64_t r = N % 256;
  if (r == 0 || r > 64) return 0;
  double full = 0.0, main = 0.0;
  pick_tile(M, N, K, 1, bf16, ta, &full);
  pick_tile(M, N - r, K, 1, bf16, ta, &main);
  return main + 0.3 * launch_cost(TILE_L8D2, 1, K, bf16, ta) < full * 0.97 ? N - r : 0;
}

// Split-K for plain products whose tiles fill at most a quarter of the CU
// slots over a long K (e.g. 1024 x 2048 outputs with K = 32768; a two-way
// split of half-empty grids measured slower): the K
// range is cut into chunks of a multiple of 64 elements, each chunk's fp32
// partial product goes to the workspace and one pass sums them.
// QUTAI_AMD_SPLITK=<n> forces n chunks (tuning and tests; read per call).
size_t split_bytes(int64_t rows, int64_t cols, int64_t batch, int splits) {
  return ((size_t)splits * batch * rows * cols * 4 + 255) / 256 * 256;
}

// rows of an output tile (the M extent a grouped launch counts tiles in)
int tile_rows(Tile tile) {
  switch (tile) {
    case TILE_S:
    case TILE_X:
    case TILE_Y:
    case TILE_S2: return 128;
    case TILE_T: return 192;
    case TILE_Z:
    case TILE_W: return 64;
    default: return 256;
  }
}

// Tile of a grouped (per-expert rows) launch, the M tile count estimated as
// ceil(rows / tile rows) plus half a partial tile per group: 256x64 for thin
// outputs of many rows; 256x256 or 256x192 (bf16) where these fill the CUs
// (config 5's down product, cols 2048: 256x192 109 us against 123 us for
// 256x256; 256x128 and 128x128 measured slower there); eight-wave 128x128 or
// 64x64 tiles where a few hundred rows over many experts would leave most of
// the CUs idle or a 256-row tile mostly empty.
Tile grouped_tile(int64_t rows, int64_t inner, int64_t cols, int groups, bool bf16) {
  if (forced_tile() >= 0) return (Tile)forced_tile();
  if (cols <= 64) return rows >= 512 * cu_count() ? TILE_N : TILE_Z;
  Tile pick = TILE_L8D2;
  double best = 1e30;
  for (Tile t : {TILE_L8D2, TILE_U, TILE_X, TILE_Z}) {
    if (!bf16 && t == TILE_U) continue;
    const int64_t bm = tile_rows(t), tiles_m = (rows + bm - 1) / bm + groups / 2;
    const double cost = launch_cost(t, tiles_m * tile_count(t, 1, cols, 1), inner, bf16, false);
    if (cost < best * 0.97) best = cost, pick = t;
  }
  return pick;
}

// K chunks of a plain product (batch 1): the tile and the chunk count with the
// lowest launch_cost over one chunk plus the partial sums' traffic ((2 s + 1)
// x rows x cols fp32 values at 5 TB/s) and 4 us for the launch that adds them
// up, if that is at least 15% below the product in one piece; below K = 512 the
// second launch and its workspace cost the host more than the GPU gains.  For
// the last kind below the bar is 5% above it: one piece of them measures 9 to
// 16% more than its price (512 x 2048 over K = 4096: 27.5 and 31.4 us) and the
// chunks, whose sums stay in the memory-side cache, up to 16% less (28 and 24);
// of 210 such shapes that the rule splits, every one gained, by a fifth to
// three quarters.  Which products try:
//  * fp32 and thin outputs (<= 64 columns or rows): every one, on the small
//    tiles; their tiles are long (fp32) or few (512 x 4096 x 512 fp32: 128 us
//    in one piece, 32 in eight; a router's 8 logits; 30 x 2048 x 300 bf16:
//    17 -> 14 us);
//  * other bf16 products: K >= 4096 over at most a quarter of the 128x128
//    tile slots (the decoder head's dX, 1024 x 2048 outputs over K = 32768:
//    158 -> 129 us with 256x256 tiles in 8 chunks), on the large tiles; with
//    shorter K the chunks measured slower.
int choose_split(int64_t rows, int64_t cols, int64_t inner, int64_t batch, Tile* tile, bool bf16, bool ta,
                 int64_t* chunk) {
  const int64_t cus = cu_count();
  const bool thin = rows <= 64 || cols <= 64;
  int64_t s = 1;
  const char* forced = getenv("QUTAI_AMD_SPLITK");
  if (forced && atoi(forced) > 0) {
    s = atoi(forced);
  } else if (batch == 1 && forced_tile() < 0 && inner >= 512 && *tile != TILE_N && *tile != TILE_W &&
             (!bf16 || thin || (inner >= 4096 && tile_count(TILE_S, rows, cols, 1) * 2 <= cus))) {
    const double whole = launch_cost(*tile, tile_count(*tile, rows, cols, 1), inner, bf16, ta);
    double best = (bf16 && !thin ? 1.05 : 0.85) * whole;
    for (Tile t : {TILE_L8D2, TILE_H, TILE_S, TILE_X, TILE_Z}) {
      const bool small = t == TILE_X || t == TILE_Z;
      if (thin ? t != TILE_Z : small == bf16) continue;
      const int64_t n = tile_count(t, rows, cols, 1);
      for (int64_t st = 2; st <= (thin ? 16 : 8) && inner >= 64 * st; st++) {
        const int64_t c = ((inner + st - 1) / st + 63) / 64 * 64;
        if ((inner + c - 1) / c != st || (!thin && c < (bf16 ? 512 : 128))) continue;
        const double cost = launch_cost(t, n * st, c, bf16, ta) + 4 + (2.0 * st + 1) * rows * cols * 4 / 5.0e6;
        if (cost < best) {
          best = cost;
          *tile = t;
          s = st;
        }
      }
    }
  }
  if (s <= 1 || inner < 128) return 1;
  const int64_t c = ((inner + s - 1) / s + 63) / 64 * 64;
  s = (inner + c - 1) / c;
  if (s <= 1) return 1;
  *chunk = c;
  return (int)s;
}

// How one operand reaches the kernel: in place, or re-laid out in the
// workspace (dtype change and/or zero-padded 16-byte-aligned rows).
struct Operand {
  const void* ptr;
  int64_t ld, stride, src_stride;
  bool copy;
  int64_t outer, inner, pitch, batches;
  size_t bytes;  // workspace bytes when copied
};

Operand plan_operand(const void* p, int dtype, bool compute_bf16, int64_t outer, int64_t inner, int64_t batch,
                     int64_t stride) {
  const int64_t E = compute_bf16 ? 8 : 4;
  const int64_t es = compute_bf16 ? 2 : 4;
  bool same = (dtype == QA_BF16) == compute_bf16;
  bool aligned = ((uintptr_t)p % 16 == 0) && (inner % E == 0) && (batch <= 1 || stride % E == 0);
  Operand o = {p, inner, stride, stride, !(same && aligned), outer, inner, inner, 1, 0};
  if (o.copy) {
    o.pitch = (inner + E - 1) / E * E;
    o.batches = (stride == 0 || batch <= 1) ? 1 : batch;
    o.ld = o.pitch;
    o.stride = stride == 0 ? 0 : outer * o.pitch;
    o.bytes = (size_t)(o.batches * outer * o.pitch * es + 255) / 256 * 256;
  }
  return o;
}

void plan(int64_t rows, int64_t inner, int64_t cols, int64_t batch, int64_t left_stride, int64_t right_stride,
          int ta, int tb, int a_dtype, int b_dtype, bool bf16, const void* a, const void* b, Operand* pa,
          Operand* pb) {
  *pa = ta ? plan_operand(a, a_dtype, bf16, inner, rows, batch, left_stride)
           : plan_operand(a, a_dtype, bf16, rows, inner, batch, left_stride);
  *pb = tb ? plan_operand(b, b_dtype, bf16, cols, inner, batch, right_stride)
           : plan_operand(b, b_dtype, bf16, inner, cols, batch, right_stride);
}

// A re-laid-out row must fit the kernel's 32-bit chunk indices (any row of
// a valid operand does); larger operands take several launches.
bool prepare_fits(const Operand& o) { return o.pitch < (1ll << 31) && o.inner < (1ll << 32); }

// The re-layout launches of one operand: rows [base, base + r) per launch,
// r * pitch / E below 2^31 chunks.
int prepare_launches(const Operand& o, bool bf16) {
  const int64_t rows = o.batches * o.outer, per_row = o.pitch / (bf16 ? 8 : 4);
  const int64_t step = std::max<int64_t>(1, ((1ll << 31) - 1) / per_row);
  return (int)((rows + step - 1) / step);
}

PrepareArgs prepare_args(const Operand& o, bool bf16, char* ws, int64_t base, uint32_t rows) {
  PrepareArgs a;
  a.src = o.ptr;
  a.dst = ws;
  a.row_base = base;
  a.outer = o.outer;
  a.stride = o.src_stride;
  a.rows = rows;
  a.inner = (uint32_t)o.inner;
  a.pitch = (uint32_t)o.pitch;
  (void)bf16;
  return a;
}

void launch_prepare(Operand& o, int src_dtype, bool bf16, char* ws, hipStream_t stream) {
  const int64_t rows = o.batches * o.outer, per_row = o.pitch / (bf16 ? 8 : 4);
  const int64_t step = std::max<int64_t>(1, ((1ll << 31) - 1) / per_row);  // rows per launch
  for (int64_t base = 0; base < rows; base += step) {
    const uint32_t r = (uint32_t)std::min<int64_t>(step, rows - base);
    const dim3 grid((unsigned)(((int64_t)r * per_row + 256 * PREP_CHUNKS - 1) / (256 * PREP_CHUNKS)));
    const PrepareArgs a = prepare_args(o, bf16, ws, base, r);
    if (src_dtype == QA_BF16 && bf16) hipLaunchKernelGGL((prepare_operand<true, true>), grid, dim3(256), 0, stream, a);
    else if (bf16) hipLaunchKernelGGL((prepare_operand<false, true>), grid, dim3(256), 0, stream, a);
    else if (src_dtype == QA_BF16) hipLaunchKernelGGL((prepare_operand<true, false>), grid, dim3(256), 0, stream, a);
    else hipLaunchKernelGGL((prepare_operand<false, false>), grid, dim3(256), 0, stream, a);
  }
  o.ptr = ws;
}

// The column remainder alone (B used in place: its source dtype is the
// compute type).
void launch_remainder(const RemainderArgs& r, bool bf16, bool kb, hipStream_t stream) {
  const dim3 grid((unsigned)((r.M + RBLOCK - 1) / RBLOCK)), block(64 * RWAVES);
  if (bf16 && kb) hipLaunchKernelGGL((remainder_columns<true, true, true>), grid, block, 0, stream, r);
  else if (bf16) hipLaunchKernelGGL((remainder_columns<true, true, false>), grid, block, 0, stream, r);
  else if (kb) hipLaunchKernelGGL((remainder_columns<false, false, true>), grid, block, 0, stream, r);
  else hipLaunchKernelGGL((remainder_columns<false, false, false>), grid, block, 0, stream, r);
}

// B's re-layout (one launch) with the column remainder in the same grid.
void launch_prepare_remainder(Operand& o, int src_dtype, bool bf16, bool kb, char* ws, const RemainderArgs& r,
                              hipStream_t stream) {
  const int64_t rows = o.batches * o.outer, per_row = o.pitch / (bf16 ? 8 : 4);
  const unsigned rem = (unsigned)((r.M + RBLOCK - 1) / RBLOCK);
  const dim3 grid((unsigned)(rem + (rows * per_row + 256 * PREP_CHUNKS - 1) / (256 * PREP_CHUNKS)));
  const PrepareArgs a = prepare_args(o, bf16, ws, 0, (uint32_t)rows);
  const bool sb = src_dtype == QA_BF16;
  if (sb && bf16 && kb) hipLaunchKernelGGL((prepare_remainder<true, true, true>), grid, dim3(256), 0, stream, a, r, rem);
  else if (sb && bf16) hipLaunchKernelGGL((prepare_remainder<true, true, false>), grid, dim3(256), 0, stream, a, r, rem);
  else if (bf16 && kb) hipLaunchKernelGGL((prepare_remainder<false, true, true>), grid, dim3(256), 0, stream, a, r, rem);
  else if (bf16) hipLaunchKernelGGL((prepare_remainder<false, true, false>), grid, dim3(256), 0, stream, a, r, rem);
  else if (sb && kb) hipLaunchKernelGGL((prepare_remainder<true, false, true>), grid, dim3(256), 0, stream, a, r, rem);
  else if (sb) hipLaunchKernelGGL((prepare_remainder<true, false, false>), grid, dim3(256), 0, stream, a, r, rem);
  else if (kb) hipLaunchKernelGGL((prepare_remainder<false, false, true>), grid, dim3(256), 0, stream, a, r, rem);
  else hipLaunchKernelGGL((prepare_remainder<false, false, false>), grid, dim3(256), 0, stream, a, r, rem);
  o.ptr = ws;
}

// Short-K strip launch (tile R): the call's rows are K-major for both
// operands (NT), K <= 64, bf16 output without accumulation, output rows
// 16-byte aligned and N a multiple of 16 (every 16-byte store is inside or
// wholly outside a row).  Each workgroup
// sweeps `strip` 128-column chunks; strips shrink (halving) until the grid
// holds at least 16 rounds of the two workgroups a CU runs at once.  Config
// 3's score product (128 x 2048 x 2048, K 64): 208 us with one chunk per
// workgroup, 181-185 us with 2, 4 or 8 (the rule gives 4), 200 us with 16.
// The two-slot ring (50 KiB of LDS) under a 168-register cap fits three
// workgroups per CU instead of two: 179-183 -> 166-170 us alone, the bmm
// sequence 789 -> 772 us, bit-identical.
bool short_fits(const GemmArgs& p, bool bf16, bool ta, bool tb) {
  return bf16 && !ta && tb && p.out_bf16 && !p.accumulate && p.K > 0 && p.K <= 64 && p.N % 16 == 0 &&
         p.vec_c == 2 && p.ldc * 128 * 2 < (1ll << 31);
}
hipError_t launch_short(const GemmArgs& p, hipStream_t stream) {
  ShortArgs s = {};
  s.a = (const bf16_t*)p.a;
  s.b = (const bf16_t*)p.b;
  s.out = p.out;
  s.M = p.M;
  s.N = p.N;
  s.K = p.K;
  s.lda = p.lda;
  s.ldb = p.ldb;
  s.ldc = p.ldc;
  s.sa = p.sa;
  s.sb = p.sb;
  s.sc = p.sc;
  s.batch = p.batch;
  s.alpha = p.alpha;
  s.tiles_m = (int)((p.M + 127) / 128);
  s.chunks = (int)((p.N + 127) / 128);
  int strip = s.chunks;
  typedef ShortKernel<2> Kern;
  const int64_t slots = Kern::MIN_BLOCKS * cu_count();
  while (strip > 1 && p.batch * s.tiles_m * ((s.chunks + strip - 1) / strip) < 16 * slots) strip = (strip + 1) / 2;
  s.strip_chunks = strip;
  s.strips = (s.chunks + strip - 1) / strip;
  if (p.batch * s.tiles_m * s.strips > 0x7fffffff) return hipErrorInvalidValue;
  hipLaunchKernelGGL(short_entry<Kern>, dim3((unsigned)(p.batch * s.tiles_m * s.strips)), dim3(Kern::NT), 0, stream,
                     s);
  return hipGetLastError();
}

// 4-wide output stores need 4 | ldc, 4 | batch stride and an aligned base.
// 2: every output row starts 16-byte aligned for both element sizes;
// 1: 16-byte aligned fp32 rows / 8-byte aligned bf16 rows; 0: neither.
int vec_out(const void* p, int64_t ldc, int64_t stride) {
  if ((uintptr_t)p % 16 != 0) return 0;
  if (ldc % 8 == 0 && stride % 8 == 0) return 2;
  return (ldc % 4 == 0 && stride % 4 == 0) ? 1 : 0;
}

// One launch of a plain product over output columns [c0, c0 + n): its tile,
// K chunks and fp32 partial bytes.
struct Window {
  int64_t c0, n;
  Tile tile;
  int splits;
  int64_t chunk;
  size_t partial;
  bool rows_kernel;  // remainder_columns instead of a tile
};

// The launches of a plain product: one window over every column or, with a
// column remainder (column_split), the large-tile columns and the rest: up
// to 8 columns of a K-major A on remainder_columns (one launch, no partial
// sums), wider remainders on the thin tile.
int plan_windows(int64_t rows, int64_t inner, int64_t cols, int64_t batch, bool bf16, int transpose_left,
                 Window (&w)[2]) {
  const int64_t main_cols = inner > 0 ? column_split(rows, cols, inner, batch, bf16, transpose_left) : 0;
  const int count = main_cols ? 2 : 1;
  for (int i = 0; i < count; i++) {
    Window& x = w[i];
    x.c0 = i == 0 ? 0 : main_cols;
    x.n = count == 1 ? cols : i == 0 ? main_cols : cols - main_cols;
    x.rows_kernel = i == 1 && x.n <= 8 && !transpose_left;
    x.tile = choose_tile(rows, x.n, inner, batch, bf16, transpose_left);
    x.chunk = 0;
    x.splits = inner > 0 && !x.rows_kernel ? choose_split(rows, x.n, inner, batch, &x.tile, bf16, transpose_left, &x.chunk) : 1;
    x.partial = x.splits > 1 ? split_bytes(rows, x.n, batch, x.splits) : 0;

  }
  return count;
}

}  // namespace

extern "C" {

size_t qutai_amd_gemm_workspace_size(int64_t rows, int64_t inner, int64_t cols, int64_t batch,
                                     int64_t left_stride, int64_t right_stride, int transpose_left,
                                     int transpose_right, int a_dtype, int b_dtype, int bf16_compute) {
  if (a_dtype == QA_F64 || b_dtype == QA_F64 || batch <= 0 || rows * cols == 0 || inner == 0) return 0;
  bool bf16 = bf16_compute || a_dtype == QA_BF16 || b_dtype == QA_BF16;
  Operand pa, pb;
  // 256-byte aligned pointers: only dtype and row alignment decide
  plan(rows, inner, cols, batch, left_stride, right_stride, transpose_left, transpose_right, a_dtype, b_dtype, bf16,
       (const void*)256, (const void*)256, &pa, &pb);
  Window w[2];
  const int count = plan_windows(rows, inner, cols, batch, bf16, transpose_left, w);
  size_t partial = 0;
  for (int i = 0; i < count; i++) partial += w[i].partial;
  if (!pa.copy && !pb.copy && !partial) return 0;
  return (pa.copy ? pa.bytes : 0) + (pb.copy ? pb.bytes : 0) + partial + 256;
}

}  // extern "C"

namespace qa {

// A plain product.  With `spare`, K chunks whose partial sums do not fit beside
// the operands' re-layouts are given up for the product in one piece (the
// caller's workspace is fixed, or there is none); without, a small workspace is
// an error.
int gemm_plain(const void* a, const void* b, void* out, int64_t rows, int64_t inner, int64_t cols,
                   int64_t batch, int64_t left_stride, int64_t right_stride, int transpose_left,
                   int transpose_right, int a_dtype, int b_dtype, int out_dtype, int accumulate,
                   int bf16_compute, void* workspace, size_t workspace_bytes, bool spare, void* stream_) {
  hipStream_t stream = (hipStream_t)stream_;
  if (rows < 0 || inner < 0 || cols < 0 || batch < 0 || left_stride < 0 || right_stride < 0) return QA_EINVAL;
  bool f64 = a_dtype == QA_F64 || b_dtype == QA_F64;
  for (int d : {a_dtype, b_dtype})
    if (d != QA_F32 && d != QA_BF16 && d != QA_F64) return QA_EINVAL;
  if (f64 && (a_dtype != b_dtype || out_dtype != QA_F64)) return QA_EINVAL;
  if (!f64 && out_dtype != QA_F32 && out_dtype != QA_BF16) return QA_EINVAL;
  int64_t size = batch * rows * cols;
  if (size == 0) return QA_OK;
  if (!out) return QA_EINVAL;
  if (inner > 0 && (!a || !b)) return QA_EINVAL;
  if (f64) {
    int64_t tiles_m = (rows + 31) / 32, tiles_n = (cols + 31) / 32;
    int64_t blocks = tiles_m * tiles_n * batch;
    if (blocks > 0x7fffffff) return QA_EINVAL;
    hipLaunchKernelGGL(gemm_f64, dim3((unsigned)blocks), dim3(256), 0, stream, (const double*)a, (const double*)b,
                       (double*)out, rows, inner, cols, left_stride, right_stride, transpose_left, transpose_right,
                       accumulate, tiles_n, tiles_m);
    return (int)hipGetLastError();
  }
  bool bf16 = bf16_compute || a_dtype == QA_BF16 || b_dtype == QA_BF16;
  Operand pa, pb;
  plan(rows, inner, cols, batch, left_stride, right_stride, transpose_left, transpose_right, a_dtype, b_dtype, bf16,
       a, b, &pa, &pb);
  Window w[2];
  const int count = plan_windows(rows, inner, cols, batch, bf16, transpose_left, w);
  size_t partial = 0;
  for (int i = 0; i < count; i++) partial += w[i].partial;
  if (spare && partial && workspace_bytes < (pa.copy ? pa.bytes : 0) + (pb.copy ? pb.bytes : 0) + partial + 256) {
    partial = 0;
    for (int i = 0; i < count; i++)
      if (w[i].partial) {
        w[i].tile = choose_tile(rows, w[i].n, inner, batch, bf16, transpose_left);
        w[i].splits = 1;
        w[i].partial = 0;
      }
  }
  char* part = nullptr;
  // the column remainder's arguments: A as planned (re-laid out before it
  // runs), B's r columns from column c0 of `b_ptr` (row pitch ldb_src)
  const int osize_ = out_dtype == QA_BF16 ? 2 : 4;
  auto remainder_args = [&](const void* a_ptr, const void* b_ptr, const Window& x, int64_t ldb_src) {
    RemainderArgs r = {};
    r.a = a_ptr;
    r.b = b_ptr;
    r.out = (char*)out + x.c0 * osize_;
    r.M = rows;
    r.K = inner;
    r.lda = pa.ld;
    r.ldb = ldb_src;
    r.ldc = cols;
    r.col = x.c0;
    r.r = (int)x.n;
    r.out_bf16 = out_dtype == QA_BF16 ? 1 : 0;
    r.accumulate = accumulate ? 1 : 0;
    return r;
  };
  bool fused_remainder = false;
  if (inner > 0 && ((pa.copy && !prepare_fits(pa)) || (pb.copy && !prepare_fits(pb)))) return QA_EINVAL;
  if (inner > 0 && (pa.copy || pb.copy || partial)) {
    size_t need = (pa.copy ? pa.bytes : 0) + (pb.copy ? pb.bytes : 0) + partial + 256;
    if (workspace == nullptr || workspace_bytes < need) return QA_EWORKSPACE;
    char* ws = (char*)(((uintptr_t)workspace + 255) & ~(uintptr_t)255);
    if (pa.copy) {
      launch_prepare(pa, a_dtype, bf16, ws, stream);
      ws += pa.bytes;
    }
    if (pb.copy) {
      // B's re-layout shares its launch with a column remainder (which reads
      // B at its source pitch and dtype) when it takes one launch
      if (count == 2 && w[1].rows_kernel && prepare_launches(pb, bf16) == 1) {
        fused_remainder = true;
        launch_prepare_remainder(pb, b_dtype, bf16, transpose_right, ws,
                                 remainder_args(pa.ptr, b, w[1], transpose_right ? inner : cols), stream);
      } else {
        launch_prepare(pb, b_dtype, bf16, ws, stream);
      }
      ws += pb.bytes;
    }
    if (partial) part = ws;
  }
  GemmArgs p = {};
  p.a = pa.ptr;
  p.b = pb.ptr;
  p.out = out;
  p.M = rows;
  p.N = cols;
  p.K = inner;
  p.lda = pa.ld;
  p.ldb = pb.ld;
  p.ldc = cols;
  p.sa = pa.stride;
  p.sb = pb.stride;
  p.sc = rows * cols;
  p.batch = batch;
  p.accumulate = accumulate ? 1 : 0;
  p.out_bf16 = out_dtype == QA_BF16;
  p.vec_c = vec_out(out, p.ldc, p.sc);
  p.alpha = 1.0f;
  // buffer descriptors address at most 2^31 bytes per K step
  int64_t es = bf16 ? 2 : 4;
  if ((p.lda * 256 * es) >= (1ll << 31) || (p.ldb * 256 * es) >= (1ll << 31)) return QA_EINVAL;
  const int osize = out_dtype == QA_BF16 ? 2 : 4;
  for (int i = 0; i < count; i++) {
    const Window& x = w[i];
    GemmArgs q = p;
    // the window's columns: B's rows (K-major) or columns from c0, out's
    // columns from c0 at the full row pitch
    q.N = x.n;
    q.b = (const char*)pb.ptr + x.c0 * (transpose_right ? pb.ld : 1) * es;
    char* window_out = (char*)out + x.c0 * osize;
    q.out = window_out;
    q.vec_c = vec_out(window_out, q.ldc, q.sc);
    float* window_part = nullptr;
    if (x.partial && !x.rows_kernel) {
      // fp32 partials of each K chunk ([rows][n] each), then the ordered sum
      window_part = (float*)part;
      part += x.partial;
      q.out = window_part;
      q.ldc = x.n;
      q.sc = rows * x.n;
      q.k_split = x.splits;
      q.k_chunk = x.chunk;
      q.batch = batch * x.splits;
      q.accumulate = 0;
      q.out_bf16 = 0;
      q.vec_c = vec_out(window_part, q.ldc, q.sc);
    }
    if (x.rows_kernel) {
      // the last r columns: done with B's re-layout, or one launch of their own
      if (!fused_remainder) {
        launch_remainder(remainder_args(q.a, pb.ptr, x, pb.ld), bf16, transpose_right, stream);
        const hipError_t err = hipGetLastError();
        if (err != hipSuccess) return (int)err;
      }
      continue;
    }
    if (!window_part && count == 1 && ((x.tile == TILE_S2 && forced_tile() < 0) || x.tile == TILE_R) &&
        short_fits(q, bf16, transpose_left, transpose_right))
      return (int)launch_short(q, stream);
    hipError_t err = bf16 ? launch_mma<false>(x.tile, transpose_left, transpose_right, q, stream)
                          : launch_mma<true>(x.tile, transpose_left, transpose_right, q, stream);
    if (err != hipSuccess) return (int)err;
    if (!window_part) continue;
    const int64_t total = batch * rows * x.n;
    if (x.n % 4 == 0 && cols % 4 == 0 && (uintptr_t)window_out % (4 * osize) == 0 && total / 4 < (1ll << 31)) {
      const unsigned blocks4 = (unsigned)((total / 4 + 255) / 256);
      hipLaunchKernelGGL(splitk_reduce4, dim3(blocks4), dim3(256), 0, stream, (const float*)window_part,
                         (void*)window_out, (uint32_t)(rows * x.n / 4), (uint32_t)(total / 4), x.splits,
                         accumulate ? 1 : 0, out_dtype == QA_BF16 ? 1 : 0, (uint32_t)(x.n / 4), cols);
      err = hipGetLastError();
      if (err != hipSuccess) return (int)err;
      continue;
    }
    const unsigned blocks = (unsigned)std::min<int64_t>((total + 255) / 256, 1 << 20);
    hipLaunchKernelGGL(splitk_reduce, dim3(blocks), dim3(256), 0, stream, (const float*)window_part,
                       (void*)window_out, rows * x.n, total, x.splits, accumulate ? 1 : 0,
                       out_dtype == QA_BF16 ? 1 : 0, x.n, cols);
    err = hipGetLastError();
    if (err != hipSuccess) return (int)err;
  }
  return QA_OK;
}

}  // namespace qa

extern "C" {

int qutai_amd_gemm(const void* a, const void* b, void* out, int64_t rows, int64_t inner, int64_t cols,
                   int64_t batch, int64_t left_stride, int64_t right_stride, int transpose_left,
                   int transpose_right, int a_dtype, int b_dtype, int out_dtype, int accumulate,
                   int bf16_compute, void* workspace, size_t workspace_bytes, void* stream_) {
  return qa::gemm_plain(a, b, out, rows, inner, cols, batch, left_stride, right_stride, transpose_left, transpose_right,
                    a_dtype, b_dtype, out_dtype, accumulate, bf16_compute, workspace, workspace ? workspace_bytes : 0,
                    !workspace, stream_);
}

int qutai_amd_gemm_grouped(const void* a, const void* b, void* out, const int64_t* offsets, int groups,
                           int64_t max_rows, int64_t inner, int64_t cols, int64_t expert_stride,
                           int transpose_right, int dtype, int out_dtype, int accumulate, const int64_t* gather,
                           int64_t source_rows, void* stream_) {
  hipStream_t stream = (hipStream_t)stream_;
  if (groups <= 0 || max_rows < 0 || inner < 0 || cols < 0 || expert_stride < 0) return QA_EINVAL;
  if (dtype != QA_BF16 && dtype != QA_F32) return QA_EINVAL;
  if (out_dtype != QA_F32 && out_dtype != QA_BF16) return QA_EINVAL;
  if (!offsets || !out) return QA_EINVAL;
  if (max_rows == 0 || cols == 0) return QA_OK;
  GemmArgs p = {};
  p.a = a;
  p.b = b;
  p.out = out;
  p.M = max_rows;
  p.N = cols;
  p.K = inner;
  p.lda = inner;
  p.ldb = transpose_right ? inner : cols;
  p.ldc = cols;
  p.sb = expert_stride;
  p.batch = 1;
  p.accumulate = accumulate ? 1 : 0;
  p.out_bf16 = out_dtype == QA_BF16;
  int64_t E = dtype == QA_BF16 ? 8 : 4;
  if ((uintptr_t)a % 16 || (uintptr_t)b % 16 || inner % E || p.ldb % E || expert_stride % E) return QA_EINVAL;
  // a 256-row tile's operand range must fit the 31-bit buffer descriptor
  const int64_t es = dtype == QA_BF16 ? 2 : 4;
  if ((p.lda * 256 * es) >= (1ll << 31) || (p.ldb * 256 * es) >= (1ll << 31)) return QA_EINVAL;
  p.vec_c = vec_out(out, p.ldc, 0);
  p.offsets = offsets;
  p.groups = groups;
  p.alpha = 1.0f;
  if (gather) {
    // row offsets into a are 32-bit byte offsets of one buffer descriptor
    if (source_rows < 0 || source_rows * inner * es >= (1ll << 31)) return QA_EINVAL;
    p.a_rows = gather;
    p.a_bytes = source_rows * inner * es;
  }
  Tile tile = grouped_tile(max_rows, p.K, cols, groups, dtype == QA_BF16);
  if (gather && tile == TILE_L8R) tile = TILE_L8D2;  // gathered rows need the DMA ring
  const int bm = tile_rows(tile);
  p.tiles_m = (int)((max_rows + bm - 1) / bm + groups);
  bool f32 = dtype == QA_F32;
  hipError_t err = f32 ? launch_mma<true>(tile, false, transpose_right, p, stream)
                       : launch_mma<false>(tile, false, transpose_right, p, stream);
  return (int)err;
}

int qutai_amd_gemm_grouped_pair(const void* a, const void* a_tail, const void* b, const void* b_tail, void* out,
                                const int64_t* offsets, int groups, int64_t max_rows, int64_t inner, int64_t cols,
                                int64_t expert_stride, int transpose_right, int dtype, int out_dtype, int accumulate,
                                void* stream_) {
  hipStream_t stream = (hipStream_t)stream_;
  if (groups <= 0 || max_rows < 0 || inner < 0 || cols < 0 || expert_stride < 0) return QA_EINVAL;
  if (dtype != QA_BF16 && dtype != QA_F32) return QA_EINVAL;
  if (out_dtype != QA_F32 && out_dtype != QA_BF16) return QA_EINVAL;
  if (!offsets || !out) return QA_EINVAL;
  // the join must fall on a K step of every tile configuration (64 / 32)
  if (inner % 64) return QA_EINVAL;
  if (max_rows == 0 || cols == 0) return QA_OK;
  if (inner == 0) return QA_EINVAL;
  GemmArgs p = {};
  p.a = a;
  p.b = b;
  p.a_tail = a_tail;
  p.b_tail = b_tail;
  p.k_head = inner;
  p.out = out;
  p.M = max_rows;
  p.N = cols;
  p.K = 2 * inner;
  p.lda = inner;
  p.ldb = transpose_right ? inner : cols;
  p.ldc = cols;
  p.sb = expert_stride;
  p.batch = 1;
  p.accumulate = accumulate ? 1 : 0;
  p.out_bf16 = out_dtype == QA_BF16;
  const int64_t E = dtype == QA_BF16 ? 8 : 4;
  for (const void* q : {a, a_tail, b, b_tail})
    if (!q || (uintptr_t)q % 16) return QA_EINVAL;
  if (p.ldb % E || expert_stride % E) return QA_EINVAL;
  const int64_t es = dtype == QA_BF16 ? 2 : 4;
  if ((p.lda * 256 * es) >= (1ll << 31) || (p.ldb * 256 * es) >= (1ll << 31)) return QA_EINVAL;
  p.vec_c = vec_out(out, p.ldc, 0);
  p.offsets = offsets;
  p.groups = groups;
  p.alpha = 1.0f;
  Tile tile = grouped_tile(max_rows, p.K, cols, groups, dtype == QA_BF16);
  const int bm = tile_rows(tile);
  p.tiles_m = (int)((max_rows + bm - 1) / bm + groups);
  hipError_t err = dtype == QA_F32 ? launch_mma<true>(tile, false, transpose_right, p, stream)
                                   : launch_mma<false>(tile, false, transpose_right, p, stream);
  return (int)err;
}

int qutai_amd_gemm_swiglu(const void* a, const void* w_gate, const void* w_up, void* out, void* gate_out,
                          void* up_out, const int64_t* offsets, int groups, int64_t rows, int64_t inner,
                          int64_t hidden, int64_t expert_stride, int dtype, const int64_t* gather,
                          int64_t source_rows, void* stream_) {
  hipStream_t stream = (hipStream_t)stream_;
  if (rows < 0 || inner < 0 || hidden < 0 || expert_stride < 0 || (offsets && groups <= 0)) return QA_EINVAL;
  if (dtype != QA_BF16) return QA_EINVAL;
  if (!out || (rows > 0 && hidden > 0 && (!a || !w_gate || !w_up))) return QA_EINVAL;
  if (rows == 0 || hidden == 0) return QA_OK;
  if ((uintptr_t)a % 16 || (uintptr_t)w_gate % 16 || (uintptr_t)w_up % 16 || inner % 8 || expert_stride % 8)
    return QA_EINVAL;
  for (void* o : {out, gate_out, up_out})
    if (o && (uintptr_t)o % 16) return QA_EINVAL;
  GemmArgs p = {};
  p.a = a;
  p.b = w_gate;
  p.b2 = w_up;
  p.out = out;
  p.gate_out = gate_out;
  p.up_out = up_out;
  p.M = rows;
  p.N = hidden;
  p.K = inner;
  p.lda = inner;
  p.ldb = inner;
  p.ldc = hidden;
  p.sb = offsets ? expert_stride : 0;
  p.sc = rows * hidden;
  p.batch = 1;
  p.out_bf16 = 1;
  p.vec_c = vec_out(out, p.ldc, 0);
  p.alpha = 1.0f;
  if ((p.lda * 256 * 2) >= (1ll << 31)) return QA_EINVAL;
  if (gather) {
    if (!offsets || source_rows < 0 || source_rows * inner * 2 >= (1ll << 31)) return QA_EINVAL;
    p.a_rows = gather;
    p.a_bytes = source_rows * inner * 2;
  }
  if (offsets) {
    p.offsets = offsets;
    p.groups = groups;
    p.tiles_m = (int)((rows + 255) / 256 + groups);
  }
  return (int)launch_cfg<false, false, true, 256, 256, 2, 4, 64, 2, true, true>(p, stream);
}

int qutai_amd_gemm_grouped_k(const void* a, const void* b, void* out, const int64_t* offsets, int groups, int64_t rows,
                             int64_t cols, int64_t total_k, int dtype, int out_dtype, int accumulate,
                             const int64_t* gather, int64_t source_rows, void* stream_) {
  hipStream_t stream = (hipStream_t)stream_;
  if (groups <= 0 || rows < 0 || cols < 0 || total_k < 0) return QA_EINVAL;
  if (dtype != QA_BF16 && dtype != QA_F32) return QA_EINVAL;
  if (out_dtype != QA_F32 && out_dtype != QA_BF16) return QA_EINVAL;
  if (!offsets || !out) return QA_EINVAL;
  if (rows == 0 || cols == 0) return QA_OK;
  const int64_t E = dtype == QA_BF16 ? 8 : 4;
  if ((uintptr_t)a % 16 || (uintptr_t)b % 16 || rows % E || cols % E) return QA_EINVAL;
  GemmArgs p = {};
  p.a = a;
  p.b = b;
  p.out = out;
  p.M = rows;
  p.N = cols;
  p.K = total_k;
  p.lda = rows;  // A stored [K][rows]: out_g = A_g^T B_g
  p.ldb = cols;  // B stored [K][cols]
  p.ldc = cols;
  p.sc = rows * cols;
  p.batch = groups;
  p.accumulate = accumulate ? 1 : 0;
  p.out_bf16 = out_dtype == QA_BF16;
  p.vec_c = vec_out(out, p.ldc, p.sc);
  p.offsets = offsets;
  p.group_k = 1;
  p.alpha = 1.0f;
  int64_t es = dtype == QA_BF16 ? 2 : 4;
  if ((p.lda * 256 * es) >= (1ll << 31) || (p.ldb * 256 * es) >= (1ll << 31)) return QA_EINVAL;
  if (gather) {
    // row offsets into b are 32-bit byte offsets of one buffer descriptor
    if (source_rows < 0 || source_rows * cols * es >= (1ll << 31)) return QA_EINVAL;
    p.b_rows = gather;
    p.b_bytes = source_rows * cols * es;
    const Tile tile = gathered_k_tile(rows, cols, total_k / groups + 1, groups, dtype == QA_BF16);
    return (int)(dtype == QA_F32 ? launch_gathered_k<true>(tile, p, stream)
                                 : launch_gathered_k<false>(tile, p, stream));
  }
  const Tile tile = choose_tile(rows, cols, total_k / groups + 1, groups, dtype == QA_BF16, true);
  hipError_t err = dtype == QA_F32 ? launch_mma<true>(tile, true, false, p, stream)
                                   : launch_mma<false>(tile, true, false, p, stream);
  return (int)err;
}

}  // extern "C"
