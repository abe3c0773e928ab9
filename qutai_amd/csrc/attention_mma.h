// Attention for the head widths and storage types that the D = 64 bf16
// kernels do not cover, on the matrix cores: bf16 storage with any head
// dimension that is a multiple of 8 up to 256, fp32 storage with any multiple
// of 4 up to 128 (16-byte rows).  Everything that was held in fp32 by the
// one-wave-per-row kernels stays fp32-accurate:
//
//  * a fp32 value v enters v_mfma_f32_32x32x16_bf16 as the three bf16 values
//    v0 = bf16(v), v1 = bf16(v - v0), v2 = bf16(v - v0 - v1), which hold its
//    24 significant bits (every difference is exact); a product of two such
//    values takes the six MFMAs whose terms are above 2^-24 of it, so an fp32
//    product costs 6/16 of v_mfma_f32_32x32x2_f32's cycles;
//  * fp32 storage splits q, k, v and dO that way, both storage types split the
//    probabilities and dS, which are fp32 in either;
//  * values, probabilities and dS are split as 2^24 of themselves, and the
//    scale and the outputs' factors take that back: the bits of every finite
//    value, subnormals included, then end above bf16's smallest normal;
//  * the split needs finite values, and sums below 2^128 as scaled; an
//    infinity or NaN anywhere in a wave's operands reaches its accumulators as
//    a NaN or infinity, and such a wave computes its rows again with the
//    one-wave-per-row code.
//
// Shape of the work: a workgroup of four waves owns 128 queries (forward,
// dq) or 128 keys (dk, dv) of one (batch, head), 32 per wave; the other
// side streams through LDS in blocks of KB rows, loaded into registers one
// block ahead and split once per workgroup on the way into LDS.  The score
// blocks are computed transposed (S^T = K Q^T), so one lane holds one query
// (key in the dk/dv kernel), the softmax statistics are per-lane scalars, and
// the result registers are the B operand of the next product as they are
// (the same lane layout as the D = 64 kernels).
//
// What bounds it: the MFMAs (fp32: 12 per 32x32 scores and 16 dimensions in
// the forward, bf16: 4) and the splitting of the probabilities beside them.
// Measured (MI355X, causal; forward and backward), against one wave per row:
// bf16, batch 4, T 1024, 16 heads over 4 of 128: 5663 and 13510 us before, 60
// and 227 now; fp32, batch 8, T 512, 8 heads of 64: 1236 and 2862 us before, 35
// and 102 now.  With two parts (2^-17) of the probabilities and dS the first
// takes 45 and 168 us, but 2.3 of 1000 bf16 results were not float64's rounded,
// 0.5 with one wave per row, 0.3 with three parts.
#pragma once
#include "attention_rows.h"

namespace qa {

// acc += A B with operands in NA and NB parts: the terms a_i b_j with
// first <= i + j < max(NA, NB), smallest first.  Three-part operands keep the
// terms beside a_0 b_0 in an accumulator of their own (first = 1, then
// high_part): the large sum then takes one rounding per MFMA step instead of
// six, and the two chains do not wait for each other.
// SWAP: in the order in which B A adds them.
template <bool SWAP = false, int NA, int NB>
__device__ __forceinline__ f32x16 mma_parts(const bf16x8 (&a)[NA], const bf16x8 (&b)[NB], f32x16 acc, int first = 0) {
  constexpr int N = NA > NB ? NA : NB;
#pragma unroll
  for (int order = N - 1; order >= first; order--)
#pragma unroll
    for (int n = 0; n <= order; n++) {
      const int i = SWAP ? order - n : n, j = order - i;
      if (i < NA && j < NB) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[j], acc, 0, 0, 0);
    }
  return acc;
}
template <int NA, int NB>
__device__ __forceinline__ f32x16 high_part(const bf16x8 (&a)[NA], const bf16x8 (&b)[NB], f32x16 acc) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[0], acc, 0, 0, 0);
}

}  // namespace qa

namespace {

using namespace qa;

// Tiles of KB streamed rows of two tensors (K and V, or Q and dO) in LDS:
// NX bf16 planes each, rows of PC 16-byte chunks (a power of two), chunk c of
// row r at c ^ swz(r).
template <bool F32, int DP>
struct AttnTile {
  static constexpr int NX = F32 ? 3 : 1;             // parts of a stored value
  static constexpr int NP = 3;                       // parts of a probability or dS
  // what parts of stored values and of probabilities and dS are scaled by,
  // what takes a sum of products of a stored value and a weight back, and dP
  // (two stored values) to dS's scale
  static constexpr float STORED = F32 ? 0x1p24f : 1.f, WEIGHT = 0x1p24f;
  static constexpr float SUM = 1.f / (STORED * WEIGHT), DP_TO_DS = WEIGHT / (STORED * STORED);
  static constexpr int KB = F32 || DP > 128 ? 32 : 64;
  static constexpr int CK = DP / 8;                  // chunks of a row in use
  static constexpr int PC = DP <= 32 ? 4 : DP <= 64 ? 8 : DP <= 128 ? 16 : 32;
  static constexpr int PITCH = PC * 8, PLANE = KB * PITCH;
  static constexpr int ITEMS = 2 * KB * CK / 256;    // 8-element chunks per thread and block
  static_assert(2 * KB * CK % 256 == 0 && KB * CK % 64 == 0, "a wave's chunks come from one tensor");
  static constexpr int S = DP / 16, DB = DP / 32;    // MFMA k-steps over d, 32-wide d blocks

  // 8 (or 16) consecutive rows at one chunk, and the transpose read's 4 rows
  // x 64 bytes, fall into distinct banks of the 256-byte bank window.
  __device__ static __forceinline__ int swz(int r) {
    if constexpr (PC == 4) return (r >> 2) & 3;
    else if constexpr (PC == 8) return (r ^ (r >> 3)) & 7;
    else return ((r & 3) << 2) | ((r >> 2) & 3);
  }
  // Row fragment: row r, d = 16 s + 8 half + [0, 8), every plane.
  __device__ static __forceinline__ void rows(const bf16_t* x, int r, int s, int half, bf16x8 (&f)[NX]) {
    const int at = r * PITCH + (((2 * s + half) ^ swz(r)) * 8);
#pragma unroll
    for (int n = 0; n < NX; n++) f[n] = *reinterpret_cast<const bf16x8*>(x + n * PLANE + at);
  }
  // Transposed fragment (tr_frag of the D = 64 kernels): A operand rows = d
  // columns 32 db + [0, 32), k = tile rows rb + {4 half + [0, 4), 8 + ...}.
  __device__ static __forceinline__ void columns(const bf16_t* x, int db, int rb, int lane, bf16x8 (&f)[NX]) {
    typedef i16x4 __attribute__((address_space(3))) * lds_ptr;
    const int g = lane >> 4, i = lane & 15;
    const int cb = 32 * db + (g & 1) * 16 + 4 * (i & 3);
    const int r0 = rb + 4 * (g >> 1) + (i >> 2), r1 = r0 + 8;
    const int a0 = r0 * PITCH + (((cb >> 3) ^ swz(r0)) * 8) + (cb & 7);
    const int a1 = r1 * PITCH + (((cb >> 3) ^ swz(r1)) * 8) + (cb & 7);
#pragma unroll
    for (int n = 0; n < NX; n++) {
      const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(x + n * PLANE + a0));
      const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(x + n * PLANE + a1));
      const i16x8 w = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      f[n] = __builtin_bit_cast(bf16x8, w);
    }
  }
};

constexpr uint32_t ATTN_OOB = 0x80000000u;  // beyond every descriptor's range: reads as zeros

// Eight elements at byte offset `off` of a descriptor, in parts: bf16 as it
// is, fp32 as three bf16 parts.  ok / ok_hi: elements 0-3 / 4-7 exist.
template <bool F32>
struct Raw8 {
  u32x4 w[F32 ? 2 : 1];
  __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t r, uint32_t off, bool ok, bool ok_hi) {
    w[0] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, ok ? off : ATTN_OOB, 0, 0));
    if constexpr (F32)
      w[1] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, ok_hi ? off + 16 : ATTN_OOB, 0, 0));
  }
  __device__ __forceinline__ void parts(bf16x8 (&f)[F32 ? 3 : 1]) const {
    if constexpr (F32) {
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; e++) v[e] = __uint_as_float(w[e >> 2][e & 3]) * 0x1p24f;  // AttnTile::STORED
      split_bf16(v, f);
    } else {
      f[0] = __builtin_bit_cast(bf16x8, w[0]);
    }
  }
};

// The chunks of the streamed block that this thread moves: global -> registers
// (`fetch`, rows at or beyond `left` and d at or beyond D read as zeros),
// registers -> LDS planes (`put`).
template <bool F32, int DP>
struct AttnStage {
  typedef AttnTile<F32, DP> Tile;
  static constexpr int ES = F32 ? 4 : 2;
  uint32_t off[Tile::ITEMS];
  int row[Tile::ITEMS], lds[Tile::ITEMS];
  bool lo[Tile::ITEMS], hi[Tile::ITEMS];
  Raw8<F32> raw[Tile::ITEMS];

  __device__ __forceinline__ void plan(int tid, int64_t stride, int D) {
#pragma unroll
    for (int j = 0; j < Tile::ITEMS; j++) {
      const int idx = tid + 256 * j, q = idx % (Tile::KB * Tile::CK);
      const int r = q / Tile::CK, c = q % Tile::CK;
      row[j] = r;
      lo[j] = 8 * c < D;
      hi[j] = 8 * c + 4 < D;
      off[j] = (uint32_t)((r * stride + 8 * c) * ES);
      lds[j] = (idx / (Tile::KB * Tile::CK)) * Tile::NX * Tile::PLANE + r * Tile::PITCH + ((c ^ Tile::swz(r)) * 8);
    }
  }
  __device__ __forceinline__ void fetch(const char* x, const char* y, int64_t stride, int left, int wave) {
    const int64_t bytes = Tile::KB * stride * ES;
    const uint32_t n = bytes > 0x7ffffff0 ? 0x7ffffff0u : (uint32_t)bytes;
    const auto rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(x), 0, n, 0x00020000);
    const auto ry = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(y), 0, n, 0x00020000);
#pragma unroll
    for (int j = 0; j < Tile::ITEMS; j++) {
      const bool in = row[j] < left;
      const bool second = (wave * 64 + 256 * j) / (Tile::KB * Tile::CK);  // wave-uniform
      raw[j].load(second ? ry : rx, off[j], in && lo[j], in && hi[j]);
    }
  }
  __device__ __forceinline__ void put(bf16_t* tiles) const {
#pragma unroll
    for (int j = 0; j < Tile::ITEMS; j++) {
      bf16x8 f[Tile::NX];
      raw[j].parts(f);
#pragma unroll
      for (int n = 0; n < Tile::NX; n++) *reinterpret_cast<bf16x8*>(tiles + lds[j] + n * Tile::PLANE) = f[n];
    }
  }
};

// The wave's own 32 rows of a q- or kv-shaped tensor as B operands, from
// element `first` on: lane = row col, d = 16 s + 8 half + [0, 8).
template <bool F32, int DP>
__device__ __forceinline__ void own_rows(const void* base, int64_t first, int64_t stride, int col, bool in, int half,
                                         int D, Raw8<F32> (&raw)[DP / 16]) {
  constexpr int ES = F32 ? 4 : 2;
  const char* p = uniform_ptr((const char*)base + first * ES);
  const auto r = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(p), 0, 0x7ffffff0u, 0x00020000);
#pragma unroll
  for (int s = 0; s < DP / 16; s++) {
    const int d = 16 * s + 8 * half;
    raw[s].load(r, (uint32_t)((col * stride + d) * ES), in && d < D, in && d + 4 < D);
  }
}

// acc += X^T W over the 32 streamed rows 32 mb + [0, 32): X^T's d block db
// from the tile, W (probabilities or dS) in parts.
template <bool F32, int DP>
__device__ __forceinline__ void add_product(const bf16_t* x, int db, int mb, int lane,
                                            const bf16x8 (&w)[2][AttnTile<F32, DP>::NP], f32x16& acc) {
  typedef AttnTile<F32, DP> Tile;
  f32x16 lo = {};
#pragma unroll
  for (int st = 0; st < 2; st++) {
    bf16x8 f[Tile::NX];
    Tile::columns(x, db, 32 * mb + 16 * st, lane, f);
    acc = high_part(f, w[st], acc);
    lo = mma_parts(f, w[st], lo, 1);
  }
  acc += lo;
}

// Four consecutive outputs d .. d+3 of one row.
template <bool F32>
__device__ __forceinline__ void put4(void* base, int64_t at, const f32x4& v) {
  if constexpr (F32) global_store((float*)base + at, v);
  else global_store((bf16_t*)base + at, u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])});
}

// Zero when every element is finite, NaN otherwise.
template <int N>
__device__ __forceinline__ float not_finite(const f32x16 (&x)[N]) {
  float z = 0.f;
#pragma unroll
  for (int i = 0; i < N; i++)
#pragma unroll
    for (int e = 0; e < 16; e++) z = __builtin_fmaf(x[i][e], 0.f, z);
  return z;
}

// 2^(s c - ref) with c = scale log2(e), one fma; for fp32 storage the rounding
// errors of c and ref come back as a second fma (scale_log2_lo, ref_lo).
// Masked scores are -inf and give 0.
template <bool F32>
__device__ __forceinline__ float weight_of(float s, const AttnGenArgs& p, float ref, float ref_lo) {
  float x = __builtin_fmaf(s, p.scale_log2, -ref);
  if constexpr (F32) x += __builtin_fmaf(s == -INFINITY ? 0.f : s, p.scale_log2_lo, -ref_lo);
  return __builtin_amdgcn_exp2f(x);
}
// lse log2(e) and its rounding error
__device__ __forceinline__ float log2_of(float lse, float& lo) {
  const float hi = lse * LOG2E;
  lo = __builtin_fmaf(lse, LOG2E, -hi) + lse * LOG2E_LO;
  return hi;
}

template <bool F32, int DP>
__global__ void __launch_bounds__(256, F32 && DP > 64 || DP > 128 ? 1 : 2) attention_fwd_mma(AttnGenArgs p) {
  typedef AttnTile<F32, DP> Tile;
  typedef AttnStage<F32, DP> Stage;
  typedef typename std::conditional<F32, float, bf16_t>::type T_;
  constexpr int KB = Tile::KB, QPB = 128, ES = F32 ? 4 : 2;
  __shared__ __attribute__((aligned(16))) bf16_t tiles[2 * Tile::NX * Tile::PLANE];  // [K, V][plane]
  const int tid = threadIdx.x, lane = tid & 63, wave = uniform32(tid >> 6), half = lane >> 5, col = lane & 31;
  const int T = (int)p.time, D = (int)p.dim;
  const int blocks_q = (T + QPB - 1) / QPB;
  // causal: the longest query blocks of every head first; otherwise one
  // head's blocks on one XCD (as the D = 64 kernels)
  int bh, qblk;
  if (p.causal) {
    const int nbh = (int)(p.batch * p.heads);
    bh = uniform32((int)blockIdx.x % nbh);
    qblk = uniform32(blocks_q - 1 - (int)blockIdx.x / nbh);
  } else {
    const int pid = uniform32(xcd_remap(blockIdx.x, gridDim.x));
    bh = uniform32(pid / blocks_q);
    qblk = uniform32(pid % blocks_q);
  }
  const int wg_q0 = qblk * QPB, q0 = uniform32(wg_q0 + wave * 32);
  const int b = bh / (int)p.heads, h = bh % (int)p.heads, kvh = h / (int)(p.heads / p.kv_heads);
  const int64_t kbase = b * p.kb + kvh * p.kh;
  const char* K = uniform_ptr((const char*)p.k + kbase * ES);
  const char* V = uniform_ptr((const char*)p.v + kbase * ES);
  const int t = q0 + col;

  bf16x8 qf[Tile::S][Tile::NX];
  {
    Raw8<F32> raw[Tile::S];
    own_rows<F32, DP>(p.q, b * p.qb + h * p.qh + q0 * p.qt, p.qt, col, t < T, half, D, raw);
#pragma unroll
    for (int s = 0; s < Tile::S; s++) raw[s].parts(qf[s]);
  }
  f32x16 o[Tile::DB];
#pragma unroll
  for (int db = 0; db < Tile::DB; db++) o[db] = f32x16{};
  float m = -INFINITY, l = 0.f;
  const float c = p.scale_log2;

  const int nkb = ((p.causal ? min(wg_q0 + QPB, T) : T) + KB - 1) / KB;
  const int nkb_w = p.causal ? min(nkb, (q0 + 32 + KB - 1) / KB) : nkb;
  const int n_full = min(nkb_w, (p.causal ? min(T, q0 + 1) : T) / KB);
  Stage stage;
  stage.plan(tid, p.kt, D);
  auto fetch = [&](int kbk) {
    const int64_t at = (int64_t)kbk * KB * p.kt * ES;
    stage.fetch(K + at, V + at, p.kt, T - kbk * KB, wave);
  };
  // block kbk into LDS (every wave has read the previous one), the next one
  // into registers
  auto advance = [&](int kbk) {
    __syncthreads();
    stage.put(tiles);
    __syncthreads();
    if (kbk + 1 < nkb) fetch(kbk + 1);
  };
  auto attend = [&](int mb, int lim, auto mask) {
    const bf16_t* sk = tiles;
    const bf16_t* sv = tiles + Tile::NX * Tile::PLANE;
    f32x16 sc = {}, sc_lo = {};
#pragma unroll
    for (int s = 0; s < Tile::S; s++) {
      bf16x8 kf[Tile::NX];
      Tile::rows(sk, 32 * mb + col, s, half, kf);
      sc = high_part(kf, qf[s], sc);
      if constexpr (F32) sc_lo = mma_parts(kf, qf[s], sc_lo, 1);
    }
    if constexpr (F32) sc += sc_lo;
    // element e: key 32 mb + 8 (e / 4) + 4 half + e % 4 of the block
    if constexpr (decltype(mask)::value) {
#pragma unroll
      for (int e = 0; e < 16; e++)
        if (32 * mb + 8 * (e >> 2) + (e & 3) >= lim) sc[e] = -INFINITY;
    }
    float peak = -INFINITY;
#pragma unroll
    for (int e = 0; e < 16; e++) peak = fmaxf(peak, sc[e]);
    // the reference point m moves only for a max more than 2^8 above it, as
    // in the D = 64 kernels
    const float cand = pair_max(peak) * c;
    const bool grow = cand > m + 8.f;
    if (__builtin_amdgcn_ballot_w64(grow)) {
      if (grow) {
        const float alpha = __builtin_amdgcn_exp2f(m - cand);
        m = cand;
        l *= alpha;
#pragma unroll
        for (int db = 0; db < Tile::DB; db++)
#pragma unroll
          for (int e = 0; e < 16; e++) o[db][e] *= alpha;
      }
    }
    const float ref = m == -INFINITY ? 0.f : m;
    float sum = 0.f;
    bf16x8 pf[2][Tile::NP];
#pragma unroll
    for (int st = 0; st < 2; st++) {
      float pv[8];
#pragma unroll
      for (int e = 0; e < 8; e++) {
        pv[e] = weight_of<F32>(sc[8 * st + e], p, ref, 0.f);
        sum += pv[e];
        pv[e] *= Tile::WEIGHT;
      }
      split_bf16(pv, pf[st]);
    }
    l += sum;
#pragma unroll
    for (int db = 0; db < Tile::DB; db++) add_product<F32, DP>(sv, db, mb, lane, pf, o[db]);
  };
  if (nkb > 0) fetch(0);
  int kbk = 0;
  for (; kbk < n_full; kbk++) {
    advance(kbk);
#pragma unroll 1
    for (int mb = 0; mb < KB / 32; mb++) attend(mb, 0, std::false_type{});
  }
  for (; kbk < nkb_w; kbk++) {
    advance(kbk);
    const int kv0 = kbk * KB;
    const int lim = min(T - kv0, p.causal ? t - kv0 + 1 : KB) - 4 * half;
#pragma unroll 1
    for (int mb = 0; mb < KB / 32; mb++) attend(mb, lim, std::true_type{});
  }
  for (; kbk < nkb; kbk++) advance(kbk);

  const float total = pair_sum(l);
  const float bad = not_finite(o) + total * 0.f + m * 0.f;
  if (__builtin_amdgcn_ballot_w64(t < T && !(bad == 0.f))) {
    for (int i = 0; i < 32 && q0 + i < T; i++) fwd_row<T_>(p, b, h, q0 + i, lane);
    return;
  }
  if (t < T) {
    const float inv = Tile::SUM / total;
    const int64_t at = b * p.qb + h * p.qh + (int64_t)t * p.qt;
#pragma unroll
    for (int db = 0; db < Tile::DB; db++)
#pragma unroll
      for (int g = 0; g < 4; g++) {
        const int d = 32 * db + 8 * g + 4 * half;
        if (d < D)
          put4<F32>(p.dq, at + d, f32x4{o[db][4 * g], o[db][4 * g + 1], o[db][4 * g + 2], o[db][4 * g + 3]} * inv);
      }
    if (p.lse && half == 0) p.lse[b * p.lb + h * p.lh + t * p.lt] = (m + __log2f(total)) * 0.6931471805599453f;
  }
}

// dQ and delta of 128 queries; K and V stream.  delta = dO . O is summed by the
// MFMAs as dP = dO . V is, term by term, so that what their difference leaves of
// a query that sees one key (or nearly so) is what O and V leave: an exact zero
// for bf16.  With delta in fp32 fmas, the two sums' roundings stayed: 1.0% of
// the bf16 dQ of 40 causal queries of 128 were not float64's rounded, 0.02% now.
template <bool F32, int DP>
__global__ void __launch_bounds__(256, F32 && DP > 64 || DP > 128 ? 1 : 2) attention_bwd_dq_mma(AttnGenArgs p) {
  typedef AttnTile<F32, DP> Tile;
  typedef AttnStage<F32, DP> Stage;
  typedef typename std::conditional<F32, float, bf16_t>::type T_;
  constexpr int KB = Tile::KB, QPB = 128, ES = F32 ? 4 : 2;
  __shared__ __attribute__((aligned(16))) bf16_t tiles[2 * Tile::NX * Tile::PLANE];
  const int tid = threadIdx.x, lane = tid & 63, wave = uniform32(tid >> 6), half = lane >> 5, col = lane & 31;
  const int T = (int)p.time, D = (int)p.dim;
  const int blocks_q = (T + QPB - 1) / QPB;
  int bh, qblk;
  if (p.causal) {
    const int nbh = (int)(p.batch * p.heads);
    bh = uniform32((int)blockIdx.x % nbh);
    qblk = uniform32(blocks_q - 1 - (int)blockIdx.x / nbh);
  } else {
    const int pid = uniform32(xcd_remap(blockIdx.x, gridDim.x));
    bh = uniform32(pid / blocks_q);
    qblk = uniform32(pid % blocks_q);
  }
  const int wg_q0 = qblk * QPB, q0 = uniform32(wg_q0 + wave * 32);
  const int b = bh / (int)p.heads, h = bh % (int)p.heads, kvh = h / (int)(p.heads / p.kv_heads);
  const int64_t qbase = b * p.qb + h * p.qh, kbase = b * p.kb + kvh * p.kh;
  const char* K = uniform_ptr((const char*)p.k + kbase * ES);
  const char* V = uniform_ptr((const char*)p.v + kbase * ES);
  const int t = q0 + col;

  bf16x8 qf[Tile::S][Tile::NX], gf[Tile::S][Tile::NX];
  float dl = 0.f, lse2 = 0.f, lse2_lo = 0.f;
  {
    Raw8<F32> raw[Tile::S];
    own_rows<F32, DP>(p.q, qbase + q0 * p.qt, p.qt, col, t < T, half, D, raw);
#pragma unroll
    for (int s = 0; s < Tile::S; s++) raw[s].parts(qf[s]);
    own_rows<F32, DP>(p.g, qbase + q0 * p.qt, p.qt, col, t < T, half, D, raw);
#pragma unroll
    for (int s = 0; s < Tile::S; s++) raw[s].parts(gf[s]);
    own_rows<F32, DP>(p.o, qbase + q0 * p.qt, p.qt, col, t < T, half, D, raw);
    f32x16 og = {}, og_lo = {};  // O dO^T of the wave's queries, whose diagonal is delta
#pragma unroll
    for (int s = 0; s < Tile::S; s++) {
      bf16x8 of[Tile::NX];
      raw[s].parts(of);
      og = high_part(of, gf[s], og);
      if constexpr (F32) og_lo = mma_parts(of, gf[s], og_lo, 1);
    }
    if constexpr (F32) og += og_lo;
#pragma unroll
    for (int e = 0; e < 16; e++)
      if (8 * (e >> 2) + 4 * half + (e & 3) == col) dl = og[e];
    dl = pair_sum(dl);
    const int64_t li = b * p.lb + h * p.lh + (int64_t)t * p.lt;
    if (t < T) lse2 = log2_of(p.lse[li], lse2_lo);
    if (t < T && half == 0) p.delta[li] = dl * (1.f / (Tile::STORED * Tile::STORED));
    dl *= Tile::DP_TO_DS;
  }
  f32x16 dqt[Tile::DB];
#pragma unroll
  for (int db = 0; db < Tile::DB; db++) dqt[db] = f32x16{};

  const int nkb = ((p.causal ? min(wg_q0 + QPB, T) : T) + KB - 1) / KB;
  const int nkb_w = p.causal ? min(nkb, (q0 + 32 + KB - 1) / KB) : nkb;
  const int n_full = min(nkb_w, (p.causal ? min(T, q0 + 1) : T) / KB);
  Stage stage;
  stage.plan(tid, p.kt, D);
  auto fetch = [&](int kbk) {
    const int64_t at = (int64_t)kbk * KB * p.kt * ES;
    stage.fetch(K + at, V + at, p.kt, T - kbk * KB, wave);
  };
  auto advance = [&](int kbk) {
    __syncthreads();
    stage.put(tiles);
    __syncthreads();
    if (kbk + 1 < nkb) fetch(kbk + 1);
  };
  auto step = [&](int mb, int lim, auto mask) {
    const bf16_t* sk = tiles;
    const bf16_t* sv = tiles + Tile::NX * Tile::PLANE;
    f32x16 sc = {}, dp = {}, sc_lo = {}, dp_lo = {};
#pragma unroll
    for (int s = 0; s < Tile::S; s++) {
      bf16x8 kf[Tile::NX], vf[Tile::NX];
      Tile::rows(sk, 32 * mb + col, s, half, kf);
      sc = high_part(kf, qf[s], sc);
      if constexpr (F32) sc_lo = mma_parts(kf, qf[s], sc_lo, 1);
      Tile::rows(sv, 32 * mb + col, s, half, vf);
      dp = high_part(vf, gf[s], dp);
      if constexpr (F32) dp_lo = mma_parts(vf, gf[s], dp_lo, 1);
    }
    if constexpr (F32) sc += sc_lo, dp += dp_lo;
    bf16x8 dsf[2][Tile::NP];
#pragma unroll
    for (int st = 0; st < 2; st++) {
      float ds[8];
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const int e = 8 * st + i;
        float x = sc[e];
        if constexpr (decltype(mask)::value)
          if (32 * mb + 8 * (e >> 2) + (e & 3) >= lim) x = -INFINITY;
        ds[i] = weight_of<F32>(x, p, lse2, lse2_lo) * __builtin_fmaf(dp[e], Tile::DP_TO_DS, -dl);
      }
      split_bf16(ds, dsf[st]);
    }
#pragma unroll
    for (int db = 0; db < Tile::DB; db++) add_product<F32, DP>(sk, db, mb, lane, dsf, dqt[db]);
  };
  if (nkb > 0) fetch(0);
  int kbk = 0;
  for (; kbk < n_full; kbk++) {
    advance(kbk);
#pragma unroll 1
    for (int mb = 0; mb < KB / 32; mb++) step(mb, 0, std::false_type{});
  }
  for (; kbk < nkb_w; kbk++) {
    advance(kbk);
    const int kv0 = kbk * KB;
    const int lim = min(T - kv0, p.causal ? t - kv0 + 1 : KB) - 4 * half;
#pragma unroll 1
    for (int mb = 0; mb < KB / 32; mb++) step(mb, lim, std::true_type{});
  }
  for (; kbk < nkb; kbk++) advance(kbk);

  if (__builtin_amdgcn_ballot_w64(t < T && !(not_finite(dqt) == 0.f))) {
    for (int i = 0; i < 32 && q0 + i < T; i++) bwd_q_row<T_>(p, b, h, q0 + i, lane);
    return;
  }
  if (t < T) {
    const int64_t at = qbase + (int64_t)t * p.qt;
#pragma unroll
    for (int db = 0; db < Tile::DB; db++)
#pragma unroll
      for (int g = 0; g < 4; g++) {
        const int d = 32 * db + 8 * g + 4 * half;
        if (d < D)
          put4<F32>(p.dq, at + d,
                    f32x4{dqt[db][4 * g], dqt[db][4 * g + 1], dqt[db][4 * g + 2], dqt[db][4 * g + 3]} *
                        (p.scale * Tile::SUM));
      }
  }
}

// dK and dV of 128 keys of one kv head (p.split: of one query head of its
// group, as unscaled fp32 partials); Q, dO, lse and delta stream.  Above 128
// dimensions the sums of both do not fit a wave's registers and each has a
// launch (bf16, batch 4, T 1024, 16 heads over 4 of 256: a backward pass takes
// 637 us, about twice that with both and their spills).
enum KeySide { KEYS_BOTH, KEYS_DK, KEYS_DV };

template <bool F32, int DP, KeySide SIDE>
__global__ void __launch_bounds__(256, F32 && DP > 32 || DP > 64 ? 1 : 2) attention_bwd_dkv_mma(AttnGenArgs p) {
  typedef AttnTile<F32, DP> Tile;
  typedef AttnStage<F32, DP> Stage;
  typedef typename std::conditional<F32, float, bf16_t>::type T_;
  constexpr int KB = Tile::KB, KPB = 128, ES = F32 ? 4 : 2;
  __shared__ __attribute__((aligned(16))) bf16_t tiles[2 * Tile::NX * Tile::PLANE];  // [Q, dO][plane]
  __shared__ __attribute__((aligned(16))) float stats[3][KB];  // lse log2(e) and its rounding error, delta as dS
  const int tid = threadIdx.x, lane = tid & 63, wave = uniform32(tid >> 6), half = lane >> 5, col = lane & 31;
  const int T = (int)p.time, D = (int)p.dim;
  const int blocks_k = (T + KPB - 1) / KPB;
  const int group = (int)(p.heads / p.kv_heads), nsplit = p.split ? group : 1;
  int bkh, kblk, gsel;
  if (p.causal) {  // the first keys see the most queries and start first
    const int nbh = (int)(p.batch * p.kv_heads) * nsplit, id = (int)blockIdx.x % nbh;
    bkh = uniform32(id / nsplit);
    gsel = uniform32(id % nsplit);
    kblk = uniform32((int)blockIdx.x / nbh);
  } else {
    const int pid = uniform32(xcd_remap(blockIdx.x, gridDim.x)), rest = pid % (blocks_k * nsplit);
    bkh = uniform32(pid / (blocks_k * nsplit));
    kblk = uniform32(rest / nsplit);
    gsel = uniform32(rest % nsplit);
  }
  const int g_lo = p.split ? gsel : 0, g_hi = p.split ? gsel + 1 : group;
  const int k0 = uniform32(kblk * KPB), kw = uniform32(k0 + wave * 32);
  const int b = bkh / (int)p.kv_heads, kvh = bkh % (int)p.kv_heads;
  const int64_t kbase = b * p.kb + kvh * p.kh;
  const int key = kw + col;

  bf16x8 kf[Tile::S][Tile::NX], vf[Tile::S][Tile::NX];
  {
    Raw8<F32> raw[Tile::S];
    own_rows<F32, DP>(p.k, kbase + kw * p.kt, p.kt, col, key < T, half, D, raw);
#pragma unroll
    for (int s = 0; s < Tile::S; s++) raw[s].parts(kf[s]);
    own_rows<F32, DP>(p.v, kbase + kw * p.kt, p.kt, col, key < T, half, D, raw);
#pragma unroll
    for (int s = 0; s < Tile::S; s++) raw[s].parts(vf[s]);
  }
  constexpr bool DK = SIDE != KEYS_DV, DV = SIDE != KEYS_DK;
  f32x16 dkt[DK ? Tile::DB : 1], dvt[DV ? Tile::DB : 1];
#pragma unroll
  for (auto& x : dkt) x = f32x16{};
#pragma unroll
  for (auto& x : dvt) x = f32x16{};

  const int qs0 = p.causal ? k0 : 0;
  const int nq = qs0 < T ? (T - qs0 + KB - 1) / KB : 0;
  const int iterations = nq * (g_hi - g_lo);
  Stage stage;
  stage.plan(tid, p.qt, D);
  float lse_next = 0.f, delta_next = 0.f;  // of query tid of the block in flight (tid < KB)
  auto fetch = [&](int it) {
    const int h = kvh * group + g_lo + it / nq, qs = qs0 + (it % nq) * KB;
    const int64_t at = (b * p.qb + h * p.qh + (int64_t)qs * p.qt) * ES;
    stage.fetch(uniform_ptr((const char*)p.q + at), uniform_ptr((const char*)p.g + at), p.qt, T - qs, wave);
    if (tid < KB) {
      const bool in = qs + tid < T;
      const int64_t li = b * p.lb + h * p.lh + (int64_t)(in ? qs + tid : 0) * p.lt;
      lse_next = in ? p.lse[li] : 0.f;
      delta_next = in ? p.delta[li] : 0.f;
    }
  };
  auto advance = [&](int it) {
    __syncthreads();
    stage.put(tiles);
    if (tid < KB) {
      float lo;
      stats[0][tid] = log2_of(lse_next, lo);
      stats[1][tid] = lo;
      stats[2][tid] = delta_next * Tile::WEIGHT;
    }
    __syncthreads();
    if (it + 1 < iterations) fetch(it + 1);
  };
  auto step = [&](int mb, int qs, auto mask) {
    const bf16_t* sq = tiles;
    const bf16_t* sg = tiles + Tile::NX * Tile::PLANE;
    f32x16 sc = {}, dp = {}, sc_lo = {}, dp_lo = {};
#pragma unroll
    for (int s = 0; s < Tile::S; s++) {
      bf16x8 qa[Tile::NX], ga[Tile::NX];
      Tile::rows(sq, 32 * mb + col, s, half, qa);
      sc = high_part(qa, kf[s], sc);
      if constexpr (F32) sc_lo = mma_parts<true>(qa, kf[s], sc_lo, 1);  // as the other kernels sum K Q^T, V dO^T
      if constexpr (DK) {
        Tile::rows(sg, 32 * mb + col, s, half, ga);
        dp = high_part(ga, vf[s], dp);
        if constexpr (F32) dp_lo = mma_parts<true>(ga, vf[s], dp_lo, 1);
      }
    }
    if constexpr (F32) sc += sc_lo, dp += dp_lo;
    // element e: query qs + 32 mb + 8 (e / 4) + 4 half + e % 4, key kw + col
    float ds[16];
    bf16x8 w[2][Tile::NP];  // the probabilities, then dS
#pragma unroll
    for (int st = 0; st < 2; st++) {
      float pr[8];
#pragma unroll
      for (int j = 0; j < 2; j++) {
        const int q4 = 32 * mb + 8 * (2 * st + j) + 4 * half;
        const f32x4 l4 = *reinterpret_cast<const f32x4*>(&stats[0][q4]);
        const f32x4 d4 = *reinterpret_cast<const f32x4*>(&stats[2][q4]);
        f32x4 lo4 = {};
        if constexpr (F32) lo4 = *reinterpret_cast<const f32x4*>(&stats[1][q4]);
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const int e = 8 * st + 4 * j + i;
          float x = sc[e];
          if constexpr (decltype(mask)::value)
            if (qs + q4 + i >= T || (p.causal && qs + q4 + i < key)) x = -INFINITY;
          pr[4 * j + i] = weight_of<F32>(x, p, l4[i], lo4[i]);
          ds[e] = pr[4 * j + i] * __builtin_fmaf(dp[e], Tile::DP_TO_DS, -d4[i]);
          pr[4 * j + i] *= Tile::WEIGHT;
        }
      }
      if constexpr (DV) split_bf16(pr, w[st]);
    }
    if constexpr (DV) {
#pragma unroll
      for (int db = 0; db < Tile::DB; db++) add_product<F32, DP>(sg, db, mb, lane, w, dvt[db]);
    }
    if constexpr (DK) {
#pragma unroll
      for (int st = 0; st < 2; st++) split_bf16(reinterpret_cast<const float(&)[8]>(ds[8 * st]), w[st]);
#pragma unroll
      for (int db = 0; db < Tile::DB; db++) add_product<F32, DP>(sq, db, mb, lane, w, dkt[db]);
    }
  };
  // per head: query blocks before every key of the wave (causal; skipped),
  // masked, with every pair visible, masked at the end of the sequence
  auto clampq = [&](int x, int lo) { return x < lo ? lo : x > nq ? nq : x; };
  const int first = p.causal ? clampq((kw - qs0) / KB, 0) : 0;
  const int full = p.causal ? clampq((kw + 31 - qs0 + KB - 1) / KB, first) : first;
  const int tail = clampq((T - qs0) / KB, full);
  if (iterations > 0) fetch(0);
  int it = 0;
  for (int g = g_lo; g < g_hi; g++) {
    int qi = 0;
    for (; qi < first; qi++, it++) advance(it);
    for (; qi < full; qi++, it++) {
      advance(it);
#pragma unroll 1
      for (int mb = 0; mb < KB / 32; mb++) step(mb, qs0 + qi * KB, std::true_type{});
    }
    for (; qi < tail; qi++, it++) {
      advance(it);
#pragma unroll 1
      for (int mb = 0; mb < KB / 32; mb++) step(mb, qs0 + qi * KB, std::false_type{});
    }
    for (; qi < nq; qi++, it++) {
      advance(it);
#pragma unroll 1
      for (int mb = 0; mb < KB / 32; mb++) step(mb, qs0 + qi * KB, std::true_type{});
    }
  }

  const bool bad = key < T && !(not_finite(dkt) + not_finite(dvt) == 0.f);
  if (__builtin_amdgcn_ballot_w64(bad)) {
    for (int i = 0; i < 32 && kw + i < T; i++) bwd_kv_row<T_>(p, b, kvh, kw + i, lane, g_lo, g_hi);
    return;
  }
  if (key < T) {
    const int64_t at = kbase + (int64_t)key * p.kt;
#pragma unroll
    for (int db = 0; db < Tile::DB; db++)
#pragma unroll
      for (int g = 0; g < 4; g++) {
        const int d = 32 * db + 8 * g + 4 * half;
        if (d >= D) continue;
        if constexpr (DK) {
          const f32x16& y = dkt[db];
          const f32x4 x = {y[4 * g], y[4 * g + 1], y[4 * g + 2], y[4 * g + 3]};
          if (p.split) global_store(p.part_k + gsel * p.part_stride + at + d, x * Tile::SUM);
          else put4<F32>(p.dk, at + d, x * (p.scale * Tile::SUM));
        }
        if constexpr (DV) {
          const f32x16& y = dvt[db];
          const f32x4 x = {y[4 * g], y[4 * g + 1], y[4 * g + 2], y[4 * g + 3]};
          if (p.split) global_store(p.part_v + gsel * p.part_stride + at + d, x * Tile::SUM);
          else put4<F32>(p.dv, at + d, x * Tile::SUM);
        }
      }
  }
}

}  // namespace
