// Delta-mode anchor selection on gfx950.
//
// Replaces chunked_eval_kernel (tritonModules.py:7-69) and its launch
// (modeling_llama.py:634-653).  One wave64 walks one chunk of one KV head
// sequentially: the first row is an anchor; every later row is compared with the
// current anchor and becomes the anchor when it is far enough (Euclidean
// ||k - a||^2 > tau^2, or cosine < tau).
//
// Lane l holds head-dimension elements 2l and 2l+1 (one 4-byte load per lane, a
// coalesced 256-byte row per wave for D = 128).  The distance is fp32 and reduced
// by a fixed perfect pairwise tree over 128 slots: the per-lane pair sum is level 1,
// DPP lane^1, lane^2, 8-lane mirror and 16-lane mirror give levels 2-5 (every lane
// of a 16-lane row then holds the row sum), and the four row sums are combined as
// (r0 + r1) + (r2 + r3).  No multiply-add is fused, so the result is bit-identical
// to the CPU restatement of the same tree.
//
// With A16 (DA_SELECT_ARITH16) the Euclidean distance rounds every difference, square
// and tree addition to the keys' 16-bit type, as the reference's Triton code evaluates
// curr - ref, diff * diff and tl.sum on 16-bit tensors (tritonModules.py:55-58); only
// the reduction order stays the fixed tree.  The cosine test is fp32 either way (the
// reference upcasts it, :48-54).
//
// Rows are prefetched 32 at a time one batch ahead, since loads never depend on
// the decisions.  The distance reaches every lane through v_permlane16/32_swap (no
// scalar round trip), the anchor update is a select, and a batch's decisions collect
// in a 32-bit mask stored as int32 (the reference's keep-mask format).
//
// That walk is select_kernel.  Rows a matrix operand can be loaded from take
// select_band_kernel instead, which decides most (anchor, row) pairs of a chunk from
// matrix products, all at once, and leaves only the close ones to the exact tree.
#include <algorithm>
#include <climits>
#include <cmath>
#include <type_traits>

#include "da_common.hpp"

namespace da {

constexpr int kSelBatch = 32;
constexpr int64_t kSelPairMinChunks = 2048;
constexpr int64_t kBandMinRows = 128;

// x rounded to the 16-bit type DT (nearest even) and widened back to fp32.  For bf16
// one v_cvt_pk_bf16_f32 with x in the high half and 0 in the low half leaves exactly
// that fp32 value in the register (the widening is free); fp16 converts there and back.
template <int DT>
__device__ __forceinline__ float round16(float x) {
  if constexpr (DT == DA_BF16) {
    // as asm: written in C the compiler swaps the halves back and adds a v_perm_b32
    float r;
    asm("v_cvt_pk_bf16_f32 %0, 0, %1" : "=v"(r) : "v"(x));
    return r;
  } else
    return E16<DT>::one(E16<DT>::bits(x));
}

// wave_tree_sum_all with every addition rounded to DT: the same pairing (DPP lane^1,
// lane^2, 8-lane and 16-lane mirror, then (r0 + r1) + (r2 + r3)).
template <int DT>
__device__ __forceinline__ float wave_tree_sum_all_r16(float t) {
#pragma clang fp contract(off)
  t = round16<DT>(t + dpp_f32<kDppXor1>(t));
  t = round16<DT>(t + dpp_f32<kDppXor2>(t));
  t = round16<DT>(t + dpp_f32<kDppHalfMirror>(t));
  t = round16<DT>(t + dpp_f32<kDppMirror>(t));
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(t), __float_as_uint(t), false, false);
  const float u = round16<DT>(__uint_as_float(r[0]) + __uint_as_float(r[1]));
  const auto q = __builtin_amdgcn_permlane32_swap(__float_as_uint(u), __float_as_uint(u), false, false);
  return round16<DT>(__uint_as_float(q[0]) + __uint_as_float(q[1]));
}

// A lane's two key elements (2l, 2l + 1) of one row: one 4-byte word of a 16-bit type,
// or two fp32 values (8 bytes; fp32 keys are compared in fp32, the reference's
// arithmetic on fp32 tensors).
template <int DT>
struct SelKey {
  using Elem = uint16_t;
  using Row = uint32_t;
  static __device__ __forceinline__ float lo(Row w) { return E16<DT>::lo(w); }
  static __device__ __forceinline__ float hi(Row w) { return E16<DT>::hi(w); }
};
template <>
struct SelKey<DA_F32> {
  using Elem = float;
  using Row = u32x2;
  static __device__ __forceinline__ float lo(Row w) { return __uint_as_float(w[0]); }
  static __device__ __forceinline__ float hi(Row w) { return __uint_as_float(w[1]); }
};

// One key of the walk: the decision and the anchor update without a branch (the
// decision is the same in every lane).
template <bool COS, bool A16, int DT>
__device__ __forceinline__ bool select_step(float x0, float x1, float& a0, float& a1, float& a_norm,
                                            float thr) {
#pragma clang fp contract(off)
  const float eps = 1e-8f;
  bool kp;
  float x_norm = 0.0f;
  if constexpr (COS) {  // tritonModules.py:48-54
    const float dot = wave_tree_sum_all(pair_dot(x0, x1, a0, a1));
    x_norm = sqrt_rn(wave_tree_sum_all(pair_dot(x0, x1, x0, x1)) + eps);
    const float sim = __fdiv_rn(dot, x_norm * a_norm);
    kp = sim < thr;
  } else if constexpr (A16) {  // tritonModules.py:55-58 in the keys' 16-bit arithmetic
    const float d0 = round16<DT>(x0 - a0), d1 = round16<DT>(x1 - a1);
    const float p0 = round16<DT>(d0 * d0), p1 = round16<DT>(d1 * d1);
    kp = wave_tree_sum_all_r16<DT>(round16<DT>(p0 + p1)) > thr;
  } else {  // tritonModules.py:55-58
    const float d0 = x0 - a0, d1 = x1 - a1;
    kp = wave_tree_sum_all(pair_dot(d0, d1, d0, d1)) > thr;
  }
  a0 = kp ? x0 : a0;  // tritonModules.py:60-63
  a1 = kp ? x1 : a1;
  if (COS) a_norm = kp ? x_norm : a_norm;
  return kp;
}

// Keys: a fixed-length batch [B, H, N, D] with the caller's chunk size cs, or (seq.cu set)
// a ragged batch of [T, H, D] tensors where sequence b is chunked by the reference's rule
// on its own length: min(cs, N_b) rows per chunk, or ceil(N_b / divide_to) when
// divide_to > 0 (modeling_llama.py:602-610).  keep is [B, H, N] for a fixed batch and
// [H, T] (row h * keep_sh + token) for a ragged one; chunk_counts is [B, H, nc].
template <bool COS, bool A16, int DT>
__global__ __launch_bounds__(256) void select_kernel(
    const uint16_t* __restrict__ k, int64_t sk_b, int64_t sk_h, int64_t sk_n, int H, int64_t N,
    int D, int64_t cs, int64_t nc, int64_t total_chunks, float thr, int32_t* __restrict__ keep,
    int32_t* __restrict__ chunk_counts, SeqMap seq, int64_t keep_sh, int divide_to) {
#pragma clang fp contract(off)
  const int lane = threadIdx.x & 63;
  const int64_t w = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (w >= total_chunks) return;
  const int64_t bh = w / nc;
  const int64_t c = w - bh * nc;
  const int64_t b = bh / H, h = bh - (bh / H) * H;
  const int64_t Nb = seq.cu ? seq.len((int)b) : N;
  int64_t csb = cs;
  if (seq.cu) csb = divide_to > 0 ? (Nb + divide_to - 1) / divide_to : (cs < Nb ? cs : Nb);
  if (Nb <= 0 || c * csb >= Nb) {  // tritonModules.py:34-35 (count stays 0, modeling_llama.py:637)
    if (lane == 0) chunk_counts[w] = 0;
    return;
  }
  // rows are 32-bit from here on (N < 2^31)
  const int s = (int)(c * csb);
  const int e = (int)((c * csb + csb < Nb) ? c * csb + csb : Nb);
  using KT = SelKey<DT>;
  using Row = typename KT::Row;
  const typename KT::Elem* base =
      (const typename KT::Elem*)(const void*)k + seq.base((int)b, sk_b, sk_n) + h * sk_h + 2 * lane;
  const bool active = 2 * lane < D;
  int32_t* keep_row = keep + (seq.cu ? h * keep_sh + seq.start((int)b) : bh * N);
  auto row_bits = [&](int r) -> Row {
    return (active && r < e) ? *(const Row*)(base + (int64_t)r * sk_n) : Row{};
  };

  const Row a_bits = row_bits(s);
  float a0 = KT::lo(a_bits), a1 = KT::hi(a_bits);
  float a_norm = 0.0f;
  if (COS) a_norm = sqrt_rn(wave_tree_sum_all(pair_dot(a0, a1, a0, a1)) + 1e-8f);
  if (lane == 0) keep_row[s] = 1;  // row s is an anchor (tritonModules.py:41)
  int count = 1;

  // Rows s + 1 .. e - 1 in batches of 32, each loaded one batch ahead (the loads never
  // depend on the decisions); a batch's 32 decisions are stored by lanes 0..31.
  Row cur[kSelBatch], nxt[kSelBatch];
#pragma unroll
  for (int j = 0; j < kSelBatch; ++j) cur[j] = row_bits(s + 1 + j);
  for (int i0 = s + 1; i0 < e; i0 += kSelBatch) {
#pragma unroll
    for (int j = 0; j < kSelBatch; ++j) nxt[j] = row_bits(i0 + kSelBatch + j);
    uint32_t bb = 0;
    if (i0 + kSelBatch <= e) {
#pragma unroll
      for (int j = 0; j < kSelBatch; ++j)
        bb |= (uint32_t)select_step<COS, A16, DT>(KT::lo(cur[j]), KT::hi(cur[j]), a0, a1, a_norm, thr) << j;
    } else {
#pragma unroll
      for (int j = 0; j < kSelBatch; ++j)
        if (i0 + j < e)
          bb |= (uint32_t)select_step<COS, A16, DT>(KT::lo(cur[j]), KT::hi(cur[j]), a0, a1, a_norm, thr) << j;
    }
    count += __builtin_popcount(bb);  // tritonModules.py:68
    if (lane < kSelBatch && i0 + lane < e) keep_row[i0 + lane] = (int32_t)((bb >> lane) & 1u);
#pragma unroll
    for (int j = 0; j < kSelBatch; ++j) cur[j] = nxt[j];
  }
  if (lane == 0) chunk_counts[w] = count;  // tritonModules.py:68-69
}

// ---- two pairs per wave, one per 32-lane half ----
// Lane q of a half holds head-dimension slots 4q .. 4q+3 of a row, so a wave decides two
// pairs in one instruction stream.  The tree keeps its pairing: levels 1-2 add slots
// inside the lane, lane^1, lane^2, the 8-lane and the 16-lane mirror give levels 3-6, and
// v_permlane16_swap pairs the two 16-lane rows of each half for level 7 -- the blocks
// that the one-row-per-wave tree pairs at each level, so the sums are bit-identical.
template <bool R16, int DT>
__device__ __forceinline__ float half_tree_sum(float p0, float p1, float p2, float p3) {
#pragma clang fp contract(off)
  auto r = [](float v) {
    if constexpr (R16) return round16<DT>(v);
    else return v;
  };
  float t = r(r(p0 + p1) + r(p2 + p3));
  t = r(t + dpp_f32<kDppXor1>(t));
  t = r(t + dpp_f32<kDppXor2>(t));
  t = r(t + dpp_f32<kDppHalfMirror>(t));
  t = r(t + dpp_f32<kDppMirror>(t));
  const auto sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(t), __float_as_uint(t), false, false);
  return r(__uint_as_float(sw[0]) + __uint_as_float(sw[1]));
}

// Four slots of a row.
template <int DT>
struct HalfKey {
  using Row = u32x2;
  static __device__ __forceinline__ float at(Row w, int i) {
    return i & 1 ? E16<DT>::hi(w[i >> 1]) : E16<DT>::lo(w[i >> 1]);
  }
};
template <>
struct HalfKey<DA_F32> {
  using Row = f32x4;
  static __device__ __forceinline__ float at(Row w, int i) { return w[i]; }
};

// A half's row's norm as the cosine test takes it (tritonModules.py:48-54).
template <int DT>
__device__ __forceinline__ float half_norm(typename HalfKey<DT>::Row xb) {
#pragma clang fp contract(off)
  float p[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) p[i] = HalfKey<DT>::at(xb, i) * HalfKey<DT>::at(xb, i);
  return sqrt_rn(half_tree_sum<false, DT>(p[0], p[1], p[2], p[3]) + 1e-8f);
}

// select_step's decision for the row (x) and the anchor (a) a 32-lane half holds, with their
// norms (the cosine test alone reads them).
template <bool COS, bool A16, int DT>
__device__ __forceinline__ bool half_keep(typename HalfKey<DT>::Row xb, typename HalfKey<DT>::Row ab, float xn,
                                          float an, float thr) {
#pragma clang fp contract(off)
  float x[4], a[4], p[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    x[i] = HalfKey<DT>::at(xb, i);
    a[i] = HalfKey<DT>::at(ab, i);
  }
  if constexpr (COS) {  // tritonModules.py:48-54
    const float dot = half_tree_sum<false, DT>(x[0] * a[0], x[1] * a[1], x[2] * a[2], x[3] * a[3]);
    return __fdiv_rn(dot, xn * an) < thr;
  } else if constexpr (A16) {  // tritonModules.py:55-58 in the keys' 16-bit arithmetic
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float d = round16<DT>(x[i] - a[i]);
      p[i] = round16<DT>(d * d);
    }
    return half_tree_sum<true, DT>(p[0], p[1], p[2], p[3]) > thr;
  } else {  // tritonModules.py:55-58
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float d = x[i] - a[i];
      p[i] = d * d;
    }
    return half_tree_sum<false, DT>(p[0], p[1], p[2], p[3]) > thr;
  }
}
template <bool COS, bool A16, int DT>
__device__ __forceinline__ bool half_keep(typename HalfKey<DT>::Row xb, typename HalfKey<DT>::Row ab, float thr) {
  return half_keep<COS, A16, DT>(xb, ab, COS ? half_norm<DT>(xb) : 0.0f, COS ? half_norm<DT>(ab) : 0.0f, thr);
}

// The lower halves of x and y side by side, then their upper ones.
template <typename Row>
__device__ __forceinline__ void swap_rows(const Row x, const Row y, Row& lower, Row& upper) {
#pragma unroll
  for (int i = 0; i < (int)(sizeof(Row) / 4); ++i) {
    const auto xi = x[i], yi = y[i];  // scalars: a bit cast of the element itself takes element 0
    const auto sw = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, xi),
                                                     __builtin_bit_cast(uint32_t, yi), false, false);
    const uint32_t lo = sw[0], up = sw[1];
    using E = std::remove_cv_t<decltype(xi)>;
    lower[i] = __builtin_bit_cast(E, lo);
    upper[i] = __builtin_bit_cast(E, up);
  }
}
__device__ __forceinline__ void swap_rows(const float x, const float y, float& lower, float& upper) {
  const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false);
  lower = __uint_as_float(sw[0]);
  upper = __uint_as_float(sw[1]);
}

// ---- two chunks per wave, one per 32-lane half ----
// select_step for the row a 32-lane half holds (x: four slots); rows with `valid` false
// are never kept.
template <bool COS, bool A16, int DT>
__device__ __forceinline__ bool half_step(const uint2 xb, float (&a)[4], float& a_norm, float thr, bool valid) {
#pragma clang fp contract(off)
  const float x[4] = {E16<DT>::lo(xb.x), E16<DT>::hi(xb.x), E16<DT>::lo(xb.y), E16<DT>::hi(xb.y)};
  bool kp;
  float x_norm = 0.0f;
  if (COS) {  // tritonModules.py:48-54
    const float dot = half_tree_sum<false, DT>(x[0] * a[0], x[1] * a[1], x[2] * a[2], x[3] * a[3]);
    x_norm = sqrt_rn(half_tree_sum<false, DT>(x[0] * x[0], x[1] * x[1], x[2] * x[2], x[3] * x[3]) + 1e-8f);
    kp = __fdiv_rn(dot, x_norm * a_norm) < thr;
  } else if (A16) {  // tritonModules.py:55-58 in the keys' 16-bit arithmetic
    float p[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float d = round16<DT>(x[i] - a[i]);
      p[i] = round16<DT>(d * d);
    }
    kp = half_tree_sum<true, DT>(p[0], p[1], p[2], p[3]) > thr;
  } else {  // tritonModules.py:55-58
    float p[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float d = x[i] - a[i];
      p[i] = d * d;
    }
    kp = half_tree_sum<false, DT>(p[0], p[1], p[2], p[3]) > thr;
  }
  kp = kp && valid;
#pragma unroll
  for (int i = 0; i < 4; ++i) a[i] = kp ? x[i] : a[i];  // tritonModules.py:60-63
  if (COS) a_norm = kp ? x_norm : a_norm;
  return kp;
}

// The chunks as select_kernel walks them, two per wave (chunk 2 w + half).  Needs D a
// multiple of 4 and 8-byte aligned rows.
template <bool COS, bool A16, int DT>
__global__ __launch_bounds__(256) void select_pair_kernel(
    const uint16_t* __restrict__ k, int64_t sk_b, int64_t sk_h, int64_t sk_n, int H, int64_t N,
    int D, int64_t cs, int64_t nc, int64_t total_chunks, float thr, int32_t* __restrict__ keep,
    int32_t* __restrict__ chunk_counts, SeqMap seq, int64_t keep_sh, int divide_to) {
#pragma clang fp contract(off)
  const int lane = threadIdx.x & 63;
  const int q = lane & 31;
  const int64_t w = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * 2 + (lane >> 5);
  // rows [s, e) of this half's chunk; none for a chunk past the grid or the sequence
  int s = 0, e = 0;
  int32_t* keep_row = keep;
  const uint16_t* base = k;
  if (w < total_chunks) {
    const int64_t bh = w / nc;
    const int64_t c = w - bh * nc;
    const int64_t b = bh / H, h = bh - (bh / H) * H;
    const int64_t Nb = seq.cu ? seq.len((int)b) : N;
    int64_t csb = cs;
    if (seq.cu) csb = divide_to > 0 ? (Nb + divide_to - 1) / divide_to : (cs < Nb ? cs : Nb);
    if (Nb > 0 && c * csb < Nb) {
      s = (int)(c * csb);
      e = (int)((c * csb + csb < Nb) ? c * csb + csb : Nb);
      base = k + seq.base((int)b, sk_b, sk_n) + h * sk_h + 4 * q;
      keep_row = keep + (seq.cu ? h * keep_sh + seq.start((int)b) : bh * N);
    } else if (q == 0) {
      chunk_counts[w] = 0;  // tritonModules.py:34-35 (count stays 0, modeling_llama.py:637)
    }
  }
  const bool active = 4 * q < D;
  auto row_bits = [&](int r) -> uint2 {
    return (active && r < e) ? *(const uint2*)(base + (int64_t)r * sk_n) : uint2{0u, 0u};
  };
  const uint2 ab = row_bits(s);
  float a[4] = {E16<DT>::lo(ab.x), E16<DT>::hi(ab.x), E16<DT>::lo(ab.y), E16<DT>::hi(ab.y)};
  float a_norm = 0.0f;
  if (COS)
    a_norm = sqrt_rn(half_tree_sum<false, DT>(a[0] * a[0], a[1] * a[1], a[2] * a[2], a[3] * a[3]) + 1e-8f);
  if (q == 0 && e > s) keep_row[s] = 1;  // row s is an anchor (tritonModules.py:41)
  int count = 1;
  // batches of both halves (wave-uniform): the longer of the two walks
  const int nbh = e > s ? (e - s - 1 + kSelBatch - 1) / kSelBatch : 0;
  const int nb = max(__builtin_amdgcn_readlane(nbh, 0), __builtin_amdgcn_readlane(nbh, 32));
  uint2 cur[kSelBatch], nxt[kSelBatch];
#pragma unroll
  for (int j = 0; j < kSelBatch; ++j) cur[j] = row_bits(s + 1 + j);
  for (int bi = 0; bi < nb; ++bi) {
    const int i0 = s + 1 + bi * kSelBatch;
#pragma unroll
    for (int j = 0; j < kSelBatch; ++j) nxt[j] = row_bits(i0 + kSelBatch + j);
    uint32_t bb = 0;
#pragma unroll
    for (int j = 0; j < kSelBatch; ++j)
      bb |= (uint32_t)half_step<COS, A16, DT>(cur[j], a, a_norm, thr, i0 + j < e) << j;
    count += __builtin_popcount(bb);  // tritonModules.py:68
    if (i0 + q < e) keep_row[i0 + q] = (int32_t)((bb >> q) & 1u);
#pragma unroll
    for (int j = 0; j < kSelBatch; ++j) cur[j] = nxt[j];
  }
  if (q == 0 && e > s) chunk_counts[w] = count;  // tritonModules.py:68-69
}

// ---- the banded walk ----
// The chain of the walk above is one exact distance per row (about 30 dependent
// instructions, 0.14 us), 511 of them in a chunk, whatever the number of chunks.  But which
// rows are compared with which anchor only matters after the fact: with
//     next(i) = the first row after i that is kept against anchor i
// known for every row i, the anchors are 0, next(0), next(next(0)), ...  select_band_kernel
// finds next(i) for all rows of a chunk at once.  One workgroup of 8 waves takes a chunk in
// segments of 512 rows, a wave two tiles of 32 anchors each:
//
// 1. Gram tiles (v_mfma_f32_32x32x16): the wave's anchors against their own tile and the
//    next one, i.e. the 32 to 63 rows that follow each anchor.  With the rows' squared norms
//    (fp32) each pair's distance (or cosine) follows to within a proven bound, and the pair
//    is kept, dropped or open (three states, two bits, in the anchor's lane).
// 2. Where these bits say that the rest would cost more than the serial walk (a wave's anchors
//    have more open rows before their first kept one than kBandAhead, or more than kBandFar of
//    them have no row at all: pairs about as far apart as the threshold, fp32 keys close together
//    against their norms, one key in sixteen kept and fewer), all waves leave out 3.
// 3. The open pairs that come first in an anchor's row of bits are decided by the exact tree
//    of the walk, two per wave and four such in one instruction stream, until every anchor's first
//    kept row is known (about 0.4 pairs an anchor in bf16 arithmetic at one key in four kept,
//    near none in fp32 arithmetic); an anchor that keeps none of its tiles' rows looks at further
//    tiles.  Both within a budget.
// 4. Each wave follows the chain inside its 64 rows from all of them at once (pointer
//    doubling between lanes), one wave joins the eight blocks.  Past an anchor whose next is not
//    known (2, or 3's budget spent) that wave walks on, two rows a step, to the end of such blocks.
//
// Every decision is either proven by its bound or the exact tree's, so the result is the
// walk's bit for bit.  The bounds, with u the unit roundoff of the walk's arithmetic:
// * Gram: the products of 16-bit elements are exact and the 128 of them (and the norms'
//   squares) are added in fp32, so |e - d2| <= 2^-15 (n_a + n_c) for e = n_a + n_c - 2 g (128
//   additions of at most 2^-23 of sum |x y| <= (n_a + n_c) / 2 each, twice, and the norms').
//   fp32 keys are rounded to bf16 for the products (u = 2^-8 an element): 2^-6.9 instead.
// * The walk's own distance S rounds the difference (twice in the square), the square and
//   seven tree levels: d2 (1 - u)^10 <= S <= d2 (1 + u)^10.  In fp16 a square below 2^-14 is
//   rounded to a multiple of 2^-24: 2^-17 more for 128 of them; sums past 65504 become
//   infinite, so nothing above 60000 is dropped.
// * Cosine: |sim - g / sqrt((n_a + 1e-8)(n_c + 1e-8))| <= 2^-14 (2^-6.5 for fp32 keys).
// * Rows with a norm at or above 2^120 (or infinite, or NaN) leave all their pairs open; a
//   threshold below 1e-28 drops nothing, and nothing below 1e-30 is kept unseen.
//
// Measured, the selection alone, 8 heads, in brackets the serial walk.  bf16 keys in their own
// arithmetic, one in four kept: 4096 keys 21 us (72), 32768 35 (73), 8192 in one chunk 0.24 ms
// (1.07); one in eight 30 and 47, one in sixteen 64 and 83, one in 64 65 and 74, none 59 and 68:
// from one in sixteen on most of it is the walk.  4096 fp32 keys: one in four 22 (60), none 54;
// 32768 bf16 keys and the cosine test 24 (104), none 79.  What is left at few chunks is a chain of
// loads (the tiles, the exact decisions' rows, five or six streams a wave).  Without 2 and the walk
// in 4 one wave scanned on alone, eight rows a load: up to four times the serial walk's time.
constexpr int kBandSeg = 512, kBandWaves = 8;
constexpr int kBandEval = 4;     // exact decisions in one instruction stream, two each
constexpr int kBandRounds = 16;  // streams a wave spends on its 64 anchors
constexpr int kBandAhead = 144;  // open rows before the first kept one, over a wave's anchors, that are too many
constexpr int kBandFar = 6;      // anchors without a candidate in their tiles that are too many
constexpr int kBandTiles = 4;    // more tiles it looks at for anchors whose own hold none
constexpr int kWalkRows = 16;    // rows the walk loads ahead

struct BandBounds {
  float c_lo, c_hi;  // e's lower and upper bound: c (n_a + n_c) - 2 g
  float keep, drop;  // kept above / dropped below (Euclidean), kept below / dropped above (cosine)
};

// The bounds of one threshold (host).
static BandBounds band_bounds(bool cosine, bool a16, int dtype, float thr) {
  BandBounds b = {};
  const double t = thr;
  if (cosine) {
    const double d = dtype == DA_F32 ? std::ldexp(1.0, -6) * 0.70710678 : std::ldexp(1.0, -14);
    b.keep = (float)(t - d - 1e-6);
    b.drop = (float)(t + d + 1e-6);
    return b;
  }
  const double g = dtype == DA_F32 ? 0.0084 : std::ldexp(1.0, -15);
  const double u = !a16 || dtype == DA_F32 ? std::ldexp(1.0, -24) : std::ldexp(1.0, dtype == DA_BF16 ? -8 : -11);
  const double tiny = a16 && dtype == DA_F16 ? std::ldexp(1.0, -17) : 0.0;
  const double slack = 1.0 + std::ldexp(1.0, -18);  // the bounds' own fp32 arithmetic
  b.c_lo = (float)(1.0 - g);
  b.c_hi = (float)(1.0 + g);
  b.keep = (float)std::max((t + tiny) / std::pow(1.0 - u, 10) * (t > 0 ? slack : 1.0), 1e-30);
  double drop = (t - tiny) / std::pow(1.0 + u, 10) / slack;
  if (a16 && dtype == DA_F16) drop = std::min(drop, 60000.0);
  b.drop = t < 1e-28 ? -INFINITY : (float)drop;
  return b;
}

// A tile of 32 rows as matrix operands: lane (ql, hl) holds dims 16 t + 8 hl .. + 7 of row
// ql, and the lane's share of the row's squared norm.
template <int DT>
struct BandTile {
  u32x4 w[8];
  float n;
};

// The loads go out together: chunks at or past D repeat the row's last one and are zeroed
// after (a guarded load would be waited for before the next one).
template <int DT, bool FULL>
__device__ __forceinline__ void band_load(BandTile<DT>& x, const typename SelKey<DT>::Elem* row, int D, int hl) {
  // opaque: the chunks' limits are formed here, not held in 16 scalar registers over the loops
  if constexpr (!FULL) asm("" : "+s"(D));
  if constexpr (DT == DA_F32) {
    // converted here: the norm is of the fp32 elements, the products of their bf16 roundings
    f32x4 lo[8], hi[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const int d = FULL ? 16 * t + 8 * hl : min(16 * t + 8 * hl, D - 8);
      lo[t] = *(const f32x4*)(row + d);
      hi[t] = *(const f32x4*)(row + d + 4);
    }
    x.n = 0.0f;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const bool in = FULL || 16 * t + 8 * hl < D;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        lo[t][i] = in ? lo[t][i] : 0.0f;
        hi[t][i] = in ? hi[t][i] : 0.0f;
        x.n = __builtin_fmaf(lo[t][i], lo[t][i], __builtin_fmaf(hi[t][i], hi[t][i], x.n));
      }
      x.w[t] = u32x4{pack_bf16x2(lo[t][0], lo[t][1]), pack_bf16x2(lo[t][2], lo[t][3]),
                     pack_bf16x2(hi[t][0], hi[t][1]), pack_bf16x2(hi[t][2], hi[t][3])};
    }
  } else {
    if constexpr (FULL) {
#pragma unroll
      for (int t = 0; t < 8; ++t) x.w[t] = *(const u32x4*)(row + 8 * hl + 16 * t);
    } else {
#pragma unroll
      for (int t = 0; t < 8; ++t) x.w[t] = *(const u32x4*)(row + min(16 * t + 8 * hl, D - 8));
#pragma unroll
      for (int t = 0; t < 8; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) x.w[t][i] = 16 * t + 8 * hl < D ? x.w[t][i] : 0u;
    }
  }
}

// Gram tile: lane (ql, hl) gets row ql of b against rows 8 (r / 4) + 4 hl + r % 4 of a.
template <int DT>
__device__ __forceinline__ f32x16 band_gram(const BandTile<DT>& a, const BandTile<DT>& b) {
  f32x16 g = f32x16{};
#pragma unroll
  for (int t = 0; t < 8; ++t) g = E16<DT == DA_F16 ? DA_F16 : DA_BF16>::mfma(a.w[t], b.w[t], g);
  return g;
}

// The squared norm of row ql, in both halves: the diagonal of the tile's own Gram tile
// (an eighth of the instructions of unpacking and squaring the row).
template <int DT>
__device__ __forceinline__ float band_norm(const BandTile<DT>& x, int ql, int hl) {
  float n = 0.0f;
  if constexpr (DT == DA_F32) {
    n = x.n;
  } else {
    const f32x16 g = band_gram<DT>(x, x);
#pragma unroll
    for (int r = 0; r < 16; ++r) n = ql - 4 * hl == 8 * (r >> 2) + (r & 3) ? g[r] : n;
  }
  return n + swap_halves(n);
}

// FULL: D = 128 (rows at immediate offsets from one address; the registers of 16-bit keys then
// hold two workgroups a CU).
template <bool COS, bool A16, int DT, bool FULL>
__global__ __launch_bounds__(64 * kBandWaves) __attribute__((amdgpu_waves_per_eu(FULL && DT != DA_F32 ? 4 : 2)))
void select_band_kernel(
    const uint16_t* __restrict__ k, int64_t sk_b, int64_t sk_h, int64_t sk_n, int H, int64_t N,
    int D_arg, int cs, int nc, float thr, BandBounds bounds, int32_t* __restrict__ keep,
    int32_t* __restrict__ chunk_counts, SeqMap seq, int64_t keep_sh, int divide_to) {
  __shared__ float s_norm[kBandWaves][2][32];     // a wave's candidates' norms (cosine: 1 / norm)
  __shared__ u32x2 s_path[kBandSeg];              // the chain from a row, inside its block of 64
  __shared__ int s_to[kBandSeg];                  // and where it leads, from the block's first row
  __shared__ int s_from[kBandSeg];
  __shared__ uint64_t s_bits[kBandSeg / 64];
  __shared__ u32x4 s_ku[kBandSeg];                // K and U of a row, put down while its wave looks at more tiles
  __shared__ int s_hard[kBandWaves];              // the wave's tiles say that the walk is faster
  __shared__ int s_left[kBandWaves];              // the wave left its anchors to the walk
  __shared__ int s_cur;
  const int D = FULL ? 128 : D_arg;
  const int tid = threadIdx.x;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  int lane = tid & 63, ql = lane & 31, hl = lane >> 5;
  // 32 bits are enough for the chunk's place (the grid, N and the chunks are below 2^31)
  const unsigned w = blockIdx.x;
  const unsigned bh = w / (unsigned)nc;
  const unsigned c = w - bh * (unsigned)nc;
  const unsigned b = bh / (unsigned)H, h = bh - b * (unsigned)H;
  const unsigned Nb = seq.cu ? seq.len((int)b) : (int)N;
  unsigned csb = (unsigned)cs;
  if (seq.cu) csb = divide_to > 0 ? (Nb + divide_to - 1) / divide_to : min(csb, Nb);
  const int64_t s64 = (int64_t)c * csb;
  if (Nb == 0 || s64 >= Nb) {  // tritonModules.py:34-35 (count stays 0, modeling_llama.py:637)
    if (tid == 0) chunk_counts[w] = 0;
    return;
  }
  const int s = (int)s64;
  const int e = (int)(s64 + csb < Nb ? s64 + csb : Nb);
  using Elem = typename SelKey<DT>::Elem;
  using Row = typename HalfKey<DT>::Row;
  const Elem* base = (const Elem*)(const void*)k + seq.base((int)b, sk_b, sk_n) + (int64_t)h * sk_h;
  int32_t* keep_row = keep + (seq.cu ? (int64_t)h * keep_sh + seq.start((int)b) : (int64_t)bh * N);
  // the exact decisions' operands: a half-wave's row
  auto row_bits = [&](int r) -> Row {
    Row x = *(const Row*)(base + (int64_t)r * sk_n + (FULL ? 4 * ql : min(4 * ql, D - 4)));
    if constexpr (!FULL) {
#pragma unroll
      for (int i = 0; i < (int)(sizeof(Row) / 4); ++i) x[i] = 4 * ql < D ? x[i] : 0;
    }
    return x;
  };
  auto load_tile = [&](BandTile<DT>& x, int tb) {  // rows past the chunk repeat its last one
    band_load<DT, FULL>(x, base + (int64_t)min(tb + ql, e - 1) * sk_n, D, hl);
  };

  int cur = s;  // the next anchor
  int count = 0;
  const int seg = blockDim.x;  // rows a segment: 64 a wave
  // the wave that joins the blocks and walks: another SIMD's for each of a CU's workgroups, in
  // whatever order it gets them
  const int lead = (int)((blockIdx.x >> 3) + (blockIdx.x >> 8)) & (seg >= 256 ? 3 : seg >= 128 ? 1 : 0);
  // ---- the walk of the rows from r on, two a step: both against the anchor, one a half, and
  // the second against the first (of two steps at once), which does not wait for the anchor.
  // Ends at the first anchor at or past `stop`, which it returns; the kept rows before go into
  // s_bits (of the segment at sb). ----
  auto walk_on = [&](Row a, int r, const int stop, const int sb) -> int {
    float an = COS ? half_norm<DT>(a) : 0.0f;
    Row x[kWalkRows / 2], y[kWalkRows / 2];
    auto load = [&](Row (&v)[kWalkRows / 2], const int from) {
      if (from + kWalkRows <= e) {
        const Elem* p = base + (int64_t)(from + hl) * sk_n + (FULL ? 4 * ql : min(4 * ql, D - 4));
#pragma unroll
        for (int j = 0; j < kWalkRows / 2; ++j, p += 2 * sk_n) {
          v[j] = *(const Row*)p;
          if constexpr (!FULL) {
#pragma unroll
            for (int i = 0; i < (int)(sizeof(Row) / 4); ++i) v[j][i] = 4 * ql < D ? v[j][i] : 0;
          }
        }
      } else {
#pragma unroll
        for (int j = 0; j < kWalkRows / 2; ++j) v[j] = row_bits(min(from + 2 * j + hl, e - 1));
      }
    };
    load(x, r);
    for (; r < e; r += kWalkRows) {
      load(y, r + kWalkRows);
      uint32_t bb = 0;
#pragma unroll
      for (int j = 0; j < kWalkRows / 2; j += 2) {
        Row odd, even;  // rows 1 and 3, and 2 and 4, of these four
        swap_rows(x[j], x[j + 1], odd, even);
        float xn[2] = {}, on = 0.0f, en = 0.0f;
        if constexpr (COS) {
          xn[0] = half_norm<DT>(x[j]);
          xn[1] = half_norm<DT>(x[j + 1]);
          swap_rows(xn[0], xn[1], on, en);
        }
        const uint64_t kc = __ballot(half_keep<COS, A16, DT>(even, odd, en, on, thr));
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          Row first, second;
          float n1 = 0.0f, n2 = 0.0f;
          swap_rows(x[j + u], x[j + u], first, second);
          if constexpr (COS) swap_rows(xn[u], xn[u], n1, n2);
          const uint64_t ka = __ballot(half_keep<COS, A16, DT>(x[j + u], a, xn[u], an, thr));
          const bool k12 = (kc >> (32 * u)) & 1ull;
          const bool k1 = ka & 1ull, k2 = k1 ? k12 : (ka >> 32) & 1ull;
          bb |= (uint32_t)k1 << (2 * (j + u)) | (uint32_t)k2 << (2 * (j + u) + 1);
#pragma unroll
          for (int i = 0; i < (int)(sizeof(Row) / 4); ++i) a[i] = k2 ? second[i] : k1 ? first[i] : a[i];
          if constexpr (COS) an = k2 ? n2 : k1 ? n1 : an;
        }
      }
      if (e - r < kWalkRows) bb &= (1u << (e - r)) - 1u;
      const int in = stop - r;  // rows of this batch before `stop`
      const uint32_t mine = in >= kWalkRows ? ~0u : in > 0 ? (1u << in) - 1u : 0u;
      count += __builtin_popcount(bb & mine);
      const int rel = r + lane - sb;
      if (lane < kWalkRows && ((bb & mine) >> lane) & 1u)
        atomicOr((unsigned long long*)&s_bits[rel >> 6], 1ull << (rel & 63));
      if (bb & ~mine) return r + __builtin_ctz(bb & ~mine);
#pragma unroll
      for (int j = 0; j < kWalkRows / 2; ++j) x[j] = y[j];
    }
    return e;
  };
  for (int sb = s; sb < e; sb += seg) {
    // opaque: what derives from the lane is formed here, not held in registers over the loop
    lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));
    ql = lane & 31;
    hl = lane >> 5;
    count = __builtin_amdgcn_readfirstlane(count);
    const int se = min(sb + seg, e);
    if (cur < se) {
      const int tb = sb + 64 * wid;  // the wave's anchors: tiles tb and tb + 32
      const bool active = tb < se && tb + 63 >= cur;
      BandTile<DT> x, y;
      // K, U: the kept and the open rows among those from tb + base to tb + end: the 64 from the
      // anchor's tile on, or, where these hold none, the tile looked at last (base 64 and up)
      uint64_t K = 0, U = 0;
      int base = lane & 32;
      auto window_end = [&]() { return base + (base < 64 ? 64 : 32); };
      const bool mine = tb + lane >= cur && tb + lane < e;
      constexpr uint32_t huge = 0x7b800000u;  // 2^120
      auto is_bad = [](float n) { return (__float_as_uint(n) & 0x7fffffffu) >= huge; };
      auto scaled = [](float n) { return COS ? __builtin_amdgcn_rsqf(n + 1e-8f) : n; };
      // The kept and the open ones of a tile's rows (cand, its norms in s_norm[wid][j], its
      // first row at tb + pos) against the lane's anchor, row ql of the tile in x
      auto tile_bits = [&](const BandTile<DT>& cand, const int j, const float na, const bool bad,
                           const uint32_t bad_rows, const int pos, uint32_t& kept, uint32_t& open) {
        const f32x16 g = band_gram<DT>(cand, x);
        uint32_t kb = 0, db = 0;
        // S^T layout: the lane holds anchor ql and candidates 8 q + 4 hl + i
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const f32x4 nc4 = *(const f32x4*)(&s_norm[wid][j][8 * q + 4 * hl]);
          uint32_t kq = 0, dq = 0;  // the bits of these four: 1, 2, 4 and 8 need no register
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float dot = g[4 * q + i];
            const uint32_t bit = 1u << i;
            if (COS) {
              const float sim = dot * (na * nc4[i]);
              kq |= sim < bounds.keep ? bit : 0u;
              dq |= sim > bounds.drop ? bit : 0u;
            } else {
              const float n2 = na + nc4[i];
              kq |= __builtin_fmaf(n2, bounds.c_lo, -2.0f * dot) > bounds.keep ? bit : 0u;
              dq |= __builtin_fmaf(n2, bounds.c_hi, -2.0f * dot) < bounds.drop ? bit : 0u;
            }
          }
          asm("" : "+v"(kq), "+v"(dq));  // or the shift would go into the bits
          kb |= kq << (8 * q);
          db |= dq << (8 * q);
        }
        kb <<= 4 * hl;
        db <<= 4 * hl;
        kb |= __shfl_xor(kb, 32, 64);
        db |= __shfl_xor(db, 32, 64);
        const int lim = e - (tb + pos);  // rows of the tile before the chunk's end
        const uint32_t valid = lim >= 32 ? ~0u : lim > 0 ? (1u << lim) - 1u : 0u;
        const uint32_t sure = bad ? 0u : ~bad_rows;
        kept = kb & valid & sure;
        open = ~((kb | db) & sure) & valid;
        __builtin_amdgcn_sched_barrier(0);  // one Gram tile's registers at a time
      };
      auto norms_written = [&]() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
      };
      if (active) {
        load_tile(x, tb);
        load_tile(y, tb + 32);
        float nx = band_norm<DT>(x, ql, hl);
#pragma unroll
        for (int half = 0; half < 2; ++half) {
          // ---- anchors: the tile in x; candidates: x and y ----
          const float ny = band_norm<DT>(y, ql, hl);
          if (lane < 32) {
            s_norm[wid][0][ql] = scaled(nx);
            s_norm[wid][1][ql] = scaled(ny);
          }
          const uint32_t bad0 = (uint32_t)__ballot(is_bad(nx)), bad1 = (uint32_t)__ballot(is_bad(ny));
          norms_written();
          uint32_t kept[2], open[2];
          tile_bits(x, 0, scaled(nx), is_bad(nx), bad0, 32 * half, kept[0], open[0]);
          tile_bits(y, 1, scaled(nx), is_bad(nx), bad1, 32 * half + 32, kept[1], open[1]);
          const uint32_t after = ~((2u << ql) - 1u);  // candidates of the own tile: after the anchor
          kept[0] &= after;
          open[0] &= after;
          __builtin_amdgcn_wave_barrier();  // the norms are read before the next tile's are written
          if (half == 0) {
            x = y;
            nx = ny;
            load_tile(y, tb + 64);
          }
          if (hl == half) {  // lane l ends with row tb + l
            K = kept[0] | (uint64_t)kept[1] << 32;
            U = open[0] | (uint64_t)open[1] << 32;
          }
        }
        // Where the bounds decide little (pairs all about as far apart as the threshold, or close
        // together against their norms) or the tiles hold too little (an anchor's next lies
        // further on) the walk is faster, and the wave leaves its rows to it at once.
        const float ahead = (float)__builtin_popcountll(U & ((K & (0ull - K)) - 1ull));
        const bool far = __builtin_popcountll(__ballot(mine && (K | U) == 0 && tb + window_end() < e)) > kBandFar;
        const bool open = __builtin_amdgcn_readfirstlane((int)wave_tree_sum_all(mine ? ahead : 0.0f)) > kBandAhead;
        if (lane == 0) s_hard[wid] = far || open;
      } else if (lane == 0) {
        s_hard[wid] = 0;
      }
      __syncthreads();
      if (active) {
        // one such wave stands for all: none then holds the segment up with rows that the walk
        // passes anyway (bf16 arithmetic, one key in eight kept: at most 128 open and none without
        // a row in any wave; one in sixteen: above the line in every chunk)
        bool hard = __ballot(lane < seg / 64 && s_hard[lane & (kBandWaves - 1)]) != 0;
        int rounds = 0, tiles = 0;
        while (!hard) {
          // ---- exact decisions, until every anchor's first candidate is a kept one ----
          for (;; ++rounds) {
            const uint64_t any = K | U;
            const int first = any ? __builtin_ctzll(any) : 0;
            uint64_t m = __ballot(mine && any != 0 && ((U >> first) & 1ull));
            if (m == 0) break;
            if (rounds == kBandRounds) {
              hard = true;
              break;
            }
            int l[2 * kBandEval];
            Row ra[kBandEval], rx[kBandEval];
            uint64_t kp[kBandEval];
#pragma unroll
            for (int i = 0; i < 2 * kBandEval; ++i) {
              l[i] = m ? __builtin_ctzll(m) : l[i > 0 ? i - 1 : 0];
              m &= m - 1ull;
            }
#pragma unroll
            for (int i = 0; i < kBandEval; ++i) {
              const int f0 = __builtin_amdgcn_readlane(base + first, l[2 * i]);
              const int f1 = __builtin_amdgcn_readlane(base + first, l[2 * i + 1]);
              ra[i] = row_bits(tb + (hl ? l[2 * i + 1] : l[2 * i]));
              rx[i] = row_bits(tb + (hl ? f1 : f0));
            }
#pragma unroll
            for (int i = 0; i < kBandEval; ++i) kp[i] = __ballot(half_keep<COS, A16, DT>(rx[i], ra[i], thr));
#pragma unroll
            for (int i = 0; i < 2 * kBandEval; ++i)
              if (lane == l[i]) {
                U &= ~(1ull << first);
                if ((kp[i >> 1] >> (32 * (i & 1))) & 1ull) K |= 1ull << first;
              }
          }
          // ---- the anchors whose rows so far hold none: tile after tile, until all have one ----
          uint64_t want = __ballot(mine && (K | U) == 0 && tb + window_end() < e);
          if (__builtin_expect(hard || want == 0, 1)) break;
          s_ku[64 * wid + lane] = u32x4{(uint32_t)K, (uint32_t)(K >> 32), (uint32_t)U, (uint32_t)(U >> 32)};
#pragma unroll 1
          for (int half = 0; half < 2; ++half) {
            if ((uint32_t)(want >> (32 * half)) == 0) continue;
            load_tile(x, tb + 32 * half);
            int pos = hl == half && ((want >> lane) & 1ull) ? window_end() : INT_MAX;  // the least of them
#pragma unroll
            for (int d = 32; d >= 1; d >>= 1) pos = min(pos, __shfl_xor(pos, d, 64));
            pos = __builtin_amdgcn_readfirstlane(pos);
            const float nx = band_norm<DT>(x, ql, hl);
#pragma unroll 1
            for (; tb + pos < e && tiles < kBandTiles; pos += 32, ++tiles) {
              load_tile(y, tb + pos);
              const float ny = band_norm<DT>(y, ql, hl);
              if (lane < 32) s_norm[wid][1][ql] = scaled(ny);
              const uint32_t bad1 = (uint32_t)__ballot(is_bad(ny));
              norms_written();
              uint32_t kept, open;
              tile_bits(y, 1, scaled(nx), is_bad(nx), bad1, pos, kept, open);
              __builtin_amdgcn_wave_barrier();
              if (hl == half && ((want >> lane) & 1ull) && pos >= window_end()) {
                base = pos;
                s_ku[64 * wid + lane] = u32x4{kept, 0u, open, 0u};
              }
              want &= ~__ballot(hl == half && base == pos && (kept | open) != 0u);
              if ((uint32_t)(want >> (32 * half)) == 0) break;
            }
          }
          hard = tiles >= kBandTiles;
          norms_written();
          const u32x4 ku = s_ku[64 * wid + lane];
          K = ku[0] | (uint64_t)ku[1] << 32;
          U = ku[2] | (uint64_t)ku[3] << 32;
        }
        // ---- the chain inside the wave's 64 rows, from every row at once: path holds the
        // anchors met from row l on, to is where it leaves them (64 and up), or -1 - the anchor
        // it stops at: one whose next is not known, to be looked for from row s_from on.
        // Six doublings cover 64 steps. ----
        const uint64_t any = K | U;
        const int first = any ? __builtin_ctzll(any) : 0;
        const int at = any ? base + first : min(window_end(), e - tb);
        s_from[64 * wid + lane] = at;
        // (no next: past the block, where the chunk may end inside it)
        int to = (any ? (U >> first) & 1ull : tb + at < e) ? -1 - lane : any ? at : max(at, 64);
        uint32_t lo = lane < 32 ? 1u << ql : 0u, hi = lane < 32 ? 0u : 1u << ql;
#pragma unroll
        for (int d = 0; d < 6; ++d) {
          const int src = (unsigned)to < 64u ? to : lane;
          lo |= (uint32_t)__shfl((int)lo, src, 64);
          hi |= (uint32_t)__shfl((int)hi, src, 64);
          to = __shfl(to, src, 64);
        }
        s_path[64 * wid + lane] = u32x2{lo, hi};
        s_to[64 * wid + lane] = to;
        if (lane == 0) s_left[wid] = hard;
      }
      __syncthreads();
      if (wid == lead) {
        // ---- the segment's chain: one lookup a block of 64 rows ----
        int p = cur - sb;
        if (lane < seg / 64) s_bits[lane] = 0;
        for (int i = 0; i < seg / 64; ++i) {
          uint64_t bits = 0;
          while (p < 64 * (i + 1) && sb + p < se) {
            const u32x2 path = s_path[p];
            const int to = __builtin_amdgcn_readfirstlane(s_to[p]);
            const uint64_t on = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane(path[0]) |
                                (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane(path[1]) << 32;
            bits |= on;
            count += __builtin_popcountll(on);
            if (__builtin_expect(to < 0, 0)) {
              // on from the anchor it stops at, past the blocks that were left to the walk
              const int pa = 64 * i + (-1 - to);
              int j = i + 1;
              while (j < seg / 64 && __builtin_amdgcn_readfirstlane(s_left[j])) ++j;
              p = walk_on(row_bits(sb + pa), sb + __builtin_amdgcn_readfirstlane(s_from[pa]) + 64 * i,
                          min(sb + 64 * j, e), sb) - sb;
            } else {
              p = 64 * i + to;
            }
          }
          if (lane == 0) atomicOr((unsigned long long*)&s_bits[i], (unsigned long long)bits);  // (no wait for a read)
        }
        if (lane == 0) s_cur = sb + p;
      }
      __syncthreads();
      cur = __builtin_amdgcn_readfirstlane(s_cur);
    } else {
      if (tid < seg / 64) s_bits[tid] = 0;
      __syncthreads();
    }
    if (sb + 64 * wid + lane < se) keep_row[sb + 64 * wid + lane] = (int32_t)((s_bits[wid] >> lane) & 1ull);
    __syncthreads();  // the bits are read before the next segment's are written
  }
  if (wid == lead && (threadIdx.x & 63) == 0) chunk_counts[w] = count;  // tritonModules.py:68-69
}

static int launch_select(const void* k, int dtype, int64_t B, int64_t Hkv, int64_t N, int64_t D, int64_t sk_b,
                         int64_t sk_h, int64_t sk_n, float threshold, bool use_cosine, bool a16, int64_t chunk_size,
                         int64_t num_chunks, int32_t* keep, int32_t* chunk_counts, SeqMap seq, int64_t keep_sh,
                         int divide_to, hipStream_t st, const char* who) {
  DA_REQUIRE(((sk_b | sk_h | sk_n) & 1) == 0 && ((uintptr_t)k & (dtype == DA_F32 ? 7 : 3)) == 0,
             "%s: key rows must be %d-byte aligned (even strides)", who, dtype == DA_F32 ? 8 : 4);
  const int64_t total = B * Hkv * num_chunks;
  const int64_t blocks = (total + 3) / 4;
  DA_REQUIRE(blocks < (1ll << 31), "%s: too many chunks", who);
  // The banded walk takes rows it can read 16 bytes at a time.  The line is one round of the chip:
  // two workgroups a CU, one for fp32 keys or other than 128 dims (their registers; fp32 keys of
  // other than 128 dims half a round, 64 chunks 59 against 60 us but 256 77 / 63 with few kept).
  // There its time is 0.2 to 0.65 of the serial walk's with one key in two to eight kept and about
  // the serial walk's with keys that it leaves to its own (0.8 to 1.05, the worst found 1.16: 512
  // chunks of bf16 keys, one in sixteen kept, 84 against 73 us).  A second round doubles the latter
  // and gains little on the former: 1024 chunks 46 us at one key in two, 78 at one in eight, 103 and
  // more from one in sixteen on, against 74; a look at a chunk's first 64 rows before the rest costs
  // 6 us and leaves 97 to 165.  Below 128 rows a chunk is too short to gain (97 rows, 680 chunks:
  // 19.5 against 17.1 us).
  const int per16 = dtype == DA_F32 ? 4 : 8;
  const int64_t rows = seq.cu && divide_to > 0 ? (N + divide_to - 1) / divide_to : std::min(chunk_size, N);
  const int64_t band_max = (dtype == DA_F32 ? 256 : 512) / (D == 128 ? 1 : 2);
  if (rows >= kBandMinRows && total <= band_max && (D & 7) == 0 && ((sk_b | sk_h | sk_n) % per16) == 0 &&
      ((uintptr_t)k & 15) == 0 && std::isfinite(threshold)) {
    const BandBounds bounds = band_bounds(use_cosine, a16, dtype, threshold);
    const unsigned threads = (unsigned)std::min<int64_t>(kBandSeg, (rows + 63) / 64 * 64);
#define DA_BAND_LAUNCH_D(COS, A16, DT, FULL)                                                                  \
  hipLaunchKernelGGL((select_band_kernel<COS, A16, DT, FULL>), dim3((unsigned)total), dim3(threads), 0, st, \
                     (const uint16_t*)k, sk_b, sk_h, sk_n, (int)Hkv, N, (int)D,                            \
                     (int)std::min<int64_t>(chunk_size, N), (int)num_chunks, threshold, bounds, keep,          \
                     chunk_counts, seq, keep_sh, divide_to)
#define DA_BAND_LAUNCH(COS, A16, DT)                                \
  do {                                                              \
    if (D == 128) DA_BAND_LAUNCH_D(COS, A16, DT, true);             \
    else DA_BAND_LAUNCH_D(COS, A16, DT, false);                     \
  } while (0)
    if (dtype == DA_F32) {
      if (use_cosine) DA_BAND_LAUNCH(true, false, DA_F32);
      else DA_BAND_LAUNCH(false, false, DA_F32);
    } else if (dtype == DA_F16) {
      if (use_cosine) DA_BAND_LAUNCH(true, false, DA_F16);
      else if (a16) DA_BAND_LAUNCH(false, true, DA_F16);
      else DA_BAND_LAUNCH(false, false, DA_F16);
    } else {
      if (use_cosine) DA_BAND_LAUNCH(true, false, DA_BF16);
      else if (a16) DA_BAND_LAUNCH(false, true, DA_BF16);
      else DA_BAND_LAUNCH(false, false, DA_BF16);
    }
#undef DA_BAND_LAUNCH
#undef DA_BAND_LAUNCH_D
    return check_launch(who);
  }
  if (dtype == DA_F32) {
    // fp32 keys: one wave per chunk, each lane two fp32 elements; the 16-bit definition
    // does not apply (the keys' own arithmetic is fp32)
    if (use_cosine)
      hipLaunchKernelGGL((select_kernel<true, false, DA_F32>), dim3((unsigned)blocks), dim3(256), 0, st,
                         (const uint16_t*)k, sk_b, sk_h, sk_n, (int)Hkv, N, (int)D, chunk_size, num_chunks, total,
                         threshold, keep, chunk_counts, seq, keep_sh, divide_to);
    else
      hipLaunchKernelGGL((select_kernel<false, false, DA_F32>), dim3((unsigned)blocks), dim3(256), 0, st,
                         (const uint16_t*)k, sk_b, sk_h, sk_n, (int)Hkv, N, (int)D, chunk_size, num_chunks, total,
                         threshold, keep, chunk_counts, seq, keep_sh, divide_to);
    return check_launch(who);
  }
  // From two chunks per SIMD on (256 CUs x 4 SIMDs), one wave per pair of chunks walks
  // both in one instruction stream and leaves the SIMDs one wave each: 79 against 85 us
  // at 131072 keys x 8 heads.  Fewer chunks keep one wave per chunk (the pair layout
  // would leave SIMDs idle).
  if (total >= kSelPairMinChunks && (D & 3) == 0 && ((sk_b | sk_h | sk_n) & 3) == 0 && ((uintptr_t)k & 7) == 0) {
    const int64_t pblocks = (total + 7) / 8;
#define DA_SELPAIR_LAUNCH(COS, A16, DT)                                                                      \
  hipLaunchKernelGGL((select_pair_kernel<COS, A16, DT>), dim3((unsigned)pblocks), dim3(256), 0, st,           \
                     (const uint16_t*)k, sk_b, sk_h, sk_n, (int)Hkv, N, (int)D, chunk_size, num_chunks, total, \
                     threshold, keep, chunk_counts, seq, keep_sh, divide_to)
    if (dtype == DA_F16) {
      if (use_cosine) DA_SELPAIR_LAUNCH(true, false, DA_F16);
      else if (a16) DA_SELPAIR_LAUNCH(false, true, DA_F16);
      else DA_SELPAIR_LAUNCH(false, false, DA_F16);
    } else {
      if (use_cosine) DA_SELPAIR_LAUNCH(true, false, DA_BF16);
      else if (a16) DA_SELPAIR_LAUNCH(false, true, DA_BF16);
      else DA_SELPAIR_LAUNCH(false, false, DA_BF16);
    }
#undef DA_SELPAIR_LAUNCH
    return check_launch(who);
  }
#define DA_SELECT_LAUNCH(COS, A16, DT)                                                                       \
  hipLaunchKernelGGL((select_kernel<COS, A16, DT>), dim3((unsigned)blocks), dim3(256), 0, st, (const uint16_t*)k, \
                     sk_b, sk_h, sk_n, (int)Hkv, N, (int)D, chunk_size, num_chunks, total, threshold, keep,  \
                     chunk_counts, seq, keep_sh, divide_to)
  if (dtype == DA_F16) {
    if (use_cosine) DA_SELECT_LAUNCH(true, false, DA_F16);
    else if (a16) DA_SELECT_LAUNCH(false, true, DA_F16);
    else DA_SELECT_LAUNCH(false, false, DA_F16);
  } else {
    if (use_cosine) DA_SELECT_LAUNCH(true, false, DA_BF16);
    else if (a16) DA_SELECT_LAUNCH(false, true, DA_BF16);
    else DA_SELECT_LAUNCH(false, false, DA_BF16);
  }
#undef DA_SELECT_LAUNCH
  return check_launch(who);
}

}  // namespace da

using namespace da;

extern "C" int da_select(const void* k, int dtype, int64_t B, int64_t Hkv, int64_t N, int64_t D,
                         int64_t sk_b, int64_t sk_h, int64_t sk_n, float threshold, int flags,
                         int64_t chunk_size, int64_t num_chunks, int32_t* keep,
                         int32_t* chunk_counts, void* stream) {
  DA_REQUIRE(k && keep && chunk_counts, "da_select: null pointer");
  DA_REQUIRE((flags & ~(DA_SELECT_COSINE | DA_SELECT_ARITH16)) == 0, "da_select: unknown flags 0x%x", flags);
  const bool use_cosine = flags & DA_SELECT_COSINE;
  const bool a16 = !use_cosine && (flags & DA_SELECT_ARITH16);
  if (dtype != DA_BF16 && dtype != DA_F16 && dtype != DA_F32)
    return set_error(DA_ERR_UNSUPPORTED, "da_select: keys must be bf16, fp16 or fp32");
  DA_REQUIRE(B > 0 && Hkv > 0 && N > 0 && D > 0, "da_select: empty shape");
  if (D > 128 || (D & 1)) return set_error(DA_ERR_UNSUPPORTED, "da_select: head_dim must be even and <= 128 (got %lld)", (long long)D);
  DA_REQUIRE(chunk_size > 0 && num_chunks > 0, "da_select: chunk_size and num_chunks must be positive");
  DA_REQUIRE(N < (1ll << 31), "da_select: sequence too long");
  return launch_select(k, dtype, B, Hkv, N, D, sk_b, sk_h, sk_n, threshold, use_cosine, a16, chunk_size,
                       num_chunks, keep, chunk_counts, SeqMap{nullptr, 0, (int)N}, N, 0, (hipStream_t)stream,
                       "da_select");
}

extern "C" int da_select_varlen(const void* k, int dtype, int64_t B, int64_t Hkv, int64_t T, int64_t D,
                                int64_t sk_t, int64_t sk_h, const int32_t* cu_seqlens, int64_t max_seqlen,
                                float threshold, int flags, int64_t chunk_size, int64_t divide_to,
                                int32_t* keep, int32_t* chunk_counts, int64_t max_chunks, void* stream) {
  const char* who = "da_select_varlen";
  DA_REQUIRE(k && keep && chunk_counts && cu_seqlens, "%s: null pointer", who);
  DA_REQUIRE((flags & ~(DA_SELECT_COSINE | DA_SELECT_ARITH16)) == 0, "%s: unknown flags 0x%x", who, flags);
  const bool use_cosine = flags & DA_SELECT_COSINE;
  const bool a16 = !use_cosine && (flags & DA_SELECT_ARITH16);
  if (dtype != DA_BF16 && dtype != DA_F16 && dtype != DA_F32)
    return set_error(DA_ERR_UNSUPPORTED, "%s: keys must be bf16, fp16 or fp32", who);
  DA_REQUIRE(B > 0 && Hkv > 0 && T > 0 && D > 0, "%s: empty shape", who);
  if (D > 128 || (D & 1)) return set_error(DA_ERR_UNSUPPORTED, "%s: head_dim must be even and <= 128 (got %lld)", who, (long long)D);
  DA_REQUIRE(T < (1ll << 31) && max_seqlen > 0 && max_seqlen <= T, "%s: need 0 < max_seqlen <= total tokens < 2^31", who);
  DA_REQUIRE(divide_to >= 0, "%s: divide_to must be >= 0", who);
  // the chunking rule of modeling_llama.py:602-610, per sequence
  const int64_t cs = chunk_size > 0 ? chunk_size : 0;
  const int div = chunk_size > 0 ? 0 : (divide_to > 0 ? (int)divide_to : 1);
  const int64_t need = chunk_size > 0 ? std::max<int64_t>(1, (max_seqlen + chunk_size - 1) / chunk_size) : div;
  DA_REQUIRE(max_chunks >= need, "%s: max_chunks must be at least %lld", who, (long long)need);
  return launch_select(k, dtype, B, Hkv, max_seqlen, D, 0, sk_h, sk_t, threshold, use_cosine, a16, cs, max_chunks,
                       keep, chunk_counts, SeqMap{cu_seqlens, (int)T, (int)max_seqlen}, T, div,
                       (hipStream_t)stream, who);
}
