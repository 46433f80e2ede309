// Causal GQA flash prefill on gfx950: the dense control and the two-phase
// compressed (delta) prefill share one kernel.
//
// Replaces _attn_fwd_flat (flashAttention.py:5-91) and
// hybrid_compressed_flash_kernel / _sanity / pure_phase1_flash_kernel
// (deltaFlashAttention.py:9-357) with their wrappers (modeling_llama.py:306-451).
//
// Work decomposition.  A workgroup is 4 waves; each wave owns 64 query rows of one query
// head, or 32 where the grid is small (launch_attn_rows).  The 4 waves always read the same KV
// head: with a GQA group of 4 they are 4 query heads of the group on the same 64 (32) rows, so
// every K/V tile staged in LDS serves 4 heads (repeat_kv is never materialised).  With smaller
// groups the waves split 128 or 256 (64 or 128) rows instead.
//
// Logical schedule (deltaFlashAttention.py:58-113).  Phase 1 takes packed blocks of
// 128 anchors while their maximum timestamp is < start_m - W; Phase 2 covers dense
// keys from ((last + 1) / 128) * 128 to the diagonal.  The prefix of safe packed
// blocks is counted over the per-head prefix maxima of the block maxima
// (hybrid_schedule_kernel), which reproduces the reference's stop-at-first-unsafe-block
// loop for any timestamps, including its zero-padding behaviour (fully padded blocks
// have maximum 0).
//
// MFMA formulation.  Scores are computed transposed, S^T = K Q^T, with
// v_mfma_f32_32x32x16_bf16 (the _f16 form for fp16 tensors; the kernels are templated on
// the 16-bit type, and P is rounded to it as the reference rounds p to V's type): K
// (32 keys x 16 dims) comes from LDS as the A operand,
// Q^T is the B operand for the whole key loop.  In the S^T accumulator a lane holds one
// query and 16 keys, so the row sum of the online softmax is in-lane.  The output is
// accumulated transposed too, O^T += V^T P^T: the 16-bit probabilities are already in the
// B-operand layout, and V^T is read from the row-major V tile with transposing LDS reads.
//
// Softmax numerics.  exp2 with the softmax scale folded in: p = 2^(s*c - m*c) with
// c = scale * log2(e) -- the same values as exp(s*scale - m*scale).  In Phase 1
// p is multiplied by the anchor count in fp32 and then rounded to bf16 for the
// P.V product while l accumulates the fp32 weights (deltaFlashAttention.py:86-98).
#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <type_traits>
#include <utility>

#include "da_common.hpp"

namespace da {

constexpr int kD = 128;
constexpr int kBlock = 128;  // logical block of the reference schedule

enum Variant : int { kHybrid = 0, kSanity = 1, kPure = 2, kDense = 3 };

// ts, cnt, their strides, no_count and cnt_is_float are the schedule kernel's: the attention
// kernels do not read them, but without them in the block run 0.6 % slower (32768 tokens, hybrid
// 1.971 against 1.959 ms, both builds in turn; with the strides aligned to 64 bytes all the same).
struct AttnArgs {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  const uint16_t* kp;
  const uint16_t* vp;
  const int32_t* ts;
  const void* cnt;
  uint16_t* out;
  int64_t sq_b, sq_h, sq_n;
  int64_t sk_b, sk_h, sk_n;
  int64_t sv_b, sv_h, sv_n;
  int64_t skp_b, skp_h, skp_n;
  int64_t svp_b, svp_h, svp_n;
  int64_t so_b, so_h, so_n;
  int64_t sts_b, sts_h;
  int64_t scnt_b, scnt_h;
  int B, Hq, Hkv, G, Nq, Nk;
  SeqMap seq;  // ragged batch (varlen): every sequence has Nq = Nk = seq.len(b)
  int D;  // head dimension: a multiple of 8, at most 128 (dims D..127 are zero-filled)
  int P_host;
  const int32_t* P_dev;  // P on the device ([B], one per sequence, for a ragged batch)
  int window;
  float scale_log2;  // softmax scale * log2(e)
  int no_count;
  int cnt_is_float;
  int causal;
  const int32_t* sched;  // [B*Hkv][2][nblk_cap]: block maxima, prefix maxima
  int nblk_cap;
  // prepared by the schedule kernel, [B*Hkv][wcap] each:
  const float* wts;    // key bias log2(w_i) / scale_log2 of packed row i (-inf where w_i = 0)
  const int32_t* tsw;  // timestamp of packed row i, INT_MAX where the weight is 0
  const float* zeros;  // 64 zero biases (the exact tiles)
  int wcap;            // nblk_cap * 128
  int hpw;          // query heads per workgroup (4, 2 or 1)
  int n_row_groups;
  int units;        // B * Hkv * (G / hpw)
  int slots;        // workgroups an XCD runs at once, two a CU
  int* queue;       // 8 work-queue counters (persistent attn_w64_kernel grid) or null
};

__device__ __forceinline__ float exp2_fast(float x) { return __builtin_amdgcn_exp2f(x); }

// Phase-1 extent of a query block (deltaFlashAttention.py:58-80): n_safe = the number of
// packed blocks whose prefix maximum timestamp is below thr -- the prefix maxima do not
// decrease, so these are exactly the blocks before the first unsafe one -- and last = the
// maximum timestamp of the last of them (-1 if none).  A ballot per 64 blocks counts
// them; the entries of 256 blocks are loaded together, so the usual case is one round
// trip to memory.  Needs all 64 lanes of the wave.
__device__ __forceinline__ void safe_prefix(const int32_t* __restrict__ bmax, const int32_t* __restrict__ pmax,
                                            int nblk, int thr, int& n_safe, int& last, int lane) {
  int n = 0, prev_last = -1;
  last = -1;
  for (int base = 0; base < nblk; base += 256) {
    int pv[4], bv[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int i = base + 64 * j + lane;
      pv[j] = i < nblk ? pmax[i] : INT_MAX;
      bv[j] = i < nblk ? bmax[i] : -1;
    }
    int cnt = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) cnt += __popcll(__ballot(pv[j] < thr));
    n += cnt;
    if (cnt > 0) {
      const int k = cnt - 1;  // the last safe block is entry k of this chunk
      const int j = k >> 6;
      const int v = j == 0 ? bv[0] : j == 1 ? bv[1] : j == 2 ? bv[2] : bv[3];
      last = __builtin_amdgcn_readlane(v, k & 63);
    } else {
      last = prev_last;
    }
    if (cnt < 256) break;
    prev_last = last;
  }
  n_safe = n;
}

// min(max(x, 0), hi) for a wave-uniform x, kept in scalar registers (the compiler would
// otherwise form a clamp that only exists as a vector instruction, v_med3).
__device__ __forceinline__ int clamp0_uniform(int x, int hi) {
  x = __builtin_amdgcn_readfirstlane(x < hi ? x : hi);
  asm volatile("" : "+s"(x));
  return x > 0 ? x : 0;
}

// Third dword of a raw buffer resource on gfx9 (32-bit data format, no swizzle).
constexpr int kBufferDword3 = 0x00020000;

// A wave-uniform pointer moved into scalar registers.
__device__ __forceinline__ const void* uniform_ptr(const void* p) {
  const uint64_t v = (uint64_t)p;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return (const void*)(((uint64_t)hi << 32) | lo);
}

// Workgroup barrier after the wave's own LDS reads and writes.  Its loads to LDS
// (buffer_load ... lds) have their own wait, vmcnt(0), just before.  The asm is a compiler
// memory barrier.
__device__ __forceinline__ void window_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

typedef short i16x4 __attribute__((ext_vector_type(4)));

// LDS byte address of a pointer into the kernel's LDS.
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char*)p;
}
// ds_read_b64_tr_b16 at addr + OFF: in each group of 16 lanes, lane i receives element
// i % 4 of the 8 bytes read by lanes 4e + i / 4, e = 0..3 (a 4 x 4 transpose of 16-bit
// elements per group of four lanes).  Issued as asm: the caller waits with lgkm_wait.
template <int OFF>
__device__ __forceinline__ i16x4 ds_read_tr16(uint32_t addr) {
  i16x4 v;
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "i"(OFF));
  return v;
}
// s_waitcnt lgkmcnt(N) that the uses of a and b cannot move above.
template <int N>
__device__ __forceinline__ void lgkm_wait(i16x4& a, i16x4& b) {
  asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(a), "+v"(b) : "i"(N));
}
// ds_read_b128 issued as asm (waited for with lgkm_wait), so that the reads stay ahead
// of the MFMAs that use them.
__device__ __forceinline__ u32x4 ds_read_b128_asm(uint32_t addr) {
  u32x4 v;
  asm volatile("ds_read_b128 %0, %1" : "=v"(v) : "v"(addr));
  return v;
}
template <int N>
__device__ __forceinline__ void lgkm_wait(u32x4& a, u32x4& b) {
  asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(a), "+v"(b) : "i"(N));
}
template <int N>
__device__ __forceinline__ void lgkm_wait(u32x4& a) {
  asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(a) : "i"(N));
}
template <typename F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
// f(integral_constant<int, i>) for i = 0 .. N-1, in order
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// Max / sum of x over lanes l and l ^ 32, without LDS (v_permlane32_swap); the order
// of the returned pair does not matter for either.
__device__ __forceinline__ float halves_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __builtin_fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float halves_sum(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// s_waitcnt immediate (gfx9 encoding) that waits for vmcnt <= n only.
constexpr int vmcnt_only(int n) { return (n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8); }

// The 16-bit kernel updates its running maximum lazily: only when a tile's maximum
// exceeds it by more than 2^8 in probability (8 in log2 units) are O and l rescaled.
constexpr float kLazyLog2 = 8.0f;
// The 16-bit kernel computes p against the current maximum before it looks at the
// tile's maximum, and needs the latter only where a lane's sum of its 16 p exceeds
// 16 * 2^8: below that bound every p is at most 2^8 * 16, and a rescale is not needed
// (p stays far from fp32's range and keeps bf16's relative precision).
constexpr float kLazySum = 16.0f * 256.0f;
// That (LAZY) is for GQA groups that are a multiple of 4.  The others take every tile's maximum:
// the largest p of a row is then 1, which 16 bits hold exactly, and their error against 64
// bits stays what it was (fp16, 8 heads x 1067 tokens: 2.58e-4; 4 % more with the lazy rule).

// ====================================================================================
// The 16-bit attention kernel, for every GQA group.
//
// A workgroup is 4 waves, one per SIMD: 4, 2 or 1 query heads of a GQA group (hpw) over 64,
// 128 or 256 rows, each wave 64 rows of one head as two 32-row column blocks (NCB), so that
// every K fragment and every V^T fragment read from LDS feeds two MFMAs.  Small grids take
// half the rows, one column block a wave (launch_attn_rows; the rows' sums are the same bit for
// bit), with the fragments read further ahead, since each feeds one MFMA.  Two workgroups share a CU:
// while a wave runs its softmax (VALU), the other workgroup's wave on its SIMD has the matrix
// pipe (its MFMAs go out at raised priority).  Tiles are 32 keys; every tile boundary falls
// on the reference's logical 128-key grid.
//
// A window is the matrix work of a wave's tile (P.V of the previous one, then Q.K), a
// barrier, the loads of later tiles, the softmax.  K and V tiles go straight from memory to
// LDS (buffer_load ... lds), two stages each, a window ahead of their use; V is kept row-major
// and read as V^T with ds_read_b64_tr_b16.  No tile passes through registers.  Q of column
// block 0 stays in registers; Q of column block 1 sits in LDS, lane-private (each lane reads
// back only what it wrote), which keeps the wave within 256 registers and the workgroup's LDS
// (66 KiB) within half a CU's.
//
// Against one 8-wave workgroup a CU (two such groups in lockstep, half a window apart), which
// this replaces: items are half as long, so small grids end sooner (dense 1024 tokens x 32
// heads 44 against 53 us, 2048 80 / 93, 4096 162 / 180), and an item's first loads, epilogue
// and queue take run under the other workgroup's tiles (hybrid, one key in four: 32768 tokens
// 1.97 against 2.04 ms, 131072 27.9 / 28.7; ragged batches 4.5 / 4.7 ms).  It reads each tile
// twice as often from L2, which costs up to 0.3 % where neither matters (dense 32768).  Groups
// that are not a multiple of 4 ran a 32-row kernel that staged tiles through registers: 8000
// tokens x 32 heads, keys repeated to the query heads, 264 against 319 us (286 with the queues,
// 236 with them and the lazy maximum below).
// ====================================================================================
constexpr int kWTK = 32;                         // keys per tile
constexpr int kWKBytes = kWTK * kD * 2;          // 8 KiB
constexpr int kWVBytes = kWTK * kD * 2;          // 8 KiB
constexpr int kWMetaSlot = 64 * 8;               // weights[64] fp32, timestamps[64] int32
constexpr int kWCnt = 0, kWTs = 64 * 4;          // offsets inside a meta slot
constexpr int kWQBytes = 32 * kD * 2;          // Q of one 32-row column block, per wave
// LDS: two stages each of K and V, the weights' ring, the four waves' Q regions, then the
// persistent grid's item broadcast (queue, index, queues found empty)
constexpr int kWItemSlot = 2 * (kWKBytes + kWVBytes) + 4 * kWMetaSlot + 4 * kWQBytes;
constexpr int kWLds = kWItemSlot + 16;
// K stages and Q blocks start at multiples of 256 bytes (the kernel has no static LDS, so
// its dynamic LDS starts at address 0): the K / Q fragment addresses are formed by XOR.
static_assert(kWKBytes % 256 == 0 && kWVBytes % 256 == 0 && (4 * kWMetaSlot) % 256 == 0 && kWQBytes % 256 == 0,
              "K stages and Q blocks must be 256-byte aligned");

// Masks of one 32-key x 32-row score block (S^T register r holds key 8 (r / 4) + 4 hl +
// r % 4 of the tile for the lane's row).
__device__ __forceinline__ void mask_dense32(f32x16& s, int key0, int row, int hl, int Nk, bool causal) {
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int key = key0 + 8 * (r >> 2) + 4 * hl + (r & 3);
    const bool ok = key < Nk && (!causal || key <= row);
    if (!ok) s[r] = -INFINITY;
  }
}
__device__ __forceinline__ void mask_pure32(f32x16& s, const int* tl, int row, int hl) {
#pragma unroll
  for (int r4 = 0; r4 < 4; ++r4) {
    const int4 t4 = *(const int4*)(tl + 8 * r4 + 4 * hl);
    if (!(t4.x <= row)) s[4 * r4 + 0] = -INFINITY;
    if (!(t4.y <= row)) s[4 * r4 + 1] = -INFINITY;
    if (!(t4.z <= row)) s[4 * r4 + 2] = -INFINITY;
    if (!(t4.w <= row)) s[4 * r4 + 3] = -INFINITY;
  }
}

// Units of work queue q (one queue per XCD): the contiguous range [ulo, uhi) of the
// units, in the order of the static grid below.
__device__ __forceinline__ void queue_units(int q, int units, int& ulo, int& uhi) {
  ulo = (q * units) >> 3;
  uhi = ((q + 1) * units) >> 3;
}

// Item k of an XCD's n = units * n_rg (unit, row group) pairs: unit by unit, the longest row
// groups first.  Where all of them start at once, two a CU, the first half of the slots takes
// the longest, one a CU, and the rest run from the shortest up, so that every CU gets about
// the same work.
__device__ __forceinline__ void item_at(int k, int units, int n_rg, int slots, int& unit, int& rg) {
  const int n = units * n_rg, half = slots >> 1;
  if (n <= slots) {
    const int e = k < half ? k : n - 1 - (k - half);
    unit = e % units;
    rg = n_rg - 1 - e / units;
  } else {
    unit = k / n_rg;
    rg = n_rg - 1 - (k - unit * n_rg);
  }
}

// One (unit, row group) of attn_w64_kernel: a.hpw (4, 2 or 1) query heads of one (batch, KV
// head) over 128 NCB / hpw rows.  Ends with every LDS read of the window loop done (its last
// barrier) and every load landed; the finalize uses only the wave's own Q region, so the next
// item may start staging at once.
template <int VARIANT, int DT, int NCB, bool LAZY>
__device__ __forceinline__ void attn_w64_item(const AttnArgs& a, const int unit, const int rg) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  char* const kst0 = smem;
  char* const vst0 = smem + 2 * kWKBytes;
  char* const meta0 = smem + 2 * (kWKBytes + kWVBytes);
  // opaque per item: what derives from the thread index is formed here, not hoisted out
  // of the persistent grid's item loop into registers held across items
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));
  const int lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform per wave
  // Q of column block 1, lane-private: each lane reads back only the 16-byte chunks it
  // wrote (the K fragment layout), so the 32 registers it would take stay free
  char* const qs = meta0 + 4 * kWMetaSlot + wid * kWQBytes;
  const int hl = lane >> 5, ql = lane & 31;
  const int hsh = a.hpw >> 1;  // log2 of the query heads a workgroup takes
  const int hunits = a.G >> hsh;
  const int gb = unit / hunits;  // g * B + b
  const int hu = unit - gb * hunits;
  const int g = gb / a.B, b = gb - (gb / a.B) * a.B;
  const int bg = b * a.Hkv + g;
  const int h = g * a.G + (hu << hsh) + (wid & ((1 << hsh) - 1));
  const int wg_rows = (128 * NCB) >> hsh;
  const int R0 = rg * wg_rows;
  const int Nq = a.seq.cu ? a.seq.len(b) : a.Nq;
  const int Nk = a.seq.cu ? a.seq.len(b) : a.Nk;
  if (R0 >= Nq) return;  // a row group past the end of a shorter sequence (whole workgroup)
  // first row of this wave; column block cb holds r0w + 32 cb + ql
  const int r0w = R0 + 32 * NCB * (wid >> hsh);
  const int wg_end = R0 + wg_rows;

  // ---- schedule: packed tiles 0 .. n1 - 1, then exact tiles from key ds on.  A workgroup's
  // rows lie in one logical 128-row block, except where one head takes 256 rows (hpw
  // 1, NCB 2): its tiles are then the union of the two blocks' schedules, and a wave skips those
  // that its own block (n1w, dsw) does not have ----
  int P = a.P_host;
  if (a.P_dev) P = min(a.seq.cu ? a.P_dev[b] : *a.P_dev, a.P_host);
  if (a.seq.cu) P = min(P, Nk);
  int n1 = 0, ds = 0, n1w = 0, dsw = 0;
  int kend = a.causal ? min(Nk, wg_end) : Nk;
  if (VARIANT == kHybrid || VARIANT == kSanity) {
    const int nblk = (P + kBlock - 1) / kBlock;
    const int32_t* bmax = a.sched + (int64_t)bg * 2 * a.nblk_cap;
    const int32_t* pmax = bmax + a.nblk_cap;
    auto block_schedule = [&](const int start_m, int& n, int& d) {
      int n_safe, last;
      safe_prefix(bmax, pmax, nblk, start_m - a.window, n_safe, last, lane);
      d = max(0, ((last + 1) / kBlock) * kBlock);
      n = VARIANT == kHybrid ? n_safe * (kBlock / kWTK) : 0;
    };
    // a wave past the last row follows the last block that has rows: every wave of the
    // workgroup must come to the same tiles
    const int start_w = min(r0w, Nq - 1) & ~(kBlock - 1);
    block_schedule(start_w, n1w, dsw);
    n1 = n1w;
    ds = dsw;
    if (NCB == 2 && hsh == 0 && R0 + kBlock < Nq) {
      int n2w, d2w;
      block_schedule(start_w ^ kBlock, n2w, d2w);
      n1 = max(n1, n2w);
      ds = min(ds, d2w);
    }
    kend = min(Nk, wg_end);
  } else if (VARIANT == kPure) {
    // the packed blocks up to the last that holds a key at or before the last row
    const int nblk = (P + kBlock - 1) / kBlock;
    const int32_t* from = a.sched + (int64_t)bg * 2 * a.nblk_cap + a.nblk_cap;
    int last;
    safe_prefix(from, from, nblk, r0w + 32 * NCB, n1w, last, lane);
    safe_prefix(from, from, nblk, wg_end, n1, last, lane);
    n1w = min(n1w * (kBlock / kWTK), (P + kWTK - 1) / kWTK);
    n1 = min(n1 * (kBlock / kWTK), (P + kWTK - 1) / kWTK);
    kend = 0;
  }
  n1 = __builtin_amdgcn_readfirstlane(n1);
  ds = __builtin_amdgcn_readfirstlane(ds);
  const int n2 = kend > ds ? (kend - ds + kWTK - 1) / kWTK : 0;
  const int T = n1 + n2;

  const uint16_t* kp_base = a.kp + a.seq.base(b, a.skp_b, a.skp_n) + (int64_t)g * a.skp_h;
  const uint16_t* vp_base = a.vp + a.seq.base(b, a.svp_b, a.svp_n) + (int64_t)g * a.svp_h;
  const uint16_t* k_base = a.k + a.seq.base(b, a.sk_b, a.sk_n) + (int64_t)g * a.sk_h;
  const uint16_t* v_base = a.v + a.seq.base(b, a.sv_b, a.sv_n) + (int64_t)g * a.sv_h;
  const float* w_row = a.wts ? a.wts + (int64_t)bg * a.wcap : nullptr;
  const int32_t* tsw_row = a.tsw ? a.tsw + (int64_t)bg * a.wcap : nullptr;
  constexpr bool kPureV = VARIANT == kPure;
  constexpr bool kWeights = VARIANT == kHybrid || VARIANT == kPure;

  auto key0_of = [&](int t) { return t < n1 ? t * kWTK : ds + (t - n1) * kWTK; };
  // causal: a Phase-2 tile whose first key is past the wave's last row is skipped
  int t_skip = INT_MAX;
  if (a.causal) {
    const int d = r0w + 32 * NCB - 1 - ds;
    t_skip = __builtin_amdgcn_readfirstlane(d < 0 ? n1 : n1 + d / kWTK + 1);
  }
  if (kPureV) t_skip = __builtin_amdgcn_readfirstlane(n1w);
  if (r0w >= Nq) t_skip = 0;  // no rows
  // and those of the other logical block: [skip_lo, skip_hi)
  const int skip_lo = __builtin_amdgcn_readfirstlane(n1w);
  const int skip_hi = __builtin_amdgcn_readfirstlane(n1 + (dsw - ds) / kWTK);

  // ---- staging: loads straight into LDS, two stages each for K and V and a ring of
  // four slots for the tiles' weights.  Wave w loads rows 8w .. 8w + 7 of both tiles in two
  // steps of four: lane l writes 16 bytes at 1 KiB (2 w + j) + 16 l, i.e. row 8 w + 4 j + l / 16
  // at position l % 16, so it fetches the source chunk that the swizzled layout keeps there.  The buffer
  // resource covers exactly the tile's valid keys: rows past the end, and 8-dim chunks
  // at or beyond the head dimension, arrive as zeros.  A window's loads go out after its
  // barrier, and all are waited for (vmcnt(0)) before the next one. ----
  const int wid_s = __builtin_amdgcn_readfirstlane(wid);
  const char* kb1 = (const char*)uniform_ptr(kp_base);
  const char* kb2 = (const char*)uniform_ptr(k_base);
  const char* vb1 = (const char*)uniform_ptr(vp_base);
  const char* vb2 = (const char*)uniform_ptr(v_base);
  const int skpb = __builtin_amdgcn_readfirstlane((int)(2 * a.skp_n));
  const int skb = __builtin_amdgcn_readfirstlane((int)(2 * a.sk_n));
  const int svpb = __builtin_amdgcn_readfirstlane((int)(2 * a.svp_n));
  const int svb = __builtin_amdgcn_readfirstlane((int)(2 * a.sv_n));
  auto dma_rows = [&](bool isK, int t_raw, unsigned st) {
    const int t = min(t_raw, T - 1);
    const bool ph1 = t < n1;
    const int key0 = key0_of(t);
    const int limit = ph1 ? P : Nk;
    const int snb = isK ? (ph1 ? skpb : skb) : (ph1 ? svpb : svb);
    const char* src = isK ? (ph1 ? kb1 : kb2) : (ph1 ? vb1 : vb2);
    const void* base = uniform_ptr(src + (int64_t)key0 * snb);
    const int range = clamp0_uniform(limit - key0, kWTK) * snb;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<void*>(base), (short)0, range, kBufferDword3);
    char* dst = isK ? kst0 + st : vst0 + st;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int w4 = 2 * wid_s + j;
      const int rowt = w4 * 4 + (lane >> 4);
      const int pos = lane & 15;
      const int chunk = pos ^ (isK ? (rowt & 15) : 4 * (rowt & 3));
      // rowt < 32 and snb < 2^24 (the host limits sequence strides to 2^23 elements), so the
      // unsigned 24-bit multiply is exact (a signed one would read snb >= 2^23 as negative);
      // a chunk at or past the head dimension reads past the range (zeros), without a branch
      const int off = (int)__umul24((unsigned)rowt, (unsigned)snb) + chunk * 16 + (chunk * 8 < a.D ? 0 : range);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)(dst + w4 * 1024), 16,
                                               off, 0, 0, 0);
    }
  };
  // key biases (and timestamps) of the tile's 32 keys, into slot t % 4 of their ring
  // (lanes 32-63 read past the range: zeros); a packed tile reads the prepared biases,
  // an exact tile zeros; S^T starts at them
  auto meta_of = [&](int t) { return meta0 + (t & 3) * kWMetaSlot; };
  auto dma_meta = [&](int t_raw) {
    if (!kWeights) return;
    const int t = min(t_raw, T - 1);
    const bool ph1 = t < n1;
    const int key0 = ph1 ? t * kWTK : 0;
    const int nrows = ph1 ? clamp0_uniform(a.wcap - key0, kWTK) : kWTK;
    char* dst = meta_of(t_raw);
    // the lane's offset, formed here from an opaque lane index rather than held
    int mlane = lane;
    asm volatile("" : "+v"(mlane));
    const __amdgpu_buffer_rsrc_t rc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<void*>(uniform_ptr(ph1 ? w_row + key0 : a.zeros)), (short)0,
        nrows * 4, kBufferDword3);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rc, (__attribute__((address_space(3))) void*)(dst + kWCnt), 4,
                                             mlane * 4, 0, 0, 0);
    if (kPureV) {
      const __amdgpu_buffer_rsrc_t rt = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<void*>(uniform_ptr(tsw_row + key0)), (short)0, nrows * 4, kBufferDword3);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rt, (__attribute__((address_space(3))) void*)(dst + kWTs), 4,
                                               mlane * 4, 0, 0, 0);
    }
  };
  auto dma_issue = [&](int tk, int tv, unsigned kst, unsigned vst) {
    dma_rows(true, tk, kst);
    dma_rows(false, tv, vst);
    if (wid_s == 0) dma_meta(tk);
  };

  // ---- per-lane LDS offsets (stage-relative).  K: rows of 256 bytes, 16-byte chunk c
  // of row r at position c ^ (r & 15); the lane reads chunk 2 j + hl of row ql.  V^T:
  // fragments of 16 keys x 32 head dims (db) read with ds_read_b64_tr_b16 from rows
  // whose chunks sit at c ^ 4 (r & 3).  Both are recomputed in each matrix section
  // (made opaque there) rather than held in registers ----
  int k_lane = ql * 256 + (((hl ^ ql) & 1) << 4) + ((ql & 14) << 4);
  int v_lane = (4 * ((lane >> 4) >> 1) + ((lane & 15) >> 2)) * 256 +
               ((2 * ((lane >> 4) & 1) + ((lane & 3) >> 1)) << 4) + 8 * (lane & 1) + 64 * ((lane & 15) >> 2);

  f32x16 o[NCB][4];
#pragma unroll
  for (int cb = 0; cb < NCB; ++cb)
#pragma unroll
    for (int i = 0; i < 4; ++i) o[cb][i] = f32x16{};
  f32x16 s[NCB];
  u32x4 pw[NCB][2];
  // mc: the running maximum times c, the reference point of p = 2^(s c - mc).  Until a
  // lane has seen a finite score it is -FLT_MAX: every finite score then gives p = +inf
  // (the exact rule takes over), a masked one p = 0, and s c - mc is never NaN
  float mc[NCB], l_i[NCB];
#pragma unroll
  for (int cb = 0; cb < NCB; ++cb) mc[cb] = -__FLT_MAX__, l_i[cb] = 0.0f;
  const float c = a.scale_log2;

  unsigned stA = 0, stB = kWKBytes;
  if (T > 0) {
    dma_rows(true, 0, stA);
    if (wid_s == 0) dma_meta(0);
    dma_issue(1, 0, stB, stA);  // V of tile w - 1 is read in stage stB of window w
  }
  // ---- Q^T of both column blocks in registers, loaded while the first tiles are in
  // flight; rows past Nq load row Nq - 1 and dims past D dims 0..7, zeroed after ----
  u32x4 qreg[kD / 16];
  {
    // both column blocks requested before either is used: one round trip, not two
    u32x4 w[NCB][kD / 16];
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb) {
      const int row = r0w + 32 * cb + ql;
      const uint16_t* qrow = a.q + a.seq.base(b, a.sq_b, a.sq_n) + (int64_t)h * a.sq_h + (int64_t)min(row, Nq - 1) * a.sq_n;
#pragma unroll
      for (int t = 0; t < kD / 16; ++t) {
        const int d0 = 16 * t + 8 * hl;
        w[cb][t] = *(const u32x4*)(qrow + (d0 < a.D ? d0 : 0));
      }
    }
    // redefined so that the loop does not see Q as an outstanding load (the S = K Q^T
    // blocks would otherwise wait for every memory load, the staging loads included)
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb) {
      const int row = r0w + 32 * cb + ql;
#pragma unroll
      for (int t = 0; t < kD / 16; ++t) {
        asm volatile("" : "+v"(w[cb][t]));
        const u32x4 qv = (row < Nq && 16 * t + 8 * hl < a.D) ? w[cb][t] : u32x4{0, 0, 0, 0};
        if (cb == 0)
          qreg[t] = qv;
        else
          *(u32x4*)(qs + ql * 256 + (((2 * t + hl) ^ (ql & 15)) << 4)) = qv;
      }
    }
  }
  if (T > 0) {
    __builtin_amdgcn_s_waitcnt(vmcnt_only(0));
    lds_barrier();
  }

  constexpr int kWAhead = NCB == 2 ? 3 : 6;    // V^T fragments read ahead of their MFMAs
  constexpr int kWQKAhead = NCB == 2 ? 2 : 5;  // (K, Q) fragment pairs (one block: K) read ahead
  const int nwin = T > 0 ? T + 1 : 0;
  // ---- matrix work of a window: O^T += V^T P^T for tile t - 1 (PV), then S^T = K Q^T for
  // tile t (QK), each LDS fragment feeding both column blocks ----
  // One stream of LDS operand reads for the section: the V^T fragments of the P.V
  // block, then (hybrid, pure) the keys' biases, then the (K, Q) fragment pairs of
  // the S^T block, each read a few MFMA pairs ahead of its use, across the border
  // between the blocks.  The stream's order is fixed at compile time, so every wait
  // is an exact lgkmcnt.
  auto matrix_block = [&](const int t, auto PVC, auto QKC) __attribute__((always_inline)) {
    constexpr bool PV = decltype(PVC)::value, QK = decltype(QKC)::value;
    constexpr bool BIAS = QK && kWeights;
    constexpr int NPV = PV ? 8 : 0, NQK = QK ? kD / 16 : 0;
    constexpr int EBIAS = NPV;                   // stream index of the bias reads
    constexpr int EQK = NPV + (BIAS ? 1 : 0);    // stream index of (K, Q) pair 0
    constexpr int E = EQK + NQK;                 // stream length
    constexpr int NM = NPV + NQK;                // MFMA pairs
    // stream element of MFMA pair i; elements issued before pair i's wait
    constexpr auto el = [](int i) { return i < NPV ? i : EQK + (i - NPV); };
    constexpr auto size = [](int e) { return (BIAS && e == EBIAS) ? 4 : e >= EQK ? NCB : 2; };
    constexpr auto issued = [el](int i) {
      int n = 0;
      for (int k = 0; k <= i; ++k) {
        const int a = el(k) + 1 + (k < NPV ? kWAhead - 1 : kWQKAhead - 1);
        n = a > n ? a : n;
      }
      return n < E ? n : E;
    };
    constexpr auto pending = [el, size, issued](int i) {
      int c = 0;
      for (int e = el(i) + 1; e < issued(i); ++e) c += size(e);
      return c;
    };
    uint32_t va[4] = {0, 0, 0, 0};
    if constexpr (PV) {
      const uint32_t vb = lds_addr(vst0) + stB;
      // opaque: otherwise the offsets are hoisted out of the loop into registers
      asm volatile("" : "+v"(v_lane));
      const uint32_t vl = vb + v_lane;
#pragma unroll
      for (int db = 0; db < 4; ++db) va[db] = vl ^ (64u * db);
    }
    uint32_t kla = 0, qla = 0, bla = 0;
    if constexpr (QK) {
      asm volatile("" : "+v"(k_lane));
      kla = lds_addr(kst0) + stA + k_lane;
      if constexpr (NCB == 2) qla = lds_addr(qs) + k_lane;
      bla = lds_addr(meta_of(t) + kWCnt) + 16 * hl;
    }
    i16x4 vlo[8], vhi[8];
    u32x4 kw[kD / 16], qw[NCB == 2 ? kD / 16 : 1], bw[4];
    auto read = [&](auto EC) {
      constexpr int e = decltype(EC)::value;
      if constexpr (e < NPV) {
        vlo[e] = ds_read_tr16<(e >> 2) * 4096>(va[e & 3]);
        vhi[e] = ds_read_tr16<(e >> 2) * 4096 + 2048>(va[e & 3]);
      } else if constexpr (BIAS && e == EBIAS) {
#pragma unroll
        for (int r = 0; r < 4; ++r) bw[r] = ds_read_b128_asm(bla + 32 * r);
      } else {
        constexpr int j = e - EQK;
        kw[j] = ds_read_b128_asm(kla ^ (32u * j));
        if constexpr (NCB == 2) qw[j] = ds_read_b128_asm(qla ^ (32u * j));
      }
    };
    static_for<issued(0)>(read);
    static_for<NM>([&](auto I) {
      constexpr int i = decltype(I)::value;
      if constexpr (i < NPV) {
        lgkm_wait<pending(i)>(vlo[i], vhi[i]);
        const u32x4 vw = __builtin_bit_cast(u32x4, __builtin_shufflevector(vlo[i], vhi[i], 0, 1, 2, 3, 4, 5, 6, 7));
        o[0][i & 3] = E16<DT>::mfma(vw, pw[0][i >> 2], o[0][i & 3]);
        if constexpr (NCB == 2) o[1][i & 3] = E16<DT>::mfma(vw, pw[1][i >> 2], o[1][i & 3]);
      } else {
        constexpr int j = i - NPV;
        if constexpr (NCB == 2) lgkm_wait<pending(i)>(kw[j], qw[j]);
        else lgkm_wait<pending(i)>(kw[j]);
        if constexpr (j == 0) {
          // S^T starts at the keys' biases (read before pair 0, so complete now),
          // or at zero (the MFMA's inline constant)
          if constexpr (BIAS) {
            asm volatile("" : "+v"(bw[0]), "+v"(bw[1]), "+v"(bw[2]), "+v"(bw[3]));
            const f32x4 b0 = __builtin_bit_cast(f32x4, bw[0]), b1 = __builtin_bit_cast(f32x4, bw[1]);
            const f32x4 b2 = __builtin_bit_cast(f32x4, bw[2]), b3 = __builtin_bit_cast(f32x4, bw[3]);
            const f32x16 c0 = __builtin_shufflevector(__builtin_shufflevector(b0, b1, 0, 1, 2, 3, 4, 5, 6, 7),
                                                      __builtin_shufflevector(b2, b3, 0, 1, 2, 3, 4, 5, 6, 7),
                                                      0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15);
            s[0] = E16<DT>::mfma(kw[0], qreg[0], c0);
            if constexpr (NCB == 2) s[1] = E16<DT>::mfma(kw[0], qw[0], c0);
          } else {
            s[0] = E16<DT>::mfma(kw[0], qreg[0], f32x16{});
            if constexpr (NCB == 2) s[1] = E16<DT>::mfma(kw[0], qw[0], f32x16{});
          }
        } else {
          s[0] = E16<DT>::mfma(kw[j], qreg[j], s[0]);
          if constexpr (NCB == 2) s[1] = E16<DT>::mfma(kw[j], qw[j], s[1]);
        }
      }
      static_for<issued(i + 1 < NM ? i + 1 : i) - issued(i)>([&](auto K) {
        read(std::integral_constant<int, issued(i) + decltype(K)::value>{});
      });
    });
  };
  // ---- softmax of tile t: the two column blocks one after the other, one check each ----
  auto softmax_tile = [&](const int t) __attribute__((always_inline)) {
    const char* ms = meta_of(t);
    const int key0 = key0_of(t);
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb) {
      const int row = r0w + 32 * cb + ql;
      if (kPureV) {
        mask_pure32(s[cb], (const int*)(ms + kWTs), row, hl);
      } else if (t >= n1) {
        if ((a.causal && key0 + kWTK - 1 > r0w + 32 * cb) || key0 + kWTK > Nk)
          mask_dense32(s[cb], key0, row, hl, Nk, a.causal);
      }
    }
    // p against the current maximum first; only where a lane's sum of its 16 p
    // exceeds kLazySum (some p above 2^8, a score above the maximum by 8 / c; +inf
    // while the lane has no maximum yet) is the tile's maximum taken and the column
    // block redone with the lazy-rescale rule.  P in the 16-bit type for the P.V
    // MFMAs; the row sum adds the fp32 p, as deltaFlashAttention.py:86-98
    auto exps = [&](const int cb, const float neg) {
      float psa, psb;
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4) {
        float p[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) p[e] = exp2_fast(__builtin_fmaf(s[cb][4 * r4 + e], c, neg));
        pw[cb][r4 >> 1][(r4 & 1) * 2 + 0] = E16<DT>::pack(p[0], p[1]);
        pw[cb][r4 >> 1][(r4 & 1) * 2 + 1] = E16<DT>::pack(p[2], p[3]);
        psa = r4 == 0 ? p[0] + p[1] : psa + (p[0] + p[1]);
        psb = r4 == 0 ? p[2] + p[3] : psb + (p[2] + p[3]);
      }
      return psa + psb;
    };
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb) {
      float ps = LAZY ? exps(cb, -mc[cb]) : 0.0f;
      // the bound also catches an infinite sum
      if (!LAZY || __builtin_amdgcn_ballot_w64(ps > kLazySum)) {
        float m = -INFINITY;
#pragma unroll
        for (int r = 0; r < 16; r += 2) m = __builtin_fmaxf(m, __builtin_fmaxf(s[cb][r], s[cb][r + 1]));
        const float mxc = halves_max(m) * c;
        // alpha = 1 exactly where a lane keeps its maximum (also where it has none yet)
        const bool upd = mxc > mc[cb] + (LAZY ? kLazyLog2 : 0.0f);
        const float m_new = upd ? mxc : mc[cb];
        const float alpha = upd ? exp2_fast(mc[cb] - m_new) : 1.0f;
        if (LAZY || __builtin_amdgcn_ballot_w64(upd)) {
#pragma unroll
          for (int db = 0; db < 4; ++db)
#pragma unroll
            for (int r = 0; r < 16; ++r) o[cb][db][r] *= alpha;
        }
        l_i[cb] *= alpha;
        mc[cb] = m_new;
        ps = exps(cb, -m_new);
      }
      l_i[cb] += ps;
    }
  };
  using False = std::integral_constant<bool, false>;
  using True = std::integral_constant<bool, true>;
  // Window w: the matrix work, the barrier, the loads of the next windows, the softmax.
  // At the barrier every wave has read K of tile w and V of tile w - 1, and the loads of
  // window w - 1 (K of w + 1, V of w) are done: K of w + 2 and V of w + 1 take their stages.
  auto turn = [&](const int w) {
    __builtin_amdgcn_s_waitcnt(vmcnt_only(0));
    window_barrier();
    if (w < T) dma_issue(w + 2, w + 1, stA, stB);
  };
  auto swap_stages = [&]() {
    const unsigned t0 = stA;
    stA = stB;
    stB = t0;
  };
  int w = 0;
  auto idle_until = [&](const int end) {  // windows whose tiles are not the wave's
    for (; w < end; ++w) {
      turn(w);
      swap_stages();
    }
  };
  // The wave's tiles are one interval, or two around the other logical block's.  Each runs
  // a loop without conditions (with them, its registers do not fit).
  const bool gap = skip_lo < skip_hi;
#pragma nounroll
  for (int r = 0; r < 2; ++r) {
    const int lo = r ? skip_hi : 0;
    const int hi = min(min(T, t_skip), r ? (gap ? T : 0) : (gap ? skip_lo : T));
    if (lo >= hi) continue;
    idle_until(lo);
    __builtin_amdgcn_s_setprio(1);
    matrix_block(w, False{}, True{});
    __builtin_amdgcn_s_setprio(0);
    turn(w);
    softmax_tile(w);
    swap_stages();
    for (++w; w < hi; ++w) {
      __builtin_amdgcn_s_setprio(1);
      matrix_block(w, True{}, True{});
      __builtin_amdgcn_s_setprio(0);
      turn(w);
      softmax_tile(w);
      swap_stages();
    }
    matrix_block(w, True{}, False{});
    turn(w);
    swap_stages();
    ++w;
  }
  idle_until(nwin);
  __builtin_amdgcn_s_waitcnt(vmcnt_only(0));  // no load may land in LDS after the exit

  // ---- finalize: each column block goes through the wave's own Q region of LDS (its
  // last Q.K is done), 16-byte chunk c of row r at position c ^ (r & 15), and leaves as
  // whole rows, four per store instruction, instead of 16 bytes of 32 rows ----
  uint16_t* const obase = a.out + a.seq.base(b, a.so_b, a.so_n) + (int64_t)h * a.so_h;
#pragma unroll
  for (int cb = 0; cb < NCB; ++cb) {
    const float l_tot = halves_sum(l_i[cb]);
    float inv;
    if (VARIANT == kPure)
      inv = l_tot > 0.0f ? 1.0f / l_tot : 1.0f;  // deltaFlashAttention.py:353-354
    else
      inv = 1.0f / l_tot;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        u32x2 w;
        w[0] = E16<DT>::pack(o[cb][db][4 * j + 0] * inv, o[cb][db][4 * j + 1] * inv);
        w[1] = E16<DT>::pack(o[cb][db][4 * j + 2] * inv, o[cb][db][4 * j + 3] * inv);
        // dims db * 32 + 8 j + 4 hl .. + 3 of row ql: half hl of chunk 4 db + j
        *(u32x2*)(qs + ql * 256 + (((4 * db + j) ^ (ql & 15)) << 4) + 8 * hl) = w;
      }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
    const int cq = lane & 15;
    u32x4 rw[8];
#pragma unroll
    for (int it = 0; it < 8; ++it) {
      const int r = 4 * it + (lane >> 4);
      rw[it] = *(const u32x4*)(qs + r * 256 + ((cq ^ (r & 15)) << 4));
    }
#pragma unroll
    for (int it = 0; it < 8; ++it) {
      const int row = r0w + 32 * cb + 4 * it + (lane >> 4);
      if (row < Nq && cq * 8 < a.D) *(u32x4*)(obase + (int64_t)row * a.so_n + cq * 8) = rw[it];
    }
    // the reads of this block are done before the next block overwrites the region
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
  }
}

// Work distribution.  Static (a.queue null, the dense control and small grids): workgroup i runs on XCD
// i mod 8 and takes one item; when the units split evenly over the 8 XCDs, each XCD gets
// a contiguous range of units and walks their row groups longest first, so a unit's K/V
// stay in one XCD's L2.  Persistent (a.queue set, large grids of the hybrid, sanity and
// pure Phase 1 variants, whose schedule kernel zeroes the 8 counters just before): two workgroups per
// CU loop over items.  Queue q holds the units of XCD q's static share in the same
// order (unit by unit, longest row group first) and a.queue[q] counts the items taken;
// a workgroup takes from the queue of the XCD it runs on and, once that is empty, from
// the others, so the XCDs, whose clocks differ by several per cent, finish together,
// and no dispatch gap lies between two items on a CU.  Every counter only grows, so each
// workgroup's loop ends after at most 8 empty takes; workgroups never wait on each other.
template <int VARIANT, int DT, int NCB, bool LAZY>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
void attn_w64_kernel(AttnArgs a) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  int* const slot = (int*)(smem + kWItemSlot);
  const int tid = threadIdx.x;
  const int n_rg = a.n_row_groups;
  const bool persistent = a.queue != nullptr;
  unsigned xcc = 0;
  if (persistent) {
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(xcc));
    if (tid == 0) slot[2] = 0;  // queues found empty so far, from this XCD's own
  }
  for (int first = 1;; first = 0) {
    int unit, rg;
    if (!persistent) {
      if (!first) break;
      const int wg = blockIdx.x;
      if ((a.units & 7) == 0) {
        const int xcd = wg & 7, upx = a.units >> 3;
        item_at(wg >> 3, upx, n_rg, a.slots, unit, rg);
        unit += xcd * upx;
      } else if (a.units * n_rg <= 8 * a.slots) {
        item_at(wg, a.units, n_rg, 8 * a.slots, unit, rg);
      } else {
        unit = wg % a.units;
        rg = n_rg - 1 - wg / a.units;
      }
    } else {
      if (tid == 0) {
        int q = 0, k = -1, qi = slot[2];
        while (qi < 8) {
          q = (int)((xcc + qi) & 7);
          int ulo, uhi;
          queue_units(q, a.units, ulo, uhi);
          const int taken = atomicAdd(a.queue + q, 1);
          if (taken < (uhi - ulo) * n_rg) {
            k = taken;
            break;
          }
          ++qi;
        }
        slot[0] = q;
        slot[1] = k;
        slot[2] = qi;
      }
      lds_barrier();
      const int q = __builtin_amdgcn_readfirstlane(slot[0]);
      const int k = __builtin_amdgcn_readfirstlane(slot[1]);
      lds_barrier();  // the slot is read before thread 0 writes it again
      if (k < 0) break;
      int ulo, uhi;
      queue_units(q, a.units, ulo, uhi);
      item_at(k, uhi - ulo, n_rg, a.slots, unit, rg);
      unit += ulo;
    }
#if defined(__HIP_DEVICE_COMPILE__)
    // the argument block read through the kernel-argument segment's address, made
    // opaque per item: its fields are loaded inside each item instead of being held in
    // scalar registers across the loop (the block is the kernel's only argument, at
    // offset 0)
    const __attribute__((address_space(4))) AttnArgs* ap =
        (const __attribute__((address_space(4))) AttnArgs*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(ap));
    const AttnArgs ai = *ap;
    attn_w64_item<VARIANT, DT, NCB, LAZY>(ai, unit, rg);
#else
    attn_w64_item<VARIANT, DT, NCB, LAZY>(a, unit, rg);
#endif
  }
}

// Per (batch, kv head): maxima of packed blocks of 128 timestamps (lanes at or
// beyond P read seq_len_k + 1, deltaFlashAttention.py:70) and their prefix maxima; for pure
// Phase 1 the suffix minima instead, which end a row group's keys at the last block that
// holds one it sees (16384 tokens, one key in four: 587 against 1018 us).
// Blocks with blockIdx.y = 0 do that; those with blockIdx.y = 1 + c (when wts is set)
// write, for packed rows [1024 c, 1024 c + 1024), the key bias log2(w) / scale_log2 of
// the row's weight w (the count, 1 with no_count, 0 at and beyond P:
// modeling_llama.py:321-324 and the masked loads of deltaFlashAttention.py:84-90; -inf
// for w = 0), so that exp2(scale_log2 (q.k + bias) - m) = w exp2(scale_log2 q.k - m);
// with tsw set the timestamps with INT_MAX where the weight is 0; block (0, 1) writes
// 64 zero biases.
struct SchedPrep {
  const void* cnt;
  int64_t scnt_b, scnt_h;
  int cnt_is_float, no_count;
  float scale_log2;
  float* wts;
  int32_t* tsw;
  float* zeros;
  int wcap;
};
constexpr int kSchedThreads = 1024;
constexpr int kSchedWaves = kSchedThreads / 64;
__global__ __launch_bounds__(kSchedThreads) void hybrid_schedule_kernel(const int32_t* __restrict__ ts,
                                                              int64_t sts_b, int64_t sts_h,
                                                              int Hkv, int P_host,
                                                              const int32_t* P_dev, int Nk,
                                                              SeqMap seq, int nblk_cap,
                                                              int32_t* __restrict__ sched,
                                                              SchedPrep prep, int* __restrict__ queue) {
  __shared__ int32_t s_bmax[4096];
  __shared__ int32_t s_wave[kSchedWaves];
  const int tid = threadIdx.x, lane = tid & 63;
  // the attention kernel's work-queue counters start at zero
  if (queue && blockIdx.x == 0 && blockIdx.y == 0 && tid < 8) queue[tid] = 0;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform (scalar)
  const int bg = blockIdx.x;
  const int b = bg / Hkv, g = bg - (bg / Hkv) * Hkv;
  int P = P_host;
  if (P_dev) P = min(seq.cu ? P_dev[b] : *P_dev, P_host);
  if (seq.cu) {
    Nk = seq.len(b);
    P = min(P, Nk);  // a sequence's packed rows lie inside its own tokens
  }
  const int nblk = (P + kBlock - 1) / kBlock;
  const int32_t* row = ts + seq.base(b, sts_b, 1) + (int64_t)g * sts_h;
  if (blockIdx.y > 0) {
    const int32_t* crow = (const int32_t*)prep.cnt + seq.base(b, prep.scnt_b, 1) + (int64_t)g * prep.scnt_h;
    float* wrow = prep.wts + (int64_t)bg * prep.wcap;
    int32_t* trow = prep.tsw ? prep.tsw + (int64_t)bg * prep.wcap : nullptr;
    if (bg == 0 && blockIdx.y == 1 && tid < 64) prep.zeros[tid] = 0.0f;
    // the attention kernels read rows below nblk * 128 only
    const int i = (blockIdx.y - 1) * kSchedThreads + tid;
    if ((blockIdx.y - 1) * kSchedThreads >= nblk * kBlock || i >= prep.wcap) return;
    float w = 0.0f;
    int tv = INT_MAX;
    if (i < P) {
      const int32_t raw = crow[i];
      w = prep.no_count ? 1.0f : (prep.cnt_is_float ? __int_as_float(raw) : (float)raw);
      if (trow && w > 0.0f) tv = row[i];
    }
    wrow[i] = w > 0.0f ? log2f(w) / prep.scale_log2 : -INFINITY;
    if (trow) trow[i] = tv;
    return;
  }
  // Pure Phase 1 takes all packed keys, masked by timestamp <= row: its rows need the blocks
  // up to the last one that holds such a key, so the scan is of the blocks' minima (keys of
  // weight 0 left out), from the last block back, as maxima of the negated values.
  const bool pure = prep.tsw != nullptr;
  const int32_t* crow = pure ? (const int32_t*)prep.cnt + seq.base(b, prep.scnt_b, 1) + (int64_t)g * prep.scnt_h : row;
  auto weighs = [&](int32_t raw) { return prep.no_count || (prep.cnt_is_float ? __int_as_float(raw) > 0.0f : raw > 0); };
  // wave w takes blocks 8w .. 8w + 7 of every 8 kSchedWaves, their loads in flight together:
  // rows at or beyond P are clamped to row P - 1 and masked after the load (a guarded
  // load is waited for before the next one is issued); nblk > 0 implies P > 0
  for (int jb0 = wid * 8; jb0 < nblk; jb0 += 8 * kSchedWaves) {
    int m[8];
    int r0[8], r1[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int i0 = (jb0 + u) * kBlock + lane, i1 = i0 + 64;
      r0[u] = row[min(i0, P - 1)];
      r1[u] = row[min(i1, P - 1)];
    }
    if (pure) {
      int c0[8], c1[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int i0 = (jb0 + u) * kBlock + lane, i1 = i0 + 64;
        c0[u] = crow[min(i0, P - 1)];
        c1[u] = crow[min(i1, P - 1)];
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int i0 = (jb0 + u) * kBlock + lane, i1 = i0 + 64;
        m[u] = max(i0 < P && weighs(c0[u]) ? -r0[u] : -INT_MAX, i1 < P && weighs(c1[u]) ? -r1[u] : -INT_MAX);
      }
    } else {
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int i0 = (jb0 + u) * kBlock + lane, i1 = i0 + 64;
        m[u] = max(i0 < P ? r0[u] : Nk + 1, i1 < P ? r1[u] : Nk + 1);
      }
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
#pragma unroll
      for (int d = 32; d >= 1; d >>= 1) m[u] = max(m[u], __shfl_xor(m[u], d, 64));
      if (lane == 0 && jb0 + u < nblk) s_bmax[pure ? nblk - 1 - (jb0 + u) : jb0 + u] = m[u];
    }
  }
  __syncthreads();
  const int per = (nblk + kSchedThreads - 1) / kSchedThreads;
  const int j0 = min(tid * per, nblk), j1 = min(j0 + per, nblk);
  int mloc = INT_MIN;
  for (int j = j0; j < j1; ++j) mloc = max(mloc, s_bmax[j]);
  int incl = mloc;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int o = __shfl_up(incl, d, 64);
    if (lane >= d) incl = max(incl, o);
  }
  if (lane == 63) s_wave[wid] = incl;
  __syncthreads();
  int pre = INT_MIN;
  for (int w2 = 0; w2 < wid; ++w2) pre = max(pre, s_wave[w2]);
  int excl = __shfl_up(incl, 1, 64);  // maximum over earlier lanes of this wave
  if (lane == 0) excl = INT_MIN;
  int run = max(pre, excl);
  int32_t* bm = sched + (int64_t)bg * 2 * nblk_cap;
  int32_t* pm = bm + nblk_cap;
  for (int j = j0; j < j1; ++j) {
    run = max(run, s_bmax[j]);
    if (pure) {
      pm[nblk - 1 - j] = -run;  // the least timestamp from block nblk - 1 - j on
    } else {
      bm[j] = s_bmax[j];
      pm[j] = run;
    }
  }
}

// ====================================================================================
// fp32 tensors.  The reference's kernels take fp32 Q, K, V as they take 16-bit ones
// (dtype-agnostic loads, deltaFlashAttention.py:41-42, 80; flashAttention.py:94-130), and
// p.to(v.dtype) then leaves p in fp32 (:98, :137).  attn_f32_kernel computes the same
// attention in fp32 throughout on the fp32 matrix instruction v_mfma_f32_32x32x2 (256
// flops per CU and clock, twice the VALU's unpacked FMA rate, and one operand dword per
// lane for 4096 flops where the VALU form needs an LDS read per four FMAs): 32 queries a
// wave, tiles of 32 keys, an exact running maximum (O rescaled at every new maximum) and
// P.V on the fp32 p.  The logical 128-row schedule, the key biases log2(w)/c and the
// variants come from the same schedule pre-pass as the 16-bit kernels.
//
// Layout.  S^T = K Q^T: a lane holds query ql = lane % 32 and, in register r, key
// 8 (r / 4) + 4 hl + r % 4 (hl = lane / 32).  O^T += V^T P^T takes the two halves' keys of
// register r as its two-deep inner dimension, so p[r] is the B operand as it is.  Row i of
// output block db is head dimension DB i + db, so one load of DB floats of a value row
// gives a lane its A operands of all DB blocks.  K, Q and V pair the inner dimension as
// the wide loads bring it (dims 8 m + 4 hl + e).
//
// Operands go from L2 to registers, with no LDS: a tile is a stream of fragments (DB of
// K, NV of V, at most 16 registers each) in a ring of R, loaded R - 1 fragments ahead of
// their MFMAs (16 MFMAs of 64 cycles each).  Two waves a SIMD cover each other's softmax.
//
// A workgroup's four waves split the keys of the same 32 queries: tile t goes to wave
// t % 4, and the waves' (maximum, sum, O) are merged through LDS at the end.  Whole rows a wave
// (128 rows a workgroup, the tiles shared through the CU's cache) were slower at every
// size: 62 against 89 TFLOP/s at 4096 tokens x 32 heads.
//
// Measured, dense causal, 128 dims unless said: 2048 tokens x 8 heads of 64 dims 63 us
// (420 us with the VALU kernel before this one), 1024 x 32 heads 148 (513), 4096 x 32
// 1557 (6415), 8192 x 32 5.87 ms (20.7; 94 TFLOP/s of 157, the rest is operand loads from
// L2 and the last-level cache).  Error against 64 bits: 3.0e-7 to 4.6e-7 (before: 4.2e-7
// to 7.0e-7).  Eight waves a workgroup were 5% faster on grids below two a CU without the
// pairing below and up to 15% slower elsewhere; a rule between the two would give a ragged
// batch other sums than its sequences alone.
// ====================================================================================
constexpr int kFRows = 32, kFTile = 32, kFWaves = 4;

template <int VARIANT, int DB>
struct F32Frags {
  static constexpr int NV = DB <= 2 ? DB : 4;      // value fragments of a tile
  static constexpr int NR = 16 / NV;               // S^T registers (key pairs) a value fragment serves
  static constexpr int F = DB + NV;                // fragments of a tile
  // ring size; F % R == 0 keeps its slots static (pure Phase 1 at 128 dims has registers for two)
  static constexpr int R = VARIANT == kPure && DB == 4 ? 2 : F % 4 == 0 ? 4 : F;
};

template <int VARIANT, int DB>
__global__ __launch_bounds__(64 * kFWaves) __attribute__((amdgpu_waves_per_eu(2, 2)))
void attn_f32_kernel(AttnArgs a, int paired) {
  constexpr int NW = kFWaves;
  using FR = F32Frags<VARIANT, DB>;
  __shared__ float s_o[NW * 16 * DB * 64];  // the waves' O, [wave][r][db][lane]
  __shared__ float s_ml[NW][2][64];         // and their maxima and sums
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hl = lane >> 5, ql = lane & 31;
  // ---- workgroup -> (head, row block): whole heads per XCD where they split evenly, the
  // longest row blocks first.  Heads are numbered head-major, so that an XCD's share of a
  // ragged batch is some heads of every sequence: with some sequences' heads instead, a long
  // one among short ones had one XCD of eight (4096 + 15 x 64 tokens, 32 heads, dense: 12.7
  // against 1.64 ms).  A grid of at most two workgroups a CU (paired) starts all at once, each
  // CU taking one of the first half and one of the second: there the second half runs from the
  // shortest up, so that every CU gets about the same work (2048 tokens x 8 heads of 64 dims:
  // 63 us, 80 with the longest first throughout) ----
  const int nrb = (a.Nq + kFRows - 1) / kFRows;
  const int units = a.B * a.Hq;
  const bool whole = (units & 7) == 0 && (!a.seq.cu || (a.Hq & 7) == 0);
  int unit, j;  // j: row blocks from the last one
  if (paired) {
    const int nx = whole ? 8 : 1;
    const int upx = units / nx, n = upx * nrb;  // an XCD's heads and workgroups
    const int idx = blockIdx.x / nx, half = (n + 1) >> 1;
    const int e = idx < half ? idx : n - 1 - (idx - half);
    unit = (int)(blockIdx.x % nx) * upx + e % upx;
    j = e / upx;
  } else if (whole) {
    const int idx = blockIdx.x >> 3;
    unit = (blockIdx.x & 7) * (units >> 3) + idx / nrb;
    j = idx % nrb;
  } else {
    unit = blockIdx.x % units;
    j = blockIdx.x / units;
  }
  // without whole heads per XCD a long sequence's row blocks go round the XCDs (an odd number
  // of units does that by itself)
  if (a.seq.cu && !whole && !(units & 1)) unit = (unit + j) % units;
  const int rb = nrb - 1 - j;
  const int h = unit / a.B, b = unit % a.B;
  const int g = h / a.G;
  const int bg = b * a.Hkv + g;
  const int Nq = a.seq.cu ? a.seq.len(b) : a.Nq;
  const int Nk = a.seq.cu ? a.seq.len(b) : a.Nk;
  const int R0 = rb * kFRows;
  if (R0 >= Nq) return;  // a row block past the end of a shorter sequence (whole workgroup)
  const int D = a.D;
  const float c = a.scale_log2;

  // ---- schedule of the logical 128-row block holding these rows (every wave computes
  // the same values).  Phase 1: packed keys [0, n1); Phase 2: keys [ds, kend), causal.
  // Keys past the block's own last row are all masked, so Phase 2 ends there. ----
  const int start_m = (R0 / kBlock) * kBlock;
  int P = a.P_host;
  if (a.P_dev) P = min(a.seq.cu ? a.P_dev[b] : *a.P_dev, a.P_host);
  if (a.seq.cu) P = min(P, Nk);
  int n1 = 0, ds = 0;
  int kend = a.causal ? min(Nk, R0 + kFRows) : Nk;
  if (VARIANT == kHybrid || VARIANT == kSanity) {
    const int nblk = (P + kBlock - 1) / kBlock;
    const int32_t* bmax = a.sched + (int64_t)bg * 2 * a.nblk_cap;
    int n_safe, last;
    safe_prefix(bmax, bmax + a.nblk_cap, nblk, start_m - a.window, n_safe, last, lane);
    ds = max(0, ((last + 1) / kBlock) * kBlock);
    // not past P: a partly filled last block counts as safe where start_m - window > Nk + 1
    // (more queries than keys), and a tile without a packed row has no row to load
    if (VARIANT == kHybrid) n1 = min(n_safe * kBlock, P);
  } else if (VARIANT == kPure) {
    // the packed blocks up to the last that holds a key at or before the last row
    const int32_t* from = a.sched + (int64_t)bg * 2 * a.nblk_cap + a.nblk_cap;
    int last;
    safe_prefix(from, from, (P + kBlock - 1) / kBlock, R0 + kFRows, n1, last, lane);
    n1 = min(n1 * kBlock, P);
    kend = 0;
  }
  const int t1 = (n1 + kFTile - 1) / kFTile;
  const int t2 = kend > ds ? (kend - ds + kFTile - 1) / kFTile : 0;
  const int T = t1 + t2;

  const float* qg = (const float*)a.q + a.seq.base(b, a.sq_b, a.sq_n) + (int64_t)h * a.sq_h;
  const float* kg = (const float*)a.k + a.seq.base(b, a.sk_b, a.sk_n) + (int64_t)g * a.sk_h;
  const float* vg = (const float*)a.v + a.seq.base(b, a.sv_b, a.sv_n) + (int64_t)g * a.sv_h;
  const float* kpg = (const float*)a.kp + a.seq.base(b, a.skp_b, a.skp_n) + (int64_t)g * a.skp_h;
  const float* vpg = (const float*)a.vp + a.seq.base(b, a.svp_b, a.svp_n) + (int64_t)g * a.svp_h;
  const float* wrow = a.wts ? a.wts + (int64_t)bg * a.wcap : nullptr;
  const int32_t* tsrow = a.tsw ? a.tsw + (int64_t)bg * a.wcap : nullptr;

  // ---- Q^T: dims 8 m + 4 hl .. + 3 of query R0 + ql (rows past Nq and dims past D zero) ----
  const int row = R0 + ql;
  f32x4 qf[4 * DB];
#pragma unroll
  for (int m = 0; m < 4 * DB; ++m) {
    const bool in = row < Nq && 8 * m < D;
    qf[m] = in ? *(const f32x4*)(qg + (int64_t)row * a.sq_n + 8 * m + 4 * hl) : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  }

  // Fragment f of tile t.  Keys past the source's end repeat its last row (a row of the
  // same tile) and get no weight; dims past D are zero (K) or never stored (V).  A row is a
  // scalar tile base plus a 32-bit lane offset (below 32 rows of less than 2^25 bytes).
  auto load = [&](auto FC, const int t, float (&x)[16]) {
    constexpr int f = decltype(FC)::value;
    const bool ph1 = t < t1;
    const int key0 = ph1 ? t * kFTile : ds + (t - t1) * kFTile;
    const unsigned last = (unsigned)((ph1 ? P : Nk) - 1 - key0);
    const unsigned sn = (unsigned)(f < DB ? (ph1 ? a.skp_n : a.sk_n) : (ph1 ? a.svp_n : a.sv_n));
    const float* base = (f < DB ? (ph1 ? kpg : kg) : (ph1 ? vpg : vg)) + (int64_t)key0 * sn;
    // opaque: the rows' offsets are formed here, not held in registers across tiles
    int ql = lane & 31, hl = lane >> 5;
    asm volatile("" : "+v"(ql), "+v"(hl));
    if constexpr (f < DB) {
      const unsigned off = min((unsigned)ql, last) * sn + 4 * hl;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int m = 4 * f + u;
        const f32x4 w = 8 * m < D ? *(const f32x4*)(base + off + 8 * m) : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int e = 0; e < 4; ++e) x[4 * u + e] = w[e];
      }
    } else {
#pragma unroll
      for (int u = 0; u < FR::NR; ++u) {
        const int r = (f - DB) * FR::NR + u;
        const unsigned off = min((unsigned)(8 * (r >> 2) + 4 * hl + (r & 3)), last) * sn;
        struct __attribute__((packed, aligned(4))) Row { float v[DB]; };
        if (D == 32 * DB) {
          const Row w = *(const Row*)(base + off + DB * ql);
#pragma unroll
          for (int e = 0; e < DB; ++e) x[DB * u + e] = w.v[e];
        } else {
#pragma unroll
          for (int e = 0; e < DB; ++e) x[DB * u + e] = base[off + min(DB * ql + e, D - 1)];
        }
      }
    }
  };

  f32x16 o[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) o[db] = f32x16{};
  float m_i = -INFINITY, l_i = 0.0f;
  float ring[FR::R][16];

  int t = wid;
  if (t < T)
    static_for<FR::R - 1>([&](auto FC) { load(FC, t, ring[decltype(FC)::value]); });
  for (; t < T; t += NW) {
    const bool ph1 = t < t1;
    const int key0 = ph1 ? t * kFTile : ds + (t - t1) * kFTile;
    const int tn = min(t + NW, T - 1);  // past the last tile: loaded again, never used
    // fragment f + R - 1 goes out before fragment f is used
    auto ahead = [&](auto FC) {
      constexpr int n = decltype(FC)::value + FR::R - 1;
      load(std::integral_constant<int, n % FR::F>{}, n < FR::F ? t : tn, ring[n % FR::R]);
      __builtin_amdgcn_sched_barrier(0);
    };
    f32x16 s = f32x16{};
    static_for<DB>([&](auto FC) {
      constexpr int f = decltype(FC)::value;
      ahead(FC);
#pragma unroll
      for (int u = 0; u < 16; ++u)
        s = __builtin_amdgcn_mfma_f32_32x32x2f32(ring[f % FR::R][u], qf[4 * f + (u >> 2)][u & 3], s, 0, 0, 0);
    });
    // ---- masks, online softmax (exact maximum) ----
    float mt = -INFINITY;
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4) {
      const int kl = key0 + 8 * r4 + 4 * hl;
      f32x4 bias = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      int4 ts = {0, 0, 0, 0};
      if ((VARIANT == kHybrid || VARIANT == kPure) && ph1) bias = *(const f32x4*)(wrow + kl);
      if (VARIANT == kPure) ts = *(const int4*)(tsrow + kl);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        bool ok = bias[e] != -INFINITY;
        if (!ph1) ok = ok && kl + e < kend && (!a.causal || kl + e <= row);     // deltaFlashAttention.py:126-130
        if (VARIANT == kPure) ok = ok && (e == 0 ? ts.x : e == 1 ? ts.y : e == 2 ? ts.z : ts.w) <= row;  // :338-341
        s[4 * r4 + e] = ok ? (s[4 * r4 + e] + bias[e]) * c : -INFINITY;
        mt = __builtin_fmaxf(mt, s[4 * r4 + e]);
      }
    }
    const float mn = __builtin_fmaxf(m_i, halves_max(mt));
    const float alpha = mn == -INFINITY ? 1.0f : exp2f(m_i - mn);
    float ps = 0.0f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = mn == -INFINITY ? 0.0f : exp2f(s[r] - mn);
      ps += s[r];
    }
    l_i = l_i * alpha + ps;
    m_i = mn;
    if (__builtin_amdgcn_ballot_w64(alpha != 1.0f)) {
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[db][r] *= alpha;
    }
    // ---- O^T += V^T P^T ----
    static_for<FR::NV>([&](auto VC) {
      constexpr int fv = decltype(VC)::value;
      ahead(std::integral_constant<int, DB + fv>{});
#pragma unroll
      for (int u = 0; u < FR::NR; ++u)
#pragma unroll
        for (int db = 0; db < DB; ++db)
          o[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(ring[(DB + fv) % FR::R][DB * u + db], s[fv * FR::NR + u],
                                                       o[db], 0, 0, 0);
    });
  }

  // ---- merge: wave w adds up registers kOwn w .. + kOwn - 1 (kOwn DB consecutive dims
  // of the lane's row) of all waves, normalises and stores rows < Nq, dims < D ----
  constexpr int kOwn = 16 / NW;
#pragma unroll
  for (int r = 0; r < 16; ++r)
#pragma unroll
    for (int db = 0; db < DB; ++db) s_o[((wid * 16 + r) * DB + db) * 64 + lane] = o[db][r];
  s_ml[wid][0][lane] = m_i;
  s_ml[wid][1][lane] = halves_sum(l_i);
  __syncthreads();
  float M = -INFINITY, L = 0.0f, f[NW];
#pragma unroll
  for (int w = 0; w < NW; ++w) M = __builtin_fmaxf(M, s_ml[w][0][lane]);
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    f[w] = M == -INFINITY ? 0.0f : exp2f(s_ml[w][0][lane] - M);
    L += s_ml[w][1][lane] * f[w];
  }
  // a row without any key (pure Phase 1) stays zero, deltaFlashAttention.py:353-354
  const float inv = L > 0.0f ? 1.0f / L : 0.0f;
  float x[kOwn * DB];
#pragma unroll
  for (int i = 0; i < kOwn * DB; ++i) {
    x[i] = 0.0f;
#pragma unroll
    for (int w = 0; w < NW; ++w) x[i] += s_o[((w * 16 + kOwn * wid) * DB + i) * 64 + lane] * f[w];
    x[i] *= inv;
  }
  if (row >= Nq) return;
  const int r0 = kOwn * wid, d0 = DB * (8 * (r0 >> 2) + 4 * hl + (r0 & 3));
  float* orow = (float*)a.out + a.seq.base(b, a.so_b, a.so_n) + (int64_t)h * a.so_h + (int64_t)row * a.so_n;
#pragma unroll
  for (int i = 0; i < kOwn * DB; i += 2)  // D is even: two dims are both in or both out
    if (d0 + i < D) *(f32x2*)(orow + d0 + i) = f32x2{x[i], x[i + 1]};
}

// Compute units of the current device (cached per device).
static int cu_count() {
  static int n[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (!n[dev]) {
    int v = 0;
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || v <= 0) v = 256;
    n[dev] = v;
  }
  return n[dev];
}

// Items (the units times their row groups) of attn_w64_kernel with ncb column blocks a wave.
static int64_t attn_items(const AttnArgs& a, int ncb) {
  const int rows = 128 * ncb / a.hpw;
  return (int64_t)((a.Nq + rows - 1) / rows) * a.units;
}

// Those of them that hold rows: a ragged batch's tokens as if its sequences were one.
static int64_t attn_items_real(const AttnArgs& a, int ncb) {
  const int64_t items = attn_items(a, ncb);
  if (!a.seq.cu) return items;
  const int rows = 128 * ncb / a.hpw;
  return std::min<int64_t>(items, (int64_t)((a.seq.total + rows - 1) / rows) * (a.units / a.B));
}

template <int V, int DT, int NCB, bool LAZY>
static int launch_attn_cb(AttnArgs& a, hipStream_t st) {
  static int done = 0;
  if (!done) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&attn_w64_kernel<V, DT, NCB, LAZY>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, kWLds);
    if (e != hipSuccess) return set_error(DA_ERR_HIP, "hipFuncSetAttribute: %s", hipGetErrorString(e));
    done = 1;
  }
  a.slots = 2 * cu_count() / 8;
  const int64_t items = attn_items(a, NCB);
  a.n_row_groups = (int)(items / a.units);
  // persistent: as many workgroups as run at once (two a CU) take items until the queues are
  // empty.  Only from more than four items a slot on, of which a quarter or more hold rows:
  // before the queues gain anything each workgroup's looks at eight of them, and a take for every
  // empty item of a ragged batch, cost more than they save (hybrid 8192 tokens, 1024 items: 276
  // against 262 us static, sanity 107 / 81, 16384 tokens 171 / 160; 30 x 64 + 3500 + 200 tokens,
  // 14080 items 958 of them with rows: 328 / 209)
  const int64_t real = attn_items_real(a, NCB);
  if (NCB == 1 || real <= 8 * cu_count() || 4 * real < items) a.queue = nullptr;
  const unsigned grid = (unsigned)(a.queue ? 2 * cu_count() : items);
  hipLaunchKernelGGL((attn_w64_kernel<V, DT, NCB, LAZY>), dim3(grid), dim3(256), kWLds, st, a);
  return check_launch("attention kernel");
}

template <int V, int DT, bool LAZY>
static int launch_attn_rows(AttnArgs& a, hipStream_t st) {
  // Up to two 64-row items a CU, 32 rows a wave.  Two workgroups a CU run at once either way, but
  // the longest item, which the causal triangle's end waits for, takes half as long, and a chip
  // that 64-row items fill by half is full.  Dense, 32 heads in groups of 4: 1024 tokens 29.4
  // against 44.0 us, 2048 53 / 80, 4096 139 / 163, beyond the line 6000 302 / 286, 8000 508 / 444;
  // delta step of 1531 tokens 64.9 / 78.9, 2300 73 / 87, beyond 6000 168 / 171, 8190 248 / 242;
  // heads of their own, 1067 tokens x 32 37 / 52.  Without the causal mask all items are as long,
  // and only the second reason is left: one item a CU (2048 tokens 72 / 83, 4096, two a CU, 260 /
  // 228), unless half of a 64-row item would be past the rows (100 tokens x 16 x 32 heads of their
  // own 17 / 20).  A ragged batch's items are counted by its tokens, not by the longest sequence (4096 +
  // 15 x 64 tokens, dense, 12 heads in groups of 3: 149 / 246; 8 heads 109 / 172).
  const bool short_gains = a.causal || attn_items(a, 1) == attn_items(a, 2);
  return attn_items_real(a, 2) <= (short_gains ? 2 : 1) * cu_count() ? launch_attn_cb<V, DT, 1, LAZY>(a, st)
                                                                    : launch_attn_cb<V, DT, 2, LAZY>(a, st);
}

template <int V, int DT>
static int launch_attn_t(AttnArgs& a, hipStream_t st) {
  return a.hpw == 4 ? launch_attn_rows<V, DT, true>(a, st) : launch_attn_rows<V, DT, false>(a, st);
}

template <int DT>
static int launch_attn_dt(int variant, AttnArgs& a, hipStream_t st) {
  switch (variant) {
    case kHybrid: return launch_attn_t<kHybrid, DT>(a, st);
    case kSanity: return launch_attn_t<kSanity, DT>(a, st);
    case kPure: return launch_attn_t<kPure, DT>(a, st);
    default: return launch_attn_t<kDense, DT>(a, st);
  }
}

template <int V, int DB>
static int launch_attn_f32_t(const AttnArgs& a, hipStream_t st) {
  const int64_t grid = (int64_t)a.B * a.Hq * ((a.Nq + kFRows - 1) / kFRows);
  if (grid >= (1ll << 31)) return set_error(DA_ERR_INVALID, "attention (fp32): grid too large");
  hipLaunchKernelGGL((attn_f32_kernel<V, DB>), dim3((unsigned)grid), dim3(64 * kFWaves), 0, st, a,
                     grid <= 2 * cu_count() ? 1 : 0);
  return check_launch("attention kernel (fp32)");
}

template <int V>
static int launch_attn_f32(const AttnArgs& a, hipStream_t st) {
  switch ((a.D + 31) / 32) {
    case 1: return launch_attn_f32_t<V, 1>(a, st);
    case 2: return launch_attn_f32_t<V, 2>(a, st);
    case 3: return launch_attn_f32_t<V, 3>(a, st);
    default: return launch_attn_f32_t<V, 4>(a, st);
  }
}

static int launch_attn(int variant, int dtype, AttnArgs& a, hipStream_t st) {
  if (dtype == DA_F32) {
    switch (variant) {
      case kHybrid: return launch_attn_f32<kHybrid>(a, st);
      case kSanity: return launch_attn_f32<kSanity>(a, st);
      case kPure: return launch_attn_f32<kPure>(a, st);
      default: return launch_attn_f32<kDense>(a, st);
    }
  }
  return dtype == DA_F16 ? launch_attn_dt<DA_F16>(variant, a, st) : launch_attn_dt<DA_BF16>(variant, a, st);
}

static bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

static int fill_common(AttnArgs& a, const void* q, const void* k, const void* v, void* out,
                       int64_t B, int64_t Hq, int64_t Hkv, int64_t Nq, int64_t Nk, int64_t D,
                       const int64_t* st, float scale, const char* who) {
  DA_REQUIRE(q && k && v && out && st, "%s: null pointer", who);
  DA_REQUIRE(B > 0 && Hq > 0 && Hkv > 0 && Nq > 0 && Nk > 0, "%s: empty shape", who);
  if (D <= 0 || D > kD || (D & 7))
    return set_error(DA_ERR_UNSUPPORTED, "%s: head_dim must be a multiple of 8 in [8, 128] (got %lld)", who,
                     (long long)D);
  DA_REQUIRE(Hq % Hkv == 0, "%s: Hq (%lld) must be a multiple of Hkv (%lld)", who, (long long)Hq, (long long)Hkv);
  DA_REQUIRE(Nq < (1ll << 30) && Nk < (1ll << 30), "%s: sequence too long", who);
  DA_REQUIRE(scale > 0.0f, "%s: scale must be positive", who);
  for (int i = 0; i < 18; ++i)
    DA_REQUIRE((st[i] & 7) == 0, "%s: strides must be multiples of 8 elements (stride %d = %lld)", who, i, (long long)st[i]);
  DA_REQUIRE(aligned16(q) && aligned16(k) && aligned16(v) && aligned16(out), "%s: tensors must be 16-byte aligned", who);
  for (int i : {DA_STRIDE_K + 2, DA_STRIDE_V + 2})
    DA_REQUIRE(st[i] >= D && st[i] < (1ll << 23),
               "%s: key/value sequence strides must be in [head_dim, 2^23) (stride %d = %lld)", who, i, (long long)st[i]);
  a.q = (const uint16_t*)q; a.k = (const uint16_t*)k; a.v = (const uint16_t*)v; a.out = (uint16_t*)out;
  a.sq_b = st[DA_STRIDE_Q]; a.sq_h = st[DA_STRIDE_Q + 1]; a.sq_n = st[DA_STRIDE_Q + 2];
  a.sk_b = st[DA_STRIDE_K]; a.sk_h = st[DA_STRIDE_K + 1]; a.sk_n = st[DA_STRIDE_K + 2];
  a.sv_b = st[DA_STRIDE_V]; a.sv_h = st[DA_STRIDE_V + 1]; a.sv_n = st[DA_STRIDE_V + 2];
  a.so_b = st[DA_STRIDE_OUT]; a.so_h = st[DA_STRIDE_OUT + 1]; a.so_n = st[DA_STRIDE_OUT + 2];
  a.B = (int)B; a.Hq = (int)Hq; a.Hkv = (int)Hkv; a.G = (int)(Hq / Hkv);
  a.Nq = (int)Nq; a.Nk = (int)Nk;
  a.D = (int)D;
  a.scale_log2 = scale * 1.4426950408889634f;
  a.hpw = (a.G % 4 == 0) ? 4 : (a.G % 2 == 0 ? 2 : 1);
  a.units = (int)(B * Hkv * (a.G / a.hpw));
  DA_REQUIRE(attn_items(a, 2) < (1ll << 31), "%s: grid too large", who);
  return DA_OK;
}

}  // namespace da

using namespace da;

// Workspace of da_hybrid_prefill: the schedule ([B*Hkv][2][nblk] int32), then, each at
// a 256-byte boundary, the key biases ([B*Hkv][wcap] fp32), the timestamps of the pure
// Phase-1 variant ([B*Hkv][wcap] int32), 64 zeros and the attention kernel's 8
// work-queue counters; nblk = ceil(num_packed / 128) (at least 1), wcap = 128 nblk.
struct HybridWs {
  int nblk, wcap;
  int64_t w_off, ts_off, zeros_off, queue_off, total;
};
static int64_t round256(int64_t x) { return (x + 255) & ~(int64_t)255; }
static HybridWs hybrid_ws(int64_t B, int64_t Hkv, int64_t num_packed) {
  HybridWs w;
  const int64_t nblk = std::max<int64_t>(1, (num_packed + kBlock - 1) / kBlock);
  w.nblk = (int)nblk;
  w.wcap = (int)(nblk * kBlock);
  w.w_off = round256(B * Hkv * 2 * nblk * (int64_t)sizeof(int32_t));
  w.ts_off = w.w_off + round256(B * Hkv * w.wcap * (int64_t)sizeof(float));
  w.zeros_off = w.ts_off + round256(B * Hkv * w.wcap * (int64_t)sizeof(int32_t));
  w.queue_off = w.zeros_off + 256;
  w.total = w.queue_off + 256;
  return w;
}

extern "C" int64_t da_hybrid_workspace_size(int64_t B, int64_t Hkv, int64_t num_packed) {
  return hybrid_ws(B, Hkv, num_packed).total;
}

// Everything of da_hybrid_prefill / da_hybrid_prefill_varlen after the shapes are known:
// validation of the packed tensors and workspace, the schedule pre-pass, the launch.
// P_bound is the host upper bound of P (num_packed, or the longest sequence of a ragged
// batch), which sizes the workspace.
static int hybrid_impl(const char* who, AttnArgs& a, const void* k_packed, const void* v_packed,
                       const int32_t* timestamps, const void* counts, int counts_dtype, int dtype,
                       int64_t B, int64_t Hkv, int64_t Nk, const int64_t* strides, int64_t P_bound,
                       const int32_t* num_packed_dev, int64_t window, int variant, int no_count,
                       void* workspace, int64_t workspace_bytes, hipStream_t st) {
  DA_REQUIRE(variant == DA_VARIANT_HYBRID || variant == DA_VARIANT_SANITY ||
                 variant == DA_VARIANT_PURE_PHASE1,
             "%s: unknown variant %d", who, variant);
  DA_REQUIRE(k_packed && v_packed && timestamps && counts, "%s: null packed tensor", who);
  DA_REQUIRE(counts_dtype == DA_I32 || counts_dtype == DA_F32, "%s: counts must be int32 or fp32", who);
  DA_REQUIRE(P_bound > 0 && P_bound <= 4096 * kBlock, "%s: num_packed must be in [1, %d]", who, 4096 * kBlock);
  DA_REQUIRE(window >= 0 && window < (1ll << 30), "%s: window must be >= 0", who);
  DA_REQUIRE(aligned16(k_packed) && aligned16(v_packed), "%s: packed tensors must be 16-byte aligned", who);
  for (int i : {DA_STRIDE_KP + 2, DA_STRIDE_VP + 2})
    DA_REQUIRE(strides[i] >= a.D && strides[i] < (1ll << 23),
               "%s: packed sequence strides must be in [head_dim, 2^23) (stride %d = %lld)", who, i,
               (long long)strides[i]);
  DA_REQUIRE(strides[DA_STRIDE_TS + 2] == 1 && strides[DA_STRIDE_CNT + 2] == 1,
             "%s: timestamps and counts must be contiguous along the packed axis", who);
  const int64_t need = da_hybrid_workspace_size(B, Hkv, P_bound);
  if (!workspace || workspace_bytes < need)
    return set_error(DA_ERR_WORKSPACE, "%s: workspace of %lld bytes required", who, (long long)need);
  a.kp = (const uint16_t*)k_packed; a.vp = (const uint16_t*)v_packed;
  a.ts = timestamps; a.cnt = counts;
  a.skp_b = strides[DA_STRIDE_KP]; a.skp_h = strides[DA_STRIDE_KP + 1]; a.skp_n = strides[DA_STRIDE_KP + 2];
  a.svp_b = strides[DA_STRIDE_VP]; a.svp_h = strides[DA_STRIDE_VP + 1]; a.svp_n = strides[DA_STRIDE_VP + 2];
  a.sts_b = strides[DA_STRIDE_TS]; a.sts_h = strides[DA_STRIDE_TS + 1];
  a.scnt_b = strides[DA_STRIDE_CNT]; a.scnt_h = strides[DA_STRIDE_CNT + 1];
  a.P_host = (int)P_bound;
  a.P_dev = num_packed_dev;
  a.window = (int)window;
  a.no_count = no_count ? 1 : 0;
  a.cnt_is_float = counts_dtype == DA_F32;
  a.causal = 1;
  const HybridWs wl = hybrid_ws(B, Hkv, P_bound);
  char* ws = (char*)workspace;
  a.nblk_cap = wl.nblk;
  a.sched = (const int32_t*)ws;
  a.wcap = wl.wcap;
  a.wts = (const float*)(ws + wl.w_off);
  a.tsw = (const int32_t*)(ws + wl.ts_off);
  a.zeros = (const float*)(ws + wl.zeros_off);
  SchedPrep prep = {};
  if (variant != DA_VARIANT_SANITY) {
    prep.cnt = counts;
    prep.scnt_b = a.scnt_b;
    prep.scnt_h = a.scnt_h;
    prep.cnt_is_float = a.cnt_is_float;
    prep.no_count = a.no_count;
    prep.scale_log2 = a.scale_log2;
    prep.wts = (float*)(ws + wl.w_off);
    prep.tsw = variant == DA_VARIANT_PURE_PHASE1 ? (int32_t*)(ws + wl.ts_off) : nullptr;
    prep.zeros = (float*)(ws + wl.zeros_off);
    prep.wcap = wl.wcap;
  }
  const unsigned prep_chunks = prep.wts ? (unsigned)((wl.wcap + kSchedThreads - 1) / kSchedThreads) : 0u;
  // the 16-bit kernel's persistent grid takes its items from 8 counters in the workspace
  a.queue = dtype != DA_F32 ? (int*)(ws + wl.queue_off) : nullptr;
  hipLaunchKernelGGL(hybrid_schedule_kernel, dim3((unsigned)(B * Hkv), 1 + prep_chunks), dim3(kSchedThreads), 0, st,
                     timestamps, a.sts_b, a.sts_h, (int)Hkv, (int)P_bound, num_packed_dev, (int)Nk, a.seq,
                     a.nblk_cap, (int32_t*)ws, prep, a.queue);
  if (int rc = check_launch("hybrid prefill (schedule)")) return rc;
  const int kv = variant == DA_VARIANT_HYBRID ? kHybrid : (variant == DA_VARIANT_SANITY ? kSanity : kPure);
  return launch_attn(kv, dtype, a, st);
}

extern "C" int da_hybrid_prefill(const void* q, const void* k, const void* v, const void* k_packed,
                                 const void* v_packed, const int32_t* timestamps,
                                 const void* counts, int counts_dtype, void* out, int dtype,
                                 int64_t B, int64_t Hq, int64_t Hkv, int64_t Nq, int64_t Nk,
                                 int64_t D, const int64_t* strides, int64_t num_packed,
                                 const int32_t* num_packed_dev, int64_t window, float scale,
                                 int variant, int no_count, void* workspace,
                                 int64_t workspace_bytes, void* stream) {
  const char* who = "da_hybrid_prefill";
  if (dtype != DA_BF16 && dtype != DA_F16 && dtype != DA_F32)
    return set_error(DA_ERR_UNSUPPORTED, "%s: tensors must be bf16, fp16 or fp32", who);
  AttnArgs a = {};
  if (int rc = fill_common(a, q, k, v, out, B, Hq, Hkv, Nq, Nk, D, strides, scale, who)) return rc;
  a.seq = SeqMap{nullptr, 0, (int)Nq};
  return hybrid_impl(who, a, k_packed, v_packed, timestamps, counts, counts_dtype, dtype, B, Hkv, Nk, strides,
                     num_packed, num_packed_dev, window, variant, no_count, workspace, workspace_bytes,
                     (hipStream_t)stream);
}

extern "C" int da_dense_prefill(const void* q, const void* k, const void* v, void* out, int dtype,
                                int64_t B, int64_t Hq, int64_t Hkv, int64_t Nq, int64_t Nk,
                                int64_t D, const int64_t* strides, int causal, float scale,
                                void* stream) {
  if (dtype != DA_BF16 && dtype != DA_F16 && dtype != DA_F32)
    return set_error(DA_ERR_UNSUPPORTED, "da_dense_prefill: tensors must be bf16, fp16 or fp32");
  AttnArgs a = {};
  int rc = fill_common(a, q, k, v, out, B, Hq, Hkv, Nq, Nk, D, strides, scale, "da_dense_prefill");
  if (rc) return rc;
  a.seq = SeqMap{nullptr, 0, (int)Nq};
  a.kp = a.k; a.vp = a.v;
  a.causal = causal ? 1 : 0;
  a.P_host = 0;
  return launch_attn(kDense, dtype, a, (hipStream_t)stream);
}

// ---- ragged (varlen) batches: sequence b is tokens cu_seqlens[b] .. cu_seqlens[b+1]-1 of
// [T, H, D] tensors; every sequence is exactly a B = 1 prefill of its own length ----
static int varlen_common(const char* who, AttnArgs& a, const void* q, const void* k, const void* v, void* out,
                         int dtype, int64_t B, int64_t Hq, int64_t Hkv, int64_t T, int64_t D,
                         const int64_t* strides, const int32_t* cu_seqlens, int64_t max_seqlen, float scale) {
  if (dtype != DA_BF16 && dtype != DA_F16 && dtype != DA_F32)
    return set_error(DA_ERR_UNSUPPORTED, "%s: tensors must be bf16, fp16 or fp32", who);
  DA_REQUIRE(cu_seqlens, "%s: null cu_seqlens", who);
  DA_REQUIRE(T > 0 && max_seqlen > 0 && max_seqlen <= T, "%s: need 0 < max_seqlen <= total tokens", who);
  DA_REQUIRE(T < (1ll << 31), "%s: too many tokens", who);
  if (int rc = fill_common(a, q, k, v, out, B, Hq, Hkv, max_seqlen, max_seqlen, D, strides, scale, who)) return rc;
  a.seq = SeqMap{cu_seqlens, (int)T, (int)max_seqlen};
  return DA_OK;
}

extern "C" int64_t da_hybrid_varlen_workspace_size(int64_t B, int64_t Hkv, int64_t max_seqlen) {
  return da_hybrid_workspace_size(B, Hkv, max_seqlen);
}

extern "C" int da_hybrid_prefill_varlen(const void* q, const void* k, const void* v, const void* k_packed,
                                        const void* v_packed, const int32_t* timestamps, const void* counts,
                                        int counts_dtype, void* out, int dtype, int64_t B, int64_t Hq,
                                        int64_t Hkv, int64_t T, int64_t D, const int64_t* strides,
                                        const int32_t* cu_seqlens, int64_t max_seqlen,
                                        const int32_t* num_packed, int64_t window, float scale, int variant,
                                        int no_count, void* workspace, int64_t workspace_bytes, void* stream) {
  const char* who = "da_hybrid_prefill_varlen";
  AttnArgs a = {};
  if (int rc = varlen_common(who, a, q, k, v, out, dtype, B, Hq, Hkv, T, D, strides, cu_seqlens, max_seqlen, scale))
    return rc;
  DA_REQUIRE(num_packed, "%s: null num_packed", who);
  return hybrid_impl(who, a, k_packed, v_packed, timestamps, counts, counts_dtype, dtype, B, Hkv, max_seqlen,
                     strides, max_seqlen, num_packed, window, variant, no_count, workspace, workspace_bytes,
                     (hipStream_t)stream);
}

extern "C" int da_dense_prefill_varlen(const void* q, const void* k, const void* v, void* out, int dtype,
                                       int64_t B, int64_t Hq, int64_t Hkv, int64_t T, int64_t D,
                                       const int64_t* strides, const int32_t* cu_seqlens, int64_t max_seqlen,
                                       int causal, float scale, void* stream) {
  AttnArgs a = {};
  if (int rc = varlen_common("da_dense_prefill_varlen", a, q, k, v, out, dtype, B, Hq, Hkv, T, D, strides,
                             cu_seqlens, max_seqlen, scale))
    return rc;
  a.kp = a.k; a.vp = a.v;
  a.causal = causal ? 1 : 0;
  a.P_host = 0;
  return launch_attn(kDense, dtype, a, (hipStream_t)stream);
}
