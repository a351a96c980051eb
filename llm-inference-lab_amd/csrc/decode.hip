// Matrix products for few rows (decode steps and short portions; up to 1,024 rows of
// a small matrix, in tiles of 16 to 64 rows), gfx950.  At this size a step is bound by launch count and by memory
// latency, not by arithmetic, so one kernel does what the general path does in
// three or four:
//
//   [RMSNorm of the float32 residual rows]  ->  x . W^T  ->  K-split reduction
//   ->  epilogue: bias / add into the residual / float32 logits / SwiGLU /
//                 rotary + write of q, and of k and v into their cache pages
//
// W comes packed in MFMA fragment order (see llmlab_pack_weight): the 16 rows x 32
// columns a wave multiplies in one step are 1 KB of consecutive memory, lane l
// owning bytes 16 l .. 16 l + 15, and the steps of a strip follow each other.  A
// wave therefore streams one contiguous run of memory with full cache lines,
// which at these sizes is worth a factor of two over rows of 64 bytes each.
//
// A block owns `nsb` strips of 16 weight rows (for the q/k/v projection: one head,
// or two strips of one) and splits K over `kw` waves per strip, so blockDim =
// 64 * nsb * kw.  Every wave streams its slice of W from HBM straight into MFMA B
// fragments through a ring of registers, and leaves its partial sums in LDS; the
// block adds the partial sums in a fixed order (no atomics, results do not depend
// on timing) and applies the epilogue.
//
// The rows of x are staged once per block in LDS as bfloat16 (STAGE), so the strips
// of a block share them; or every wave reads its slice from global memory (plain
// products only).  The norm is folded in without a pass of its own:
//   norm(x) . W^T = inv_rms[m] * ((x * w_norm) . W^T)
// x * w_norm is what is staged (or built on the fly), the sum of squares falls out
// of the same read, and inv_rms[m] scales the reduced sums in the epilogue.
//
// What the epilogue needs from global memory (bias, positions, page numbers,
// rotary frequencies, the residual value it adds to) is asked for at the start of the
// kernel, so those latencies overlap the weight stream instead of following it.
//
// What a block does before its first load counts: a wave issues about 450 instructions a
// microsecond, and loads come back in the order they were asked for.  So the rows of x are
// asked for first, then what the epilogue needs, then the weights; nothing is waited for in between;
// sizes that need a division come from the host (SkinnyArgs).  By clock stamps inside the kernels
// (0.5B shape, one row, from a block's start): gate/up has all its loads on their way after 0.5 us and its
// rows staged after 1.1 (0.9 and 2.9 with the weights first), q/k/v, which waited for positions and pages as
// well, after 1.5 and 2.7 (2.6 and 3.9).  A decode step of 8 requests in
// float32 takes 1,286 us where it took 1,371; in bfloat16, together with the merge of the attention's waves, 1 / 8 / 64
// requests 854 / 942 / 1,461 -> 785 / 906 / 1,392 us, 8 of the 7B shape 3,801 -> 3,697.
//
// A compute unit draws only about 50 GB/s from HBM, so a product with a narrow
// output (few strips, hence few blocks) is bound by the units it uses, not by the
// chip.  Epilogue SK_PART cuts such a product along K over `ksplit` groups of blocks
// as well and leaves one piece of the result per group, unsummed: no second kernel
// and no atomics.  The pieces are owed to the float32 rows they would have been
// added to; the next kernel that reads those rows (under a fused norm) adds them on
// the fly in their order, and the next SK_RESID product into those rows folds them
// in for good (`pend` below).
//
// More than 16 rows are cut into tiles of 16 MB rows (MB = 1, 2 or 4) that separate
// blocks take: a block then stages, norms and multiplies its own rows only, and
// four times the blocks hide each other's latencies.  The tiles of one set of
// columns read the same part of W; their block numbers are equal modulo 8 and
// adjacent there, so that they run on one XCD at about the same time and all but
// the first find W in its L2.  Measured at 64 rows of the 0.5B shapes, tiles of 16
// rows against one tile of 64: q/k/v 5.2 against 9.8 us, output product 4.3
// against 7.7, down product 8.7 against 21.8.
//
// Fragment layout of v_mfma_f32_16x16x32_bf16 (lane l): A row l%16, B column l%16,
// k = 8*(l/16)..+7; result element i: row 4*(l/16)+i, column l%16.
#include <stdlib.h>

#include <type_traits>

#include "common.h"

enum { SK_STORE = 0, SK_RESID = 1, SK_F32 = 2, SK_SWIGLU = 3, SK_QKV = 4, SK_PART = 5 };

struct SkinnyArgs {
  const void* x;        // NORM: float32 rows of the residual stream; else [M, K] in the compute type
  const int* x_rows;    // NORM only, optional: row of x for each m (final norm of wanted rows)
  const void* norm_w;   // NORM: [K]
  const void* W;        // [N, K]: bfloat16 packed in fragment order, float32 row by row
  const void* bias;     // [N] or null
  void* out;            // STORE/SWIGLU, QKV (q): compute type [M, ldo]; RESID/F32: float [M, ldo]
  // QKV epilogue
  const float* inv_freq;   // [d/2] or null (no rotation)
  const int* positions;    // [M]
  const int* row_req;      // [M]
  const int* table;        // block table
  void* kcache;            // may be null: q only is produced, k and v heads are skipped
  void* vcache;
  int M, N, K, ldo, n_out;
  int norm_w_bf16, bias_bf16;
  int nsb, kw;
  int qsplit;   // QKV: blocks per head (1, or d/32: a block then owns the strips p and p + d/32)
  int nq, nkv, d, table_stride, page_size;
  float eps;
  // Sums that a former product left in pieces (SK_PART) and that still belong to the
  // float32 rows this kernel reads (NORM) or adds into (RESID): pend[s][row][pend_ld],
  // s < pend_splits, added in the order of s.
  const float* pend;
  int pend_splits, pend_ld;
  size_t pend_stride;
  // SK_PART: K is split over `ksplit` groups of blocks as well; group s leaves its sums
  // (no residual, bias in group 0) in out[s][M][ldo], part_stride numbers apart.
  int ksplit;
  size_t part_stride;
  int act;         // SK_STORE: 1 = max(z, 0)^2 before the rounding; SK_SWIGLU: 2 = gelu (tanh form) gate, 3 = the clamped pair
  float limit, slope, shift;      // the clamped pair's constants
  // SK_PART: segments of the columns may read inputs of their own: the strips from seg_end[s - 1] to
  // seg_end[s] - 1 multiply the rows x + s * seg_stride (segs <= 1: all strips read x).
  int segs;
  int seg_end[7];
  size_t seg_stride;
  int tiles;       // tiles of 16 MB rows
  int col_blocks;  // blocks that a tile of rows takes (sets of columns); grid y counts the groups of K
  // What every block would otherwise work out before its first load:
  int threads;         // of a block
  int nsb_inv;         // ceil(65536 / nsb): n / nsb is (n * nsb_inv) >> 16 for n < 4096
  unsigned tiles_inv;  // ceil(2^32 / tiles), tiles > 1: j / tiles is the upper half of j * tiles_inv
  unsigned qsplit_inv; // the same of qsplit, qsplit > 1
  int steps;           // steps of the inner size
  int group_steps;     // ... of a group of K
  int wave_steps;      // ... of a wave
  int last_wave_steps; // ... of a wave of the last group that has any, which may be shorter
  int wpr_shift;       // log2 of the waves that share a staged row
};

__device__ __forceinline__ float sk_silu(float z) { return z / (1.f + __expf(-z)); }
// gelu (tanh form), 0.5 z (1 + tanh(sqrt(2/pi) (z + 0.044715 z^3))), as z * sigmoid(2 t)
__device__ __forceinline__ float sk_gelu_tanh(float z) {
  const float t = 0.7978845608028654f * (z + 0.044715f * z * z * z);
  return z / (1.f + __expf(-2.f * t));
}

// act(gate) * up; the clamped pair: g = min(gate, limit), u = up held within -limit .. limit,
// g * sigmoid(slope * g) * (u + shift)
// (bfloat16 results by the hardware's exponential, float32 results by the library's functions)
template <typename T>
__device__ __forceinline__ float sk_pair(float g, float u, const SkinnyArgs& a) {
  if constexpr (sizeof(T) == 4) {
    if (a.act == 2) {
      const float t = 0.7978845608028654f * (g + 0.044715f * g * g * g);
      return 0.5f * g * (1.f + tanhf(t)) * u;
    }
    if (a.act != 3) return g / (1.f + expf(-g)) * u;
    g = fminf(g, a.limit);
    return g / (1.f + expf(-a.slope * g)) * (fminf(fmaxf(u, -a.limit), a.limit) + a.shift);
  }
  if (a.act != 3) return (a.act == 2 ? sk_gelu_tanh(g) : sk_silu(g)) * u;
  g = fminf(g, a.limit);
  return g / (1.f + __expf(-a.slope * g)) * (fminf(fmaxf(u, -a.limit), a.limit) + a.shift);
}

// A sum of squares and two more, `alone` rounded by itself before the other is added.  The roundings are fixed here: left to
// the compiler they differ between the places it is inlined at, and a row's norm with the instance that takes it.
__device__ __forceinline__ float sk_add_squares(float sum, float other, float alone) {
#pragma clang fp contract(off)
  const float square = alone * alone;
  return sum + fmaf(other, other, square);
}

// What a step of the inner size is: 16 rows of W by 64 bytes, 16 bytes a lane.  bfloat16: 32 numbers, one
// matrix instruction.  float32: 16 numbers, four (lane (c, g) holds the numbers 4 g .. 4 g + 3 of row c; instruction
// e contracts the e-th of all four groups, the same four numbers of both operands), 32-bit products and sums in
// sixteen running sums that meet at the end: the order of a tree, so that a sum is as exact as the one of
// the kernel whose lanes split the inner size (relative error against 64 bits 1.0e-7 to 1.8e-7 where that has 0.9e-7 to
// 2.2e-7; one running sum: 2e-7 to 8.5e-7).  W lies row by row, so that a load of a wave is 16 pieces of 64 bytes; packed
// like bfloat16 it would be 8 to 20 % faster (8 rows of 9728 x 896 13.8 us against 15.0), which every other reader
// of the matrix would have to learn.  8 / 64 rows of 9728 x 896 15 / 31 us (17.4 / 59 by that kernel), of 896 x
// 4864 in four pieces 8.5 / 24 (12.7 / 26), of 151936 x 896 106 / 287 (150 / 1,120), and the norm, the rotation and the
// writing of the cache ride along: a decode step of eight requests of the 0.5B shape 2.20 -> 1.37 ms.
template <typename T>
struct SkStep;
template <>
struct SkStep<bf16_t> {
  typedef bf16x8 frag;
  static constexpr int LEN = 32, PER = 8, SUMS = 1;
  static constexpr bool KEEPS_INF = false;
  static __device__ __forceinline__ void mul(frag x, frag w, floatx4* acc, int) {
    acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, w, acc[0], 0, 0, 0);
  }
};
template <>
struct SkStep<float> {
  typedef floatx4 frag;
  static constexpr int LEN = 16, PER = 4, SUMS = 16;
  static constexpr bool KEEPS_INF = true;      // (a step past the end is zeros of both operands: an infinity of x met by a zero would be NaN)
  static __device__ __forceinline__ void mul(frag x, frag w, floatx4* acc, int step) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      floatx4& sum = acc[(step & 3) * 4 + e];
      sum = __builtin_amdgcn_mfma_f32_16x16x4f32(x[e], w[e], sum, 0, 0, 0);
    }
  }
};
// eight neighbouring numbers
template <typename T>
struct Sk8;
template <>
struct Sk8<bf16_t> {
  bf16x8 v;
  __device__ __forceinline__ void load(const bf16_t* p) { v = *(const bf16x8*)p; }
  __device__ __forceinline__ void store(bf16_t* p) const { *(bf16x8*)p = v; }
  __device__ __forceinline__ void set(int i, float f) { v[i] = (bf16_t)f; }
};
template <>
struct Sk8<float> {
  floatx4 lo, hi;
  __device__ __forceinline__ void load(const float* p) { lo = *(const floatx4*)p; hi = *(const floatx4*)(p + 4); }
  __device__ __forceinline__ void store(float* p) const { *(floatx4*)p = lo; *(floatx4*)(p + 4) = hi; }
  __device__ __forceinline__ void set(int i, float f) { if (i < 4) lo[i] = f; else hi[i - 4] = f; }
};

// Loads of W (and of x where it is not staged) run R steps ahead of the MFMAs in a
// ring of registers that is refilled slot by slot, so a wave always has R loads
// in flight and never waits for all of them at once.  Measured per decode step, staged
// ring 4 / 6 / 8 / 12 / 16 deep: one request of the 7B shape 3.21 / 3.13 / 3.07 / 3.34 /
// 3.76 ms, eight of the 32B shape 15.83 / 15.66 / 15.61 / 15.96 / 16.96, eight of the
// 0.5B shape 0.963 / 0.976 / 0.962 / 1.010 / 1.162 (a block of 16 waves has 128
// registers a lane; a wave with fewer steps than the ring is deep reads its last tile
// again for nothing); the ring of the unstaged products 4 / 6 / 8 deep: 15.61 / 15.52 /
// 15.51 and 0.965 / 0.959 / 0.971.
constexpr int SK_RING_STAGE = 8, SK_RING_DIRECT = 6;
__host__ __device__ constexpr int sk_ring(int mb, bool stage) {
  return stage ? SK_RING_STAGE : (mb >= 4 ? SK_RING_DIRECT / 2 : SK_RING_DIRECT);
}

constexpr int SK_APAD = 16;  // padding of a staged row, in bytes: 16-byte reads of 8 lanes cover all banks

// floats of LDS before the staged rows (host and device must agree)
__host__ __device__ inline size_t sk_float_words(int nsb, int kw, int mb) {
  size_t f = (size_t)kw * nsb * mb * 256;        // partial sums
  f += (size_t)mb * 16 + 16;                      // inverse rms; sums of squares of the parts of a row
  f += (size_t)16 * nsb;                          // bias
  f += (size_t)mb * 16 * 2 + 128;                 // positions, pages, frequencies
  return (f + 3) & ~(size_t)3;
}

template <typename T, int MB, int EPI, bool NORM, bool STAGE>
__global__ __launch_bounds__(MB >= 4 ? 512 : 1024) void skinny_block_kernel(SkinnyArgs a) {
  static_assert(STAGE || !NORM, "the fused norm needs the staged rows");
  using S = SkStep<T>;
  using Frag = typename S::frag;
  extern __shared__ __attribute__((aligned(16))) float smem[];
  // (the arguments that the first loads need come in one trip, not in one per branch that leads to them)
  asm volatile("" :: "s"(a.tiles), "s"(a.nsb), "s"(a.threads), "s"(a.nsb_inv), "s"(a.steps), "s"(a.group_steps),
               "s"(a.wave_steps), "s"(EPI == SK_PART ? a.last_wave_steps : a.wave_steps), "s"(a.wpr_shift), "s"(a.M), "s"(a.K), "s"(a.x), "s"(a.W), "s"(a.norm_w), "s"(a.pend_splits), "s"(a.norm_w_bf16));
  // Rows in tiles of 16 MB: a block sees its tile as if it were the whole product,
  // through pointers moved to the tile's first row.  The tiles of one set of columns
  // read the same part of W: they get block numbers that are equal modulo 8 (the
  // same XCD, hence the same L2) and follow each other there.
  int col_block = (int)blockIdx.x;
  if (a.tiles > 1) {
    const int xcd = (int)blockIdx.x & 7, j = (int)blockIdx.x >> 3;
    const int jt = (int)__umulhi((unsigned)j, a.tiles_inv), tile = j - jt * a.tiles;
    col_block = jt * 8 + xcd;
    if (col_block >= a.col_blocks) return;      // (the grid is rounded up to whole eights)
    const int m0 = tile * (MB * 16);
    a.M = min(MB * 16, a.M - m0);
    if (NORM && a.x_rows) a.x_rows += m0;       // (the pieces owed are then found by these numbers too)
    else {
      a.x = NORM ? (const void*)((const float*)a.x + (size_t)m0 * a.K)
                 : (const void*)((const T*)a.x + (size_t)m0 * a.K);
      a.pend += (size_t)m0 * a.pend_ld;
    }
    constexpr bool OUT32 = EPI == SK_RESID || EPI == SK_F32 || EPI == SK_PART;
    a.out = OUT32 ? (void*)((float*)a.out + (size_t)m0 * a.ldo) : (void*)((T*)a.out + (size_t)m0 * a.ldo);
    if constexpr (EPI == SK_QKV) {
      a.positions += m0;
      if (a.row_req) a.row_req += m0;
    }
  }
  constexpr int R = sk_ring(MB, STAGE);   // K steps whose loads a wave keeps in flight
  const int nsb = a.nsb, kw = a.kw;
  const int lane = threadIdx.x & 63, nwaves = a.threads >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);     // (what follows from it stays scalar)
  auto by_nsb = [&](int n) { return (n * a.nsb_inv) >> 16; };
  const int ks = by_nsb(wave), strip = wave - ks * nsb;
  const int c = lane & 15, g = lane >> 4;
  const int cols = 16 * nsb;
  // SK_PART: the blocks of one K group follow each other
  const int ksp = (EPI == SK_PART) ? (int)blockIdx.y : 0;
  const int bidx = col_block;
  const int n0 = bidx * cols;
  const int K = a.K, M = a.M;
  const int steps = a.steps;     // bfloat16: W is packed and zero-padded to this; float32: whole steps

  float* part = smem;                                   // [kw*nsb][MB][64][4]
  float* inv = part + (size_t)kw * nsb * MB * 256;      // [MB*16]
  float* s_ssq = inv + MB * 16;                         // [16]: a row's sum of squares, by the waves that share it
  float* s_bias = s_ssq + 16;                           // [cols]
  int* s_pos = (int*)(s_bias + cols);                   // [MB*16]
  int* s_page = s_pos + MB * 16;                        // [MB*16]
  float* s_freq = (float*)(s_page + MB * 16);           // [128]
  T* As = (T*)(smem + sk_float_words(nsb, kw, MB));   // [M][steps * S::LEN + padding]
  const int lda = steps * S::LEN + SK_APAD / (int)sizeof(T);

  // QKV with qsplit > 1: block = (head, p); its two strips are columns p*16.. and
  // d/2 + p*16.. of the head, i.e. both halves of the rotary pairs
  int qhead = 0, qp = 0;
  if constexpr (EPI == SK_QKV) {
    qhead = a.qsplit == 1 ? bidx : (int)__umulhi((unsigned)bidx, a.qsplit_inv);
    qp = bidx - qhead * a.qsplit;
  }
  auto head_col = [&](int col) {   // column of the block -> column of the head
    if (a.qsplit == 1) return col;
    return col < 16 ? qp * 16 + col : (a.d >> 1) + qp * 16 + (col - 16);
  };
  // the strip of 16 weight rows this wave multiplies (past the last one: the last
  // one again, and what comes of it is dropped by the epilogue)
  int wstrip = (EPI == SK_QKV) ? (qhead * a.d + head_col(strip * 16)) >> 4 : bidx * nsb + strip;
  wstrip = min(wstrip, ((a.N + 15) >> 4) - 1);
  constexpr bool PACKED = sizeof(T) == 2;
  // (the address of a step: a scalar part and 32 bits of a lane's own)
  const char* const wstart = (const char*)a.W + (size_t)wstrip * (PACKED ? (size_t)steps * 1024 : (size_t)64 * K);
  const uint32_t wlane = PACKED ? lane * 16 : ((uint32_t)min(c, a.N - 1 - wstrip * 16) * K + g * S::PER) * 4;
  // this block's K steps (all of them, or its group's share), split over its waves
  const int g_begin = ksp * a.group_steps, g_end = min(steps, g_begin + a.group_steps);
  const int portion = EPI == SK_PART && g_begin + a.group_steps > steps ? a.last_wave_steps : a.wave_steps;
  const int s_begin = g_begin + ks * portion;
  const int s_end = min(g_end, s_begin + portion);
  const Frag zero = {};
  const floatx4 fzero = {0.f, 0.f, 0.f, 0.f};

  // ---- What the epilogue needs from global memory is asked for at the start, behind the first rows of x and
  // before the weights, and used at the end: a thread keeps its bias, frequency, position and residual value in
  // registers until the sums are there.  Loads come back in the order they were asked for, so nothing of it
  // may be waited for before the weights are asked for.  All loads are unconditional (indexes clamped,
  // other arrays in the place of absent ones).
  // (a block has at least four threads per column, one per row and one per frequency)
  const int tid = threadIdx.x;
  const bool has_bias = a.bias && ksp == 0;
  uint16_t bias_lo = 0, bias_hi = 0;
  int pos_v = 0, req_v = 0;
  float freq_v = 0.f;
  const bool wants_page = EPI == SK_QKV && a.kcache && qhead >= a.nq;
  // the residual value this thread will add to (its first one), and the first pieces owed to it
  constexpr int RP = EPI != SK_RESID ? 1 : sizeof(T) == 4 ? 4 : 8;
  float resid_old = 0.f, resid_pieces[RP];
  auto ask_for_epilogue = [&] {
    if constexpr (EPI == SK_QKV) {
      const int row = min(tid, M - 1);
      pos_v = a.positions[row];
      req_v = (a.row_req ? a.row_req : a.positions)[row];
      freq_v = (a.inv_freq ? a.inv_freq : (const float*)a.W)[min(tid, (a.d >> 1) - 1)];
    }
    if constexpr (EPI != SK_SWIGLU) {
      const int col = min(tid, cols - 1);
      const int nn = min((EPI == SK_QKV) ? qhead * a.d + head_col(col) : n0 + col, a.N - 1);
      const uint16_t* at = has_bias ? (const uint16_t*)a.bias + (size_t)nn * (a.bias_bf16 ? 1 : 2) : (const uint16_t*)a.W;
      int upper = has_bias && !a.bias_bf16 ? 1 : 0;
      asm volatile("" : "+v"(upper));      // (else two paths, one of which waits for the first load)
      bias_lo = at[0];
      bias_hi = at[upper];
    }
    if constexpr (EPI == SK_RESID) {
      const int m = min(by_nsb(tid >> 4), M - 1), nn = min(n0 + tid - by_nsb(tid >> 4) * cols, a.N - 1);
      resid_old = ((const float*)a.out)[(size_t)m * a.ldo + nn];
      const float* from = a.pend_splits > 0 ? a.pend + (size_t)m * a.pend_ld + nn : (const float*)a.out;
#pragma unroll
      for (int j = 0; j < RP; ++j) resid_pieces[j] = from[max(min(j, a.pend_splits - 1), 0) * a.pend_stride];
    }
  };
  // pages of the rows, once their positions are known; and everything to LDS for the epilogue, before
  // the barrier that the sums wait at
  int page_v = 0;
  auto ask_for_pages = [&] {
    if constexpr (EPI == SK_QKV)
      if (wants_page) page_v = a.table[(size_t)req_v * a.table_stride + pos_v / a.page_size];
  };
  auto leave_for_epilogue = [&] {
    if (tid < cols)
      s_bias[tid] = !has_bias ? 0.f : __uint_as_float(((uint32_t)(a.bias_bf16 ? bias_lo : bias_hi) << 16) |
                                                      (a.bias_bf16 ? 0u : (uint32_t)bias_lo));
    if constexpr (EPI == SK_QKV) {
      if (tid < M) {
        s_pos[tid] = pos_v;
        s_page[tid] = page_v;
      }
      if (tid < (a.d >> 1)) s_freq[tid] = a.inv_freq ? freq_v : 0.f;
    }
  };

  floatx4 acc[MB][S::SUMS];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int i = 0; i < S::SUMS; ++i) acc[mb][i] = fzero;

  // Loads in the ring are unconditional (a step past the end reads the last tile
  // again and is multiplied by zeros): a load under a branch makes the compiler wait
  // for every load in flight at the join, and the stream stalls once per round.
  const int s_last = max(0, min(s_end, steps) - 1);      // (a wave past the end: any step that is there)
  auto wload = [&](int st) {
    return *(const Frag*)(wstart + (wlane + (uint32_t)min(st, s_last) * (PACKED ? 1024u : 64u)));
  };
  Frag b[R];

  if constexpr (STAGE) {
    // ---- Stage the rows of x.  Their first loads go out before those of the weights, which follow at
    // once: loads come back in the order they were asked for, so a wave that asked for its
    // weights first staged its rows only when its whole ring was there (gate/up of one row of the 0.5B shape:
    // 2.0 us from the first load to the barrier).
    // Fewer rows than waves: `wpr` waves share a row, each taking every wpr-th run of 64
    // chunks (one wave alone would walk a long row in many trips while the others wait)
    const int chunks = K >> 3, chunks_pad = steps * (S::LEN / 8);
    const int wpr_shift = a.wpr_shift, wpr = 1 << wpr_shift;
    // A wave walks its part of a row U chunks at a time: the loads of all U (the row, the
    // norm's weight, the first four pieces owed) are on their way before the first is used, so a part
    // costs one trip to memory per U chunks and not one per chunk.  Loads are unconditional
    // (a chunk past the end reads the last one again and is not stored).
    auto stage_rows = [&](auto u_tag, auto w_tag, auto pieces_tag) {
      constexpr int U = decltype(u_tag)::value;
      constexpr bool W_BF16 = decltype(w_tag)::value;     // (the norm's weight: no branch among the loads)
      constexpr bool PIECES = decltype(pieces_tag)::value;
      const int stride = 64 * wpr, units = M * wpr;
      floatx4 p[U], q[U], w0[U], w1[U], pp[U][4], qq[U][4];
      bf16x8 w8[U];
      Sk8<T> v[U];
      size_t row = 0;
      auto start_row = [&](int unit) {
        const int r = unit >> wpr_shift;
        row = NORM && a.x_rows ? a.x_rows[r] : r;
      };
      auto load_pieces = [&](int base, int sp0) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const float* src = a.pend + min(sp0 + j, a.pend_splits - 1) * a.pend_stride + row * a.pend_ld +
                               min(base + u * stride + lane, chunks - 1) * 8;
            pp[u][j] = *(const floatx4*)src;
            qq[u][j] = *(const floatx4*)(src + 4);
          }
      };
      auto load = [&](int base) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int ch = min(base + u * stride + lane, chunks - 1);
          if constexpr (NORM) {
            const float* src = (const float*)a.x + row * K + ch * 8;
            p[u] = *(const floatx4*)src;
            q[u] = *(const floatx4*)(src + 4);
            if constexpr (W_BF16) {
              w8[u] = *(const bf16x8*)((const bf16_t*)a.norm_w + ch * 8);
            } else {
              w0[u] = *(const floatx4*)((const float*)a.norm_w + ch * 8);
              w1[u] = *(const floatx4*)((const float*)a.norm_w + ch * 8 + 4);
            }
          } else {
            v[u].load((const T*)a.x + row * K + ch * 8);
          }
        }
        if constexpr (PIECES) load_pieces(base, 0);
      };
      // (n: how many chunks of its part a lane has behind it.  The first of every four chunks without pieces rounds the
      // squares of its lower four numbers by themselves, all others those of their upper four, whatever U is; a part taken
      // one by one without pieces is one chunk)
      auto store = [&](int base, T* dst, float& ssq, int n) {
        if constexpr (PIECES) {
          for (int sp0 = 0; sp0 < a.pend_splits; sp0 += 4) {      // in their order
            if (sp0 > 0) load_pieces(base, sp0);
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
              for (int j = 0; j < 4; ++j) {
                const float on = sp0 + j < a.pend_splits ? 1.f : 0.f;
                p[u] += pp[u][j] * on;
                q[u] += qq[u][j] * on;
              }
          }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int ch = base + u * stride + lane;
          if (ch >= chunks) break;
          if constexpr (NORM) {
            float wv[8];
            if constexpr (W_BF16) {
#pragma unroll
              for (int j = 0; j < 8; ++j) wv[j] = (float)w8[u][j];
            } else {
#pragma unroll
              for (int j = 0; j < 4; ++j) {
                wv[j] = w0[u][j];
                wv[4 + j] = w1[u][j];
              }
            }
            Sk8<T> av;
            const bool p_alone = !PIECES && u == 0 && (U != 2 || (n & 2) == 0);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              ssq = p_alone ? sk_add_squares(ssq, q[u][j], p[u][j]) : sk_add_squares(ssq, p[u][j], q[u][j]);
              av.set(j, p[u][j] * wv[j]);
              av.set(4 + j, q[u][j] * wv[4 + j]);
            }
            av.store(dst + ch * 8);
          } else {
            v[u].store(dst + ch * 8);
          }
        }
      };
      // (a wave without a part of its own asks for the last one's again and stores nothing)
      int unit = min(wave, units - 1);
      start_row(unit);
      load((unit & (wpr - 1)) * 64);
      __builtin_amdgcn_sched_barrier(0);
      ask_for_epilogue();
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < R; ++u) b[u] = wload(s_begin + u);
      __builtin_amdgcn_sched_barrier(0);
      if (wave >= units) return;
      float ssq = 0.f;
      int base = (unit & (wpr - 1)) * 64;
      T* dst = As + (size_t)(unit >> wpr_shift) * lda;
      store(base, dst, ssq, 0);      // (by itself: in the loop below the loads of W behind these would be waited for, too)
      for (int n = U;; n = 0) {
        for (base += U * stride; base < chunks; base += U * stride, n += U) {
          load(base);
          store(base, dst, ssq, n);
        }
        if constexpr (NORM) {
          ssq = full_wave_sum(ssq);
          if (lane == 0) {
            if (wpr == 1) inv[unit] = rsqrtf(ssq / (float)K + a.eps);
            else s_ssq[unit] = ssq;       // (M * wpr <= 16 waves)
          }
        }
        if ((unit & (wpr - 1)) == 0)
          for (int ch = chunks + lane; ch < chunks_pad; ch += 64) Sk8<T>{}.store(dst + ch * 8);
        unit += nwaves;
        if (unit >= units) return;
        start_row(unit);
        ssq = 0.f;
        dst = As + (size_t)(unit >> wpr_shift) * lda;
        base = (unit & (wpr - 1)) * 64 - U * stride;
      }
    };
    // (with pieces owed, a chunk's loads are as many registers as three without; with a float32 weight as
    // many as two; a part of one run of chunks asks for no more)
    using one = std::integral_constant<int, 1>;
    using two = std::integral_constant<int, 2>;
    using four = std::integral_constant<int, 4>;
    if constexpr (NORM) {
      if (a.pend_splits > 0) {
        if (a.norm_w_bf16) stage_rows(one{}, std::true_type{}, std::true_type{});
        else stage_rows(one{}, std::false_type{}, std::true_type{});
      } else if (!a.norm_w_bf16) {
        stage_rows(two{}, std::false_type{}, std::false_type{});
      } else if (chunks <= 64 * wpr) {
        stage_rows(one{}, std::true_type{}, std::false_type{});
      } else {
        stage_rows(four{}, std::true_type{}, std::false_type{});
      }
    } else {
      stage_rows(four{}, std::true_type{}, std::false_type{});
    }
    ask_for_pages();
    __syncthreads();
    if constexpr (NORM) {
      // the parts of a row in their order (read by the epilogue, behind the next barrier)
      if (wpr > 1 && (int)threadIdx.x < M) {
        float total = 0.f;
        for (int sub = 0; sub < wpr; ++sub) total += s_ssq[threadIdx.x * wpr + sub];
        inv[threadIdx.x] = rsqrtf(total / (float)K + a.eps);
      }
    }
    // rows past M are not staged: their lanes read the last row, and what they
    // compute lands in rows of the result that nobody reads
    const T* arow[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) arow[mb] = As + (size_t)min(mb * 16 + c, M - 1) * lda + g * S::PER;
    int s0 = s_begin;
    for (; s0 + R < s_end; s0 += R) {       // rounds that refill the ring
#pragma unroll
      for (int u = 0; u < R; ++u) {
        const int st = s0 + u;
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
          const Frag av = *(const Frag*)(arow[mb] + st * S::LEN);
          S::mul(av, b[u], acc[mb], u);
        }
        b[u] = wload(st + R);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int u = 0; u < R; ++u) {           // the last round drains it
      const int st = s0 + u;
      const Frag bu = st < s_end ? b[u] : zero;
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        Frag av = *(const Frag*)(arow[mb] + min(st, steps - 1) * S::LEN);
        if constexpr (S::KEEPS_INF) av = st < s_end ? av : zero;
        S::mul(av, bu, acc[mb], u);
      }
    }
  } else {
    // ---- rows of x (compute type) straight from global memory, in the same ring; a
    // piece past K or a row past M reads a valid piece instead: it meets zeros of
    // the padded W, or lands in a row of the result that nobody reads
    const T* xb[MB];
    const T* x_rows = (const T*)a.x;
    if constexpr (EPI == SK_PART) {
      if (a.segs > 1) {
        int seg = 0;
#pragma unroll
        for (int i = 0; i < 7; ++i) seg += (i + 1 < a.segs && wstrip >= a.seg_end[i]) ? 1 : 0;
        x_rows += seg * a.seg_stride;
      }
    }
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) xb[mb] = x_rows + (size_t)min(mb * 16 + c, M - 1) * K;
    auto xload = [&](int st, int mb) {
      return *(const Frag*)(xb[mb] + min(st * S::LEN + g * S::PER, K - S::PER));
    };
    Frag ab[R][MB];
    ask_for_epilogue();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < R; ++u) {     // in the order in which the loop below refills the ring
      const int st = min(s_begin + u, s_last);
      b[u] = wload(st);
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) ab[u][mb] = xload(st, mb);
      __builtin_amdgcn_sched_barrier(0);
    }
    ask_for_pages();
    int s0 = s_begin;
    for (; s0 + R < s_end; s0 += R) {       // rounds that refill the ring
#pragma unroll
      for (int u = 0; u < R; ++u) {
        const int st = s0 + u;
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
          S::mul(ab[u][mb], b[u], acc[mb], u);
        const int nx = min(st + R, s_last);
        b[u] = wload(nx);
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) ab[u][mb] = xload(nx, mb);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int u = 0; u < R; ++u) {           // the last round drains it
      const Frag bu = s0 + u < s_end ? b[u] : zero;
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        Frag av = ab[u][mb];
        if constexpr (S::KEEPS_INF) av = s0 + u < s_end ? av : zero;
        S::mul(av, bu, acc[mb], u);
      }
    }
  }

  // ---- partial sums to LDS
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
#pragma unroll
    for (int half = S::SUMS / 2; half > 0; half >>= 1)
#pragma unroll
      for (int i = 0; i < half; ++i) acc[mb][i] += acc[mb][half + i];
    *(floatx4*)(part + (((size_t)wave * MB + mb) * 64 + lane) * 4) = acc[mb][0];
  }
  leave_for_epilogue();
  __syncthreads();
  // ---- reduce over the K slices in a fixed order (four of them read at a time); epilogue
  auto total = [&](int m, int col) {
    const float* from = part + (((size_t)(col >> 4) * MB + (m >> 4)) * 64 + ((m & 15) >> 2) * 16 + (col & 15)) * 4 + (m & 3);
    const int stride = nsb * MB * 256;
    float sum = 0.f;
    for (int k2 = 0; k2 < kw; k2 += 4) {
      float v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = from[min(k2 + j, kw - 1) * stride];
#pragma unroll
      for (int j = 0; j < 4; ++j) sum += k2 + j < kw ? v[j] : 0.f;
    }
    if constexpr (NORM) sum *= inv[m];
    return sum + s_bias[col];
  };
  if constexpr (EPI == SK_SWIGLU) {
    const int half = cols >> 1;   // outputs of this block: a thread takes a gate column and its up column
    for (int idx = tid; idx < M * half; idx += a.threads) {
      const int m = by_nsb(idx >> 3), j = idx - m * half;
      const int pr = j >> 4, cc = j & 15;
      const float gv = total(m, pr * 32 + cc), uv = total(m, pr * 32 + 16 + cc);
      const int o = ((n0 >> 5) + pr) * 16 + cc;
      if (o < a.n_out) ((T*)a.out)[(size_t)m * a.ldo + o] = from_float<T>(sk_pair<T>(gv, uv, a));
    }
  } else if constexpr (EPI == SK_QKV) {
    // this block is (part of) head `qhead` of [q heads | k heads | v heads]; the low halves of
    // its rotary pairs are the first half of its columns, and a thread takes both of a pair
    const int head = qhead, d = a.d, dhalf = d >> 1, half = cols >> 1;
    const int i0 = a.qsplit == 1 ? 0 : qp * 16;
    const bool is_q = head < a.nq, is_k = !is_q && head < a.nq + a.nkv;
    for (int idx = tid; idx < M * half; idx += a.threads) {
      const int m = by_nsb(idx >> 3), il = idx - m * half;
      const int i = i0 + il;                      // pair index within the head
      float lo = total(m, il), hi = total(m, il + half);
      const int pos = s_pos[m];
      if ((is_q || is_k) && a.inv_freq) {
        float s, co;
        if constexpr (sizeof(T) == 4) {
          sincosf((float)pos * s_freq[i], &s, &co);
        } else {
          // bfloat16 results: the hardware sine and cosine of r = frac(angle / 2 pi)
          float r = (float)pos * s_freq[i] * 0.15915494309189535f;
          r -= floorf(r);
          s = __builtin_amdgcn_sinf(r);
          co = __builtin_amdgcn_cosf(r);
        }
        const float nlo = lo * co - hi * s, nhi = hi * co + lo * s;
        lo = nlo;
        hi = nhi;
      }
      if (is_q) {
        T* dst = (T*)a.out + (size_t)m * a.ldo + (size_t)head * d;
        dst[i] = from_float<T>(lo);
        dst[i + dhalf] = from_float<T>(hi);
      } else if (a.kcache) {
        const size_t page = (size_t)s_page[m];
        const int off = pos % a.page_size;
        if (is_k) {
          T* dst = (T*)a.kcache + (page * a.nkv + (head - a.nq)) * (size_t)a.page_size * d;
          dst[kcache_index(off, i, d)] = from_float<T>(lo);
          dst[kcache_index(off, i + dhalf, d)] = from_float<T>(hi);
        } else {
          T* dst = (T*)a.vcache + (page * a.nkv + (head - a.nq - a.nkv)) * (size_t)a.page_size * d;
          dst[vcache_index(off, i, d)] = from_float<T>(lo);
          dst[vcache_index(off, i + dhalf, d)] = from_float<T>(hi);
        }
      }
    }
  } else {
    for (int idx = tid; idx < M * cols; idx += a.threads) {
      const int m = by_nsb(idx >> 4), col = idx - m * cols, nn = n0 + col;
      const float sum = total(m, col);
      if (nn >= a.N) continue;
      const size_t at = (size_t)m * a.ldo + nn;
      if constexpr (EPI == SK_STORE) {
        ((T*)a.out)[at] = from_float<T>(a.act ? fmaxf(sum, 0.f) * fmaxf(sum, 0.f) : sum);
      } else if constexpr (EPI == SK_RESID) {
        const bool first = idx == tid;
        const float* from = a.pend + (size_t)m * a.pend_ld + nn;
        float old = first ? resid_old : ((float*)a.out)[at];
        if (first) {
#pragma unroll
          for (int j = 0; j < RP; ++j) old += j < a.pend_splits ? resid_pieces[j] : 0.f;
        }
        for (int sp = first ? RP : 0; sp < a.pend_splits; ++sp) old += from[sp * a.pend_stride];
        ((float*)a.out)[at] = old + sum;
      } else if constexpr (EPI == SK_PART) {
        ((float*)a.out)[ksp * a.part_stride + at] = sum;
      } else {
        ((float*)a.out)[at] = sum;
      }
    }
  }
}

// ---------------------------------------------------------------- dispatch
// (`width`: bytes of a number of W and of the staged rows, 2 or 4)
static size_t skinny_lds_bytes(int nsb, int kw, int mb, int M, int K, bool stage, int width) {
  size_t bytes = sk_float_words(nsb, kw, mb) * sizeof(float);
  if (stage) bytes += (size_t)M * ((size_t)(K + 31) / 32 * 32 * width + SK_APAD);
  return bytes;
}

// Most LDS a block may take (a compute unit of gfx950 has 160 KB).
static const size_t SK_LDS_LIMIT = 152 * 1024;
// Most rows of a call (tiles of at most 64 rows, a block each per set of columns).
constexpr int SK_MAX_ROWS = 1024;

template <typename T, int MB, int EPI, bool NORM, bool STAGE>
static int skinny_launch(const SkinnyArgs& a, int blocks, size_t lds, hipStream_t stream) {
  auto kernel = skinny_block_kernel<T, MB, EPI, NORM, STAGE>;
  if (lds > 48 * 1024) {
    static size_t raised = 0;     // per instantiation
    if (lds > raised) {
      if (hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)SK_LDS_LIMIT) != hipSuccess) {
        llmlab_set_error("skinny_linear: cannot raise the LDS limit to %zu bytes", SK_LDS_LIMIT);
        return 3;
      }
      raised = SK_LDS_LIMIT;
    }
  }
  const int grid = a.tiles > 1 ? (blocks + 7) / 8 * 8 * a.tiles : blocks;
  hipLaunchKernelGGL(kernel, dim3(grid, EPI == SK_PART ? a.ksplit : 1), dim3(64 * a.nsb * a.kw), lds, stream, a);
  return 0;
}

template <int EPI, bool NORM, bool STAGE>
static int skinny_launch_mb(const SkinnyArgs& a, int width, int mb, int blocks, size_t lds, hipStream_t stream) {
  if (width == 4) return skinny_launch<float, 1, EPI, NORM, STAGE>(a, blocks, lds, stream);     // (tiles of 16 rows only)
  if (mb == 1) return skinny_launch<bf16_t, 1, EPI, NORM, STAGE>(a, blocks, lds, stream);
  if (mb == 2) return skinny_launch<bf16_t, 2, EPI, NORM, STAGE>(a, blocks, lds, stream);
  return skinny_launch<bf16_t, 4, EPI, NORM, STAGE>(a, blocks, lds, stream);
}

template <int EPI, bool NORM>
static int skinny_launch_stage(const SkinnyArgs& a, int width, bool stage, int mb, int blocks, size_t lds,
                               hipStream_t stream) {
  if constexpr (NORM) {
    return skinny_launch_mb<EPI, true, true>(a, width, mb, blocks, lds, stream);   // the norm is staged always
  } else {
    if (stage) return skinny_launch_mb<EPI, false, true>(a, width, mb, blocks, lds, stream);
    return skinny_launch_mb<EPI, false, false>(a, width, mb, blocks, lds, stream);
  }
}

// Debug interface (kernels/debug.py): a block shape can be forced, for tests and
// measurements (0 = choose).
static int g_force_nsb = 0, g_force_kw = 0, g_force_stage = -1, g_force_mb = 0, g_force_epi = -1;
extern "C" void llmlab_debug_skinny_shape(int nsb, int kw, int stage, int mb) {
  g_force_nsb = nsb;
  g_force_kw = kw;
  g_force_stage = stage;
  g_force_mb = mb;
}
// ... for one epilogue only (-1: for all)
extern "C" void llmlab_debug_skinny_epilogue(int epilogue) { g_force_epi = epilogue; }

struct SkinnyShape {
  int nsb, kw;
  bool stage;
  int qsplit;
  int mb;       // row blocks of 16 per tile of rows (1, 2 or 4); tiles = ceil(M / 16 mb)
};

static inline int sk_tiles(int M, int mb) { return (M + 16 * mb - 1) / (16 * mb); }

// Pick strips per block, K slices per strip and staging by an estimate of the
// kernel's time: a fixed part, plus what the busiest compute unit needs to stream
// its share of W and of x (a unit sustains far less than 1/256 of the chip's
// bandwidth would suggest, so spreading the matrix over all units matters most),
// or the memory round trips of a wave if those take longer.
static SkinnyShape skinny_choose_tile(int epilogue, bool norm, int mb, int M, int tiles, int N, int K, int d,
                                      int num_cus, int ksplit, int width, double* cost_out) {
  const int steps = ((K + 31) / 32 + ksplit - 1) / ksplit * (width / 2);     // per K group of blocks
  const int strips = (N + 15) / 16;
  const int max_waves = mb >= 4 ? 8 : 16;
  SkinnyShape best{0, 0, false, 1, mb};
  double best_cost = 1e30;
  int cand[5], ncand = 0;
  if (epilogue == SK_QKV) {
    cand[ncand++] = d / 16;                   // a block per head
    if (d % 32 == 0 && d > 32) cand[ncand++] = 2;   // or d/32 blocks per head, two strips each
  } else {
    for (int nsb = (epilogue == SK_SWIGLU ? 2 : 1); nsb <= 16; nsb *= 2) cand[ncand++] = nsb;
  }
  for (int ci = 0; ci < ncand; ++ci) {
    const int nsb = cand[ci];
    if (nsb > max_waves) continue;
    for (int kw = 1; kw * nsb <= max_waves && kw <= steps; ++kw) {
      for (int st = norm ? 1 : 0; st < (epilogue == SK_PART ? 1 : 2); ++st) {     // pieces of K: no staging
        const bool stage = st == 1;
        const size_t lds = skinny_lds_bytes(nsb, kw, mb, M, K, stage, width);
        if (lds > SK_LDS_LIMIT) continue;
        const int blocks = (strips + nsb - 1) / nsb * ksplit * tiles;     // (for QKV: heads, or heads * d/32)
        const int per_cu = (blocks + num_cus - 1) / num_cus;       // blocks the busiest unit runs
        int resident = 16 / (nsb * kw);                             // of which so many at a time
        if (resident > per_cu) resident = per_cu;
        // (as many as LDS would hold with a block's results there, as where this was fitted; by what is left without
        // them gate/up of 16 rows of the 1.5B shape takes 2 strips x 2 slices, 21.7 us, and not 8 x 1, 16.6, of 5 of the
        // 7B shape 2 x 2, 57, and not 2 x 4, 52)
        const size_t results = epilogue == SK_SWIGLU || epilogue == SK_QKV ? (size_t)M * 16 * nsb * sizeof(float) : 0;
        const int by_lds = (int)((160 * 1024) / (lds + results > 1024 ? lds + results : 1024));
        if (resident > by_lds) resident = by_lds;
        if (resident < 1) resident = 1;
        const int rounds = (per_cu + resident - 1) / resident;
        // a compute unit streams about 50 GB/s from HBM (a good 3 GB/s per resident wave
        // until that limit) and more from the caches; rows of x read by every wave on its own
        // (not staged) come in short strided pieces and cost about twice that
        // (fitted twice: a large matrix is bound by what the waves of a unit keep in
        // flight, up to about 50 GB/s; a small one by latencies, which the lower figures
        // stand for)
        const bool large = (double)N * K * width >= 64e6;
        double rate = (large ? 3.2e3 : 3.5e3) * resident * nsb * kw;
        // (more than one tile of rows of a wide output: all but the first tile of a set of
        // columns find W in the L2 of their die, and sixteen waves a block draw what eight
        // cannot: gate/up of the 0.5B shape at 48 rows, 10.5 us with 8 strips x 2 slices, 14.3
        // with 4 x 2; a narrow output gains nothing from more slices)
        const double cap = (large || (tiles > 1 && strips >= num_cus)) ? 50.0e3 : 25.0e3;
        if (rate > cap) rate = cap;
        const double t_stream = per_cu * (16.0 * nsb * K * width) / rate;
        const double x_bytes = (double)(stage ? 1 : 2 * nsb) * M * K * (norm ? 4.0 : width);
        const double t_x = per_cu * x_bytes / 50.0e3;
        const int per = (steps + kw - 1) / kw;
        const int u = sk_ring(mb, stage);
        const double trips = stage ? 1.0 + 0.3 * ((per + u - 1) / u - 1) : (double)((per + u - 1) / u);
        const double busy = t_stream + t_x > 0.8 * trips ? t_stream + t_x : 0.8 * trips;
        // a fixed part per kernel, and again (in part hidden by the neighbours) for every
        // further round of blocks on the busiest unit
        const double cost = 3.3 + (stage ? 0.3 : 0.0) + busy + (rounds - 1) * 2.4 / resident +
                            0.03 * kw * nsb;
        if (cost < best_cost) {
          best_cost = cost;
          best = SkinnyShape{nsb, kw, stage, (epilogue == SK_QKV && nsb != d / 16) ? d / 32 : 1, mb};
        }
      }
    }
  }
  *cost_out = best_cost;
  return best;
}

// The rows may be cut into tiles of 16, 32 or 64 as well: smaller tiles give more
// blocks, each of which stages (and norms) fewer rows, and W is read once per tile
// (from the cache after the first).
static SkinnyShape skinny_choose(int epilogue, bool norm, int M, int N, int K, int d, int num_cus,
                                 int ksplit = 1, int width = 2) {
  SkinnyShape best{0, 0, false, 1, 1};
  double best_cost = 1e30;
  // (q/k/v of more than 64 rows: tiles of 16 rows, measured; 576 rows of 1152 x 896 take
  // 13.4 us so, 16.4 in tiles of 32 and 26 in tiles of 64)
  const int mb_max = width == 4 || M <= 16 || (epilogue == SK_QKV && M > 64) ? 1 : (M <= 32 ? 2 : 4);
  for (int mb = mb_max; mb >= 1; mb >>= 1) {
    if (g_force_mb > 0 && (g_force_epi < 0 || g_force_epi == epilogue) && mb != g_force_mb &&
        !(g_force_mb > mb_max && mb == mb_max))
      continue;
    const int tiles = sk_tiles(M, mb);
    double cost;
    const SkinnyShape s = skinny_choose_tile(epilogue, norm, mb, M < 16 * mb ? M : 16 * mb, tiles, N, K, d,
                                             num_cus, ksplit, width, &cost);
    if (s.nsb > 0 && cost < best_cost) {
      best_cost = cost;
      best = s;
    }
  }
  return best;
}

// The shape the chooser takes for a product (for tests and tuning): out = {nsb, kw, stage, qsplit, mb}.
extern "C" void llmlab_skinny_shape(int epilogue, int norm, int M, int N, int K, int d, int num_cus, int ksplit,
                                    int* out) {
  const SkinnyShape s = skinny_choose(epilogue, norm != 0, M, N, K, d, num_cus, ksplit < 1 ? 1 : ksplit);
  out[0] = s.nsb; out[1] = s.kw; out[2] = s.stage; out[3] = s.qsplit; out[4] = s.mb;
}

// One entry point for the whole family.
//   norm != 0: x is the float32 residual stream (rows x_rows[m] or m), norm_w/eps its RMSNorm
//   epilogue SK_QKV: N = (nq + 2 nkv) * d, one block per head, `out` is q [M, ldo]
//   epilogue SK_PART: K is split over `ksplit` groups of blocks, `out` is float32
//     [ksplit][M][ldo] (part_stride numbers from one piece to the next); nothing is added up
//   pend / pend_splits / pend_ld / pend_stride: pieces that a former SK_PART call left and
//     that belong to the rows of x (norm != 0: added while the rows are read) or to the
//     rows of out (SK_RESID: added with the product, which folds them into the stream)
//   segs > 1 (SK_PART): the strips of 16 rows of W below seg_ends[0] multiply x, the ones from there to
//     below seg_ends[1] x + seg_stride, and so on (seg_ends: segs - 1 numbers in host memory)
extern "C" int llmlab_skinny_linear(const void* x, int norm, const int* x_rows, const void* norm_w,
                                    int norm_w_dtype, float eps, const void* w, int dtype, const void* bias,
                                    int bias_dtype, int epilogue, void* out, int M, int N, int K,
                                    int ldo, int n_out, const float* inv_freq, const int* positions,
                                    const int* row_req, const int* table, int table_stride,
                                    int page_size, void* kcache, void* vcache, int nq, int nkv, int d,
                                    int num_cus, const float* pend, int pend_splits, int pend_ld,
                                    size_t pend_stride, int ksplit, size_t part_stride, int segs,
                                    const int* seg_ends, size_t seg_stride, float limit, float slope,
                                    float shift, hipStream_t stream) {
  LLMLAB_REQUIRE(segs <= 1 || (segs <= 8 && seg_ends && epilogue == SK_PART && seg_stride % 8 == 0),
                 "skinny_linear: up to 8 segments with inputs of their own, in pieces, got %d", segs);
  LLMLAB_REQUIRE(M >= 0 && M <= SK_MAX_ROWS, "skinny_linear: takes at most %d rows, got %d", SK_MAX_ROWS, M);
  LLMLAB_REQUIRE(N > 0 && K > 0 && K % (dtype == DT_F32 ? 16 : 8) == 0,
                 "skinny_linear: bad sizes N=%d K=%d (K must be a multiple of 8, in float32 of 16)", N, K);
  const int width = dtype == DT_F32 ? 4 : 2;
  // (6 at this interface: STORE through the squared relu; 7: the paired product with a gelu gate;
  // 8: the clamped pair)
  const int act = epilogue == 6 ? 1 : epilogue == 7 ? 2 : epilogue == 8 ? 3 : 0;
  if (act == 1) epilogue = SK_STORE;
  if (act > 1) epilogue = SK_SWIGLU;
  LLMLAB_REQUIRE(epilogue >= 0 && epilogue <= 5, "skinny_linear: unknown epilogue %d", epilogue);
  LLMLAB_REQUIRE(pend_splits >= 0 && (pend_splits == 0 || (pend != nullptr && (norm || epilogue == SK_RESID))),
                 "skinny_linear: pending sums go with a norm or into the residual");
  LLMLAB_REQUIRE(pend_splits == 0 || !norm ||
                 (pend_ld % 4 == 0 && (uintptr_t)pend % 16 == 0 && pend_stride % 4 == 0),
                 "skinny_linear: pending sums under a norm are read 16 bytes at a time: not aligned");
  if (epilogue != SK_PART) ksplit = 1;
  LLMLAB_REQUIRE(ksplit >= 1 && ksplit <= 16 && (epilogue != SK_PART || (!norm && part_stride >= (size_t)M * ldo)),
                 "skinny_linear(pieces): bad split %d", ksplit);
  LLMLAB_REQUIRE(((uintptr_t)x % 16 == 0) && ((uintptr_t)w % 16 == 0) &&
                 (norm_w == nullptr || (uintptr_t)norm_w % 16 == 0),
                 "skinny_linear: operands must be 16-byte aligned");
  LLMLAB_REQUIRE(!norm || norm_w != nullptr, "skinny_linear: a norm needs its weight");
  if (M == 0) return 0;
  if (num_cus <= 0) num_cus = 256;
  if (epilogue == SK_QKV) {
    LLMLAB_REQUIRE(d >= 16 && d % 16 == 0 && d <= 256 && N == (nq + 2 * nkv) * d,
                   "skinny_linear(qkv): head size %d / %d rows do not fit", d, N);
    LLMLAB_REQUIRE((kcache == nullptr) == (vcache == nullptr), "skinny_linear(qkv): both caches or none");
    LLMLAB_REQUIRE(positions != nullptr && (kcache == nullptr || (table && row_req && page_size > 0)),
                   "skinny_linear(qkv): positions and block table are needed");
  } else if (epilogue == SK_SWIGLU) {
    LLMLAB_REQUIRE(N % 32 == 0 && 2 * ((n_out + 15) / 16 * 16) == N && bias == nullptr,
                   "skinny_linear(swiglu): %d rows do not interleave %d outputs", N, n_out);
  } else {
    LLMLAB_REQUIRE(n_out == N, "skinny_linear: n_out %d != N %d", n_out, N);
  }
  LLMLAB_REQUIRE(ldo >= (epilogue == SK_QKV ? nq * d : n_out), "skinny_linear: output stride too small");
  SkinnyShape shape = skinny_choose(epilogue, norm != 0, M, N, K, d, num_cus, ksplit, width);
  const int mb = shape.mb, tiles = sk_tiles(M, mb), tile_rows = M < 16 * mb ? M : 16 * mb;
  const bool forced = g_force_epi < 0 || g_force_epi == epilogue;
  if (forced && g_force_nsb > 0 && epilogue != SK_QKV) shape.nsb = g_force_nsb;
  if (forced && g_force_nsb > 0 && epilogue == SK_QKV && d % 32 == 0 && d > 32) {
    shape.nsb = g_force_nsb == 2 ? 2 : d / 16;
    shape.qsplit = g_force_nsb == 2 ? d / 32 : 1;
  }
  if (forced && g_force_kw > 0) shape.kw = g_force_kw;
  if (forced && g_force_stage >= 0) shape.stage = norm || (g_force_stage != 0 && epilogue != SK_PART);
  LLMLAB_REQUIRE(shape.nsb > 0 && shape.kw > 0,
                 "skinny_linear: no block shape fits N=%d K=%d M=%d (16 rows of x to stage: %zu bytes of LDS)",
                 N, K, M, (size_t)(M < 16 ? M : 16) * ((size_t)(K + 31) / 32 * 32 * width + SK_APAD));
  const size_t lds = skinny_lds_bytes(shape.nsb, shape.kw, mb, tile_rows, K, shape.stage, width);
  LLMLAB_REQUIRE(lds <= SK_LDS_LIMIT && shape.nsb * shape.kw <= (mb >= 4 ? 8 : 16),
                 "skinny_linear: block shape %dx%d does not fit", shape.nsb, shape.kw);
  // (only a forced shape can fail these: a gate strip and its up strip share a block, and
  // every K slice has a step)
  LLMLAB_REQUIRE(!(epilogue == SK_SWIGLU && shape.nsb % 2 != 0) &&
                     shape.kw <= ((K + 31) / 32 + ksplit - 1) / ksplit * (width / 2),
                 "skinny_linear: block shape %dx%d does not fit this product", shape.nsb, shape.kw);
  const int blocks = (N + 16 * shape.nsb - 1) / (16 * shape.nsb);
  SkinnyArgs a;
  a.pend = pend; a.pend_splits = pend_splits; a.pend_ld = pend_ld; a.pend_stride = pend_stride;
  a.segs = segs;
  for (int i = 0; i < 7; ++i) a.seg_end[i] = i + 1 < segs ? seg_ends[i] : 0;
  a.seg_stride = seg_stride;
  a.ksplit = ksplit; a.part_stride = part_stride; a.tiles = tiles; a.col_blocks = blocks;
  a.qsplit = shape.qsplit;
  auto inverse = [](int n) { return n > 1 ? (unsigned)(((1ull << 32) + n - 1) / n) : 0u; };
  a.tiles_inv = inverse(tiles);
  a.qsplit_inv = inverse(shape.qsplit);
  a.steps = (K + 64 / width - 1) / (64 / width);       // (64 bytes of a row a step)
  a.group_steps = (a.steps + ksplit - 1) / ksplit;
  a.wave_steps = (a.group_steps + shape.kw - 1) / shape.kw;
  a.last_wave_steps = (a.steps % a.group_steps + shape.kw - 1) / shape.kw;
  a.wpr_shift = 0;
  while ((2 << a.wpr_shift) * tile_rows <= shape.nsb * shape.kw) ++a.wpr_shift;
  a.act = act;
  a.limit = limit; a.slope = slope; a.shift = shift;
  a.x = x; a.x_rows = x_rows; a.norm_w = norm_w; a.W = w; a.bias = bias; a.out = out;
  a.inv_freq = inv_freq; a.positions = positions; a.row_req = row_req; a.table = table;
  a.kcache = kcache; a.vcache = vcache;
  a.M = M; a.N = N; a.K = K; a.ldo = ldo; a.n_out = n_out;
  a.norm_w_bf16 = norm_w_dtype == DT_BF16; a.bias_bf16 = bias_dtype == DT_BF16;
  a.nsb = shape.nsb; a.kw = shape.kw; a.threads = 64 * shape.nsb * shape.kw; a.nsb_inv = (65536 + shape.nsb - 1) / shape.nsb; a.nq = nq; a.nkv = nkv; a.d = d; a.table_stride = table_stride;
  a.page_size = page_size; a.eps = eps;
  int rc = 0;
  if (norm) {
    switch (epilogue) {
      case SK_F32: rc = skinny_launch_stage<SK_F32, true>(a, width, shape.stage, mb, blocks, lds, stream); break;
      case SK_SWIGLU: rc = skinny_launch_stage<SK_SWIGLU, true>(a, width, shape.stage, mb, blocks, lds, stream); break;
      case SK_QKV: rc = skinny_launch_stage<SK_QKV, true>(a, width, shape.stage, mb, blocks, lds, stream); break;
      default: LLMLAB_REQUIRE(false, "skinny_linear: epilogue %d has no fused norm", epilogue);
    }
  } else {
    switch (epilogue) {
      case SK_STORE: rc = skinny_launch_stage<SK_STORE, false>(a, width, shape.stage, mb, blocks, lds, stream); break;
      case SK_RESID: rc = skinny_launch_stage<SK_RESID, false>(a, width, shape.stage, mb, blocks, lds, stream); break;
      case SK_F32: rc = skinny_launch_stage<SK_F32, false>(a, width, shape.stage, mb, blocks, lds, stream); break;
      case SK_SWIGLU: rc = skinny_launch_stage<SK_SWIGLU, false>(a, width, shape.stage, mb, blocks, lds, stream); break;
      case SK_QKV: rc = skinny_launch_stage<SK_QKV, false>(a, width, shape.stage, mb, blocks, lds, stream); break;
      case SK_PART: rc = skinny_launch_stage<SK_PART, false>(a, width, false, mb, blocks, lds, stream); break;
      default: LLMLAB_REQUIRE(false, "skinny_linear: epilogue %d needs the norm", epilogue);
    }
  }
  if (rc) return rc;
  LLMLAB_LAUNCH_CHECK("skinny_linear");
  return 0;
}
