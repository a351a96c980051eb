// Embedding gather, RMSNorm, and rotary position encoding fused with the
// write of keys and values into the paged cache.  gfx950 only.
#include <type_traits>

#include "common.h"

extern "C" const char* llmlab_last_error() { return g_llmlab_error; }

extern "C" int llmlab_abi_version() { return 11; }

// --------------------------------------------------------------- embedding
// out[r, :] = float(table[ids[r], :]); an id outside [0, vocab) is clamped (the
// host has already refused such ids; the clamp keeps a stale device-side id
// from reading outside the table).
template <typename T>
__global__ void embed_kernel(const T* __restrict__ table, const int* __restrict__ ids,
                             float* __restrict__ out, int hidden, int vocab) {
  const int r = blockIdx.x;
  int id = ids[r];
  id = id < 0 ? 0 : (id >= vocab ? vocab - 1 : id);
  const T* src = table + (size_t)id * hidden;
  float* dst = out + (size_t)r * hidden;
  for (int c = threadIdx.x; c < hidden; c += blockDim.x) dst[c] = to_float(src[c]);
}

// The same from a bfloat16 table packed in MFMA fragment order (see
// llmlab_pack_weight): row `id` is lane column id % 16 of strip id / 16, its
// columns 8 ch .. 8 ch + 7 the 16 bytes of lane (ch % 4) * 16 + id % 16 in tile ch / 4.
__global__ void embed_packed_kernel(const bf16_t* __restrict__ table, const int* __restrict__ ids,
                                    float* __restrict__ out, int hidden, int vocab) {
  const int r = blockIdx.x;
  int id = ids[r];
  id = id < 0 ? 0 : (id >= vocab ? vocab - 1 : id);
  const int tiles = (hidden + 31) >> 5;
  const bf16_t* strip = table + (size_t)(id >> 4) * tiles * 512;
  float* dst = out + (size_t)r * hidden;
  for (int ch = threadIdx.x; ch < (hidden >> 3); ch += blockDim.x) {
    const bf16x8 v = *(const bf16x8*)(strip + (size_t)(ch >> 2) * 512 + (((ch & 3) << 4) + (id & 15)) * 8);
#pragma unroll
    for (int j = 0; j < 8; ++j) dst[ch * 8 + j] = (float)v[j];
  }
}

// dtype DT_BF16 + packed != 0: the table is in fragment order (hidden a multiple of 8).
extern "C" int llmlab_embed(const void* table, int dtype, int packed, const int* ids, float* out, int rows,
                            int hidden, int vocab, hipStream_t stream) {
  LLMLAB_REQUIRE(rows >= 0 && hidden > 0 && vocab > 0, "embed: bad sizes rows=%d hidden=%d vocab=%d",
                 rows, hidden, vocab);
  LLMLAB_REQUIRE(!packed || (dtype == DT_BF16 && hidden % 8 == 0), "embed: a packed table is bfloat16, %d wide", hidden);
  if (rows == 0) return 0;
  dim3 grid(rows), block(256);
  if (packed)
    hipLaunchKernelGGL(embed_packed_kernel, grid, dim3(128), 0, stream, (const bf16_t*)table, ids, out,
                       hidden, vocab);
  else if (dtype == DT_BF16)
    hipLaunchKernelGGL(embed_kernel<bf16_t>, grid, block, 0, stream, (const bf16_t*)table, ids, out,
                       hidden, vocab);
  else
    hipLaunchKernelGGL(embed_kernel<float>, grid, block, 0, stream, (const float*)table, ids, out,
                       hidden, vocab);
  LLMLAB_LAUNCH_CHECK("embed");
  return 0;
}

// ----------------------------------------------------------------- RMSNorm
// W neighbouring weights as they lie in memory, bfloat16 or float32, and their values.  Two loads of 8 bytes without a
// branch (of the same 8 where the weights are bfloat16): converted on the way, each group was waited for
// before the next, and the row, were asked for (48 rows of 896, back to back in a graph, 2.7 us so and 2.1 now; 2,048 rows
// 4.2 and 3.4).
template <int W>
struct RawWeights {
  uint32_t u[W];
  __device__ __forceinline__ float value(int e, int w_bf16) const {
    const uint32_t b = W == 1 ? u[0] << 16 : e & 1 ? u[e / 2] & 0xffff0000u : u[e / 2] << 16;
    return __uint_as_float(w_bf16 ? b : u[e]);
  }
};

template <int W>
__device__ __forceinline__ RawWeights<W> ask_for_weights(const void* w, int w_bf16, int c) {
  RawWeights<W> raw;
  if constexpr (W == 4) {
    typedef uint32_t Pair __attribute__((ext_vector_type(2)));
    const char* at = (const char*)w + (size_t)c * (w_bf16 ? 2 : 4);
    const Pair lo = *(const Pair*)at, hi = *(const Pair*)(at + (w_bf16 ? 0 : 8));
    raw.u[0] = lo[0];
    raw.u[1] = lo[1];
    raw.u[2] = hi[0];
    raw.u[3] = hi[1];
  } else {
    raw.u[0] = w_bf16 ? ((const uint16_t*)w)[c] : ((const uint32_t*)w)[c];
  }
  return raw;
}

// out[i, :] = x[row_i, :] * rsqrt(mean(x[row_i]^2) + eps) * w, row_i = rows[i] or
// i.  The square, the mean, the rsqrt and both products are float32; one
// rounding to T at the end.
// With pieces that a product left for the stream (pend[s][row, :], s < splits), the
// row is first made whole, x[r] += sum_s pend[s][r] (written back: every element
// belongs to one thread), and then normed; rows must not be gathered then.
// A thread keeps its first KEEP groups of W elements (and their weights) in
// registers, so a row of up to KEEP * W * blockDim.x elements costs one trip to
// memory; what lies beyond is read again after the reduction.  VEC: groups of four
// (hidden % 4 == 0 and 16-byte aligned rows).  All loads of a trip are unconditional (past the row's end its last
// group again, not counted): under a branch each would be waited for before the next is asked for.
// The order of a row's sum does not depend on how many threads hold it: SHARE threads of a block of SHARE * blockDim.x are
// one here, with a sum of squares for each (which meet as the waves of that block would: within 64 neighbours,
// then one after the other).  What that block is: llmlab_rmsnorm.
template <typename T, bool VEC, int KEEP, int SHARE, int G>
__global__ void rmsnorm_kernel(float* __restrict__ x, const void* __restrict__ w, int w_bf16,
                               float eps, T* __restrict__ out, const int* __restrict__ rows,
                               int hidden, const float* __restrict__ pend, int splits, size_t pend_stride) {
  constexpr int W = VEC ? 4 : 1;
  static_assert(KEEP % SHARE == 0, "whole rounds");
  __shared__ float red[16];
  const int i = blockIdx.x;
  const int r = rows ? rows[i] : i;
  float* src = x + (size_t)r * hidden;
  const float* prow = pend + (size_t)r * hidden;
  const int stride = blockDim.x * W;
  struct alignas(4 * W) Group {
    float v[W];
  };
  auto get = [](const float* p) {
    Group g;
    if constexpr (VEC) *(floatx4*)g.v = *(const floatx4*)p;
    else g.v[0] = *p;
    return g;
  };
  auto weights = [&](int c) { return ask_for_weights<W>(w, w_bf16, c); };
  // The whole values of N groups from element c on, `stride` apart, written back if pieces came in.  Pieces come G at a
  // time (G = 0: there are none), the first G with the groups themselves: behind a loop's head the compiler waits for
  // what is on its way, so that x and one piece after the other cost a trip each (512 rows of 896 with two pieces
  // 3.4 us so and 2.7 now, 2,048 6.0 and 5.2).
  auto fetch = [&](auto count, int c, Group* g) {
    constexpr int N = decltype(count)::value;
    auto at = [&](int j) { return min(c + j * stride, hidden - W); };
#pragma unroll
    for (int j = 0; j < N; ++j) g[j] = get(src + at(j));
    if constexpr (G > 0) {
      auto pieces = [&](int s0) {
        Group p[N][G];
#pragma unroll
        for (int j = 0; j < N; ++j)
#pragma unroll
          for (int q = 0; q < G; ++q) p[j][q] = get(prow + (size_t)min(s0 + q, splits - 1) * pend_stride + at(j));
#pragma unroll
        for (int j = 0; j < N; ++j)
#pragma unroll
          for (int q = 0; q < G; ++q)
#pragma unroll
            for (int e = 0; e < W; ++e) g[j].v[e] += s0 + q < splits ? p[j][q].v[e] : 0.f;
      };
      pieces(0);
      for (int s0 = G; s0 < splits; s0 += G) pieces(s0);
    }
  };
  auto put_back = [&](int c, const Group& g) {
    if (splits > 0) {
      if constexpr (VEC) *(floatx4*)(src + c) = *(const floatx4*)g.v;
      else src[c] = g.v[0];
    }
  };
  Group keep[KEEP];
  RawWeights<W> wk[KEEP];
  float ss[SHARE];
#pragma unroll
  for (int k = 0; k < SHARE; ++k) ss[k] = 0.f;
  // (a sum's first group: the second square rounded by itself, the others into the sum; fixed here, since it would be
  // the compiler's choice, and another one in each instance)
  auto squares = [](const Group& g, bool first, float sum) {
    if constexpr (W == 4) {
      sum = first ? fmaf(g.v[0], g.v[0], g.v[1] * g.v[1]) : fmaf(g.v[1], g.v[1], fmaf(g.v[0], g.v[0], sum));
      return fmaf(g.v[3], g.v[3], fmaf(g.v[2], g.v[2], sum));
    } else {
      return fmaf(g.v[0], g.v[0], sum);
    }
  };
  const int c0 = threadIdx.x * W;
#pragma unroll
  for (int j = 0; j < KEEP; ++j) wk[j] = weights(min(c0 + j * stride, hidden - W));
  fetch(std::integral_constant<int, KEEP>{}, c0, keep);
#pragma unroll
  for (int j = 0; j < KEEP; ++j) {
    const int c = c0 + j * stride;
    if (c < hidden) put_back(c, keep[j]);
    ss[j % SHARE] = c < hidden ? squares(keep[j], j < SHARE, ss[j % SHARE]) : ss[j % SHARE];
  }
  if constexpr (SHARE == 1)          // (else the groups held are all)
    for (int c = c0 + KEEP * stride; c < hidden; c += stride) {
      Group g;
      fetch(std::integral_constant<int, 1>{}, c, &g);
      put_back(c, g);
      ss[0] = squares(g, false, ss[0]);
    }
  const int waves = blockDim.x >> 6;
  const float sums = full_wave_sums(ss);      // (whole waves, all of whose threads come here)
  float total;
  if (waves > 1) {                   // (a barrier; below a thread reads back only what it wrote itself)
#pragma unroll
    for (int k = 0; k < SHARE; ++k)
      if ((threadIdx.x & 63) == full_wave_place(k)) red[k * waves + (threadIdx.x >> 6)] = sums;
    __syncthreads();
    total = 0.f;
    for (int k = 0; k < waves * SHARE; ++k) total += red[k];
  } else {
    total = lane_value(sums, 0);
#pragma unroll
    for (int k = 1; k < SHARE; ++k) total += lane_value(sums, full_wave_place(k));
  }
  const float inv = rsqrtf(total / (float)hidden + eps);
  T* dst = out + (size_t)i * hidden;
  auto put = [&](int c, const Group& g, const RawWeights<W>& wg) {
    typedef T Out __attribute__((ext_vector_type(W)));
    Out o;
#pragma unroll
    for (int e = 0; e < W; ++e) o[e] = from_float<T>(g.v[e] * inv * wg.value(e, w_bf16));
    *(Out*)(dst + c) = o;
  };
#pragma unroll
  for (int j = 0; j < KEEP; ++j)
    if (c0 + j * stride < hidden) put(c0 + j * stride, keep[j], wk[j]);
  if constexpr (SHARE == 1)
    for (int c = c0 + KEEP * stride; c < hidden; c += stride) put(c, get(src + c), weights(c));
}

extern "C" int llmlab_rmsnorm(float* x, const void* w, int w_dtype, float eps, void* out,
                              int out_dtype, const int* rows, int n_out, int hidden,
                              const float* pend, int splits, size_t pend_stride, hipStream_t stream) {
  LLMLAB_REQUIRE(n_out >= 0 && hidden > 0, "rmsnorm: bad sizes n=%d hidden=%d", n_out, hidden);
  LLMLAB_REQUIRE(splits == 0 || (pend != nullptr && rows == nullptr && pend_stride >= (size_t)n_out * hidden),
                 "rmsnorm: pending sums go with all rows in order");
  if (n_out == 0) return 0;
  const bool vec = hidden % 4 == 0 && pend_stride % 4 == 0 &&
                   (((uintptr_t)x | (uintptr_t)pend | (uintptr_t)out) & 15) == 0 &&
                   ((uintptr_t)w & (w_dtype == DT_BF16 ? 7 : 15)) == 0;
  const int groups = hidden / (vec ? 4 : 1);
  // The block whose order a row's sum has: 256 threads (512 from 8,192 numbers on), for few rows as many as the row has
  // groups of four, up to 1,024; and the groups that one of its threads then takes.
  int order = hidden >= 8192 ? 512 : 256;
  if (n_out <= 128)
    while (order < 1024 && order * 4 < hidden) order *= 2;
  const int rounds = (groups + order - 1) / order;
  // Few rows are bound by latency (and up to 1,024 narrow ones): a thread a group, so that every thread's loads (its
  // numbers and the pieces owed to them) are one round; what 1,024 threads do not hold is read again (8 rows of 5120
  // in eight pieces 4.0 us so, 4.8 with two groups a thread).  Many rows: four groups a thread (two with many pieces:
  // registers), a row of 1,024 and less a wave of its own without a barrier.  (Back to back, before and now: 2,048 rows of 896
  // 4.2 and 3.4 us, in eight pieces 14.2 and 12.5; 2,367 of 3584 14.3 and 9.4; 512 of 5120 5.8 and 4.3.)
  const bool few = n_out <= 128 || (n_out <= 1024 && groups <= 256);
  int keep = vec && few ? 1 : rounds > 2 ? 4 : rounds, share = 1;
  if (vec && !few && rounds <= 2) {
    keep = splits > 2 ? 2 : 4;
    share = keep / rounds;
  }
  const int threads = rounds == 1 && share == 1 ? (groups + 63) / 64 * 64 : order / share;
  dim3 grid(n_out), block(threads);
#define LLMLAB_RMSNORM_KEEP(T, VEC, KEEP, SHARE, G)                                                        \
  hipLaunchKernelGGL((rmsnorm_kernel<T, VEC, KEEP, SHARE, G>), grid, block, 0, stream, x, w, w_dtype == DT_BF16, eps, \
                     (T*)out, rows, hidden, pend, splits, pend_stride)
#define LLMLAB_RMSNORM_PIECES(T, VEC, KEEP, SHARE, MANY)                                                   \
  do {                                                                                                     \
    if (splits == 0) LLMLAB_RMSNORM_KEEP(T, VEC, KEEP, SHARE, 0);                                          \
    else if (splits <= 2) LLMLAB_RMSNORM_KEEP(T, VEC, KEEP, SHARE, 2);                                     \
    else LLMLAB_RMSNORM_KEEP(T, VEC, KEEP, SHARE, MANY);                                                   \
  } while (0)
#define LLMLAB_RMSNORM(T, VEC)                                                                             \
  do {                                                                                                     \
    if (VEC && keep == 4 && share == 4) LLMLAB_RMSNORM_PIECES(T, true, 4, 4, 2);                           \
    else if (VEC && keep == 4 && share == 2) LLMLAB_RMSNORM_PIECES(T, true, 4, 2, 2);                      \
    else if (VEC && keep == 2 && share == 2) LLMLAB_RMSNORM_KEEP(T, true, 2, 2, 4);                        \
    else if (keep == 4) LLMLAB_RMSNORM_PIECES(T, VEC, 4, 1, 2);                                            \
    else if (keep == 2) LLMLAB_RMSNORM_PIECES(T, VEC, 2, 1, 4);                                            \
    else LLMLAB_RMSNORM_PIECES(T, VEC, 1, 1, 4);                                                           \
  } while (0)
  if (out_dtype == DT_BF16) { if (vec) LLMLAB_RMSNORM(bf16_t, true); else LLMLAB_RMSNORM(bf16_t, false); }
  else                      { if (vec) LLMLAB_RMSNORM(float, true);  else LLMLAB_RMSNORM(float, false); }
#undef LLMLAB_RMSNORM_KEEP
#undef LLMLAB_RMSNORM_PIECES
#undef LLMLAB_RMSNORM
  LLMLAB_LAUNCH_CHECK("rmsnorm");
  return 0;
}

// ------------------------------------------------- rotary + cache write
// One block per (row, head) of the packed projection output
//   qkv[r] = [q heads | k heads | v heads], each head `d` wide.
// q heads: rotated in place.  k heads: rotated, written in place and to the
// key page  K[page][kvh][off][d].  v heads: written to the value page, which is
// in the order of the attention kernels' fragments (kcache_index, vcache_index).  page = table[row_req[r]][pos / P],
// off = pos % P.  Angles, sine and cosine in float32; one rounding to T.
// Sine and cosine of a float32 angle.  float32 results: the library routine (exact
// range reduction).  bfloat16 results: the hardware instructions, which take
// revolutions; the reduction  r = frac(angle / 2 pi)  adds an error of the size the
// float32 angle itself has (position * frequency rounded to 24 bits).
template <typename T>
__device__ __forceinline__ void rope_sincos(float angle, float* s, float* c) {
  if constexpr (sizeof(T) == 4) {
    sincosf(angle, s, c);
  } else {
    float r = angle * 0.15915494309189535f;
    r -= floorf(r);
    *s = __builtin_amdgcn_sinf(r);
    *c = __builtin_amdgcn_cosf(r);
  }
}

// One block per row; a thread keeps its pair index over the heads it visits when
// the block size is a multiple of d/2, so its sine and cosine are computed once.
template <typename T>
__global__ __launch_bounds__(256) void rope_kv_write_kernel(
    T* __restrict__ qkv, int row_stride, int nq, int nkv, int d, const float* __restrict__ inv_freq,
    const int* __restrict__ positions, const int* __restrict__ row_req, const int* __restrict__ table,
    int table_stride, int page_size, T* __restrict__ kcache, T* __restrict__ vcache) {
  const int r = blockIdx.x;
  const int pos = positions[r];
  T* row = qkv + (size_t)r * row_stride;
  size_t page = 0;
  int off = 0;
  if (kcache) {
    page = (size_t)table[(size_t)row_req[r] * table_stride + pos / page_size];
    off = pos % page_size;
  }
  const int half = d >> 1;
  const int qk_heads = (kcache || inv_freq) ? nq + nkv : 0;     // heads rotated (k also written)
  const bool fixed_pair = (int)blockDim.x % half == 0;
  float s0 = 0.f, c0 = 1.f;
  if (inv_freq && fixed_pair) rope_sincos<T>((float)pos * inv_freq[threadIdx.x % half], &s0, &c0);
  for (int idx = threadIdx.x; idx < qk_heads * half; idx += blockDim.x) {
    const int head = idx / half, i = idx - head * half;
    T* base = row + (size_t)head * d;
    float lo = to_float(base[i]), hi = to_float(base[i + half]);
    if (inv_freq) {
      float s = s0, c = c0;
      if (!fixed_pair) rope_sincos<T>((float)pos * inv_freq[i], &s, &c);
      const float nlo = lo * c - hi * s, nhi = hi * c + lo * s;
      lo = nlo;
      hi = nhi;
      base[i] = from_float<T>(lo);
      base[i + half] = from_float<T>(hi);
    }
    if (head >= nq && kcache) {
      T* kdst = kcache + (page * nkv + (head - nq)) * (size_t)page_size * d;
      kdst[kcache_index(off, i, d)] = from_float<T>(lo);
      kdst[kcache_index(off, i + half, d)] = from_float<T>(hi);
    }
  }
  if (vcache) {
    const T* vsrc = row + (size_t)(nq + nkv) * d;
    for (int idx = threadIdx.x; idx < nkv * d; idx += blockDim.x) {
      const int head = idx / d, i = idx - head * d;
      vcache[(page * nkv + head) * (size_t)d * page_size + vcache_index(off, i, d)] = vsrc[idx];
    }
  }
}

extern "C" int llmlab_rope_kv_write(void* qkv, int dtype, int rows, int row_stride, int nq, int nkv,
                                    int d, const float* inv_freq, const int* positions,
                                    const int* row_req, const int* table, int table_stride,
                                    int page_size, void* kcache, void* vcache, hipStream_t stream) {
  LLMLAB_REQUIRE(rows >= 0 && nq > 0 && nkv >= 0 && d > 0 && d % 2 == 0,
                 "rope_kv_write: bad sizes rows=%d nq=%d nkv=%d d=%d", rows, nq, nkv, d);
  LLMLAB_REQUIRE(row_stride >= (nq + 2 * nkv) * d || (kcache == nullptr && row_stride >= nq * d),
                 "rope_kv_write: row stride %d is smaller than the heads it holds", row_stride);
  LLMLAB_REQUIRE((kcache == nullptr) == (vcache == nullptr), "rope_kv_write: need both caches or none");
  LLMLAB_REQUIRE(kcache == nullptr || (table != nullptr && row_req != nullptr && page_size > 0),
                 "rope_kv_write: a cache write needs a block table");
  if (rows == 0) return 0;
  // Without a cache only q and k heads are rotated (k in place) and v is left alone.
  if (!kcache && !inv_freq) return 0;
  dim3 grid(rows), block(256);
  if (dtype == DT_BF16)
    hipLaunchKernelGGL(rope_kv_write_kernel<bf16_t>, grid, block, 0, stream, (bf16_t*)qkv, row_stride,
                       nq, nkv, d, inv_freq, positions, row_req, table, table_stride, page_size,
                       (bf16_t*)kcache, (bf16_t*)vcache);
  else
    hipLaunchKernelGGL(rope_kv_write_kernel<float>, grid, block, 0, stream, (float*)qkv, row_stride,
                       nq, nkv, d, inv_freq, positions, row_req, table, table_stride, page_size,
                       (float*)kcache, (float*)vcache);
  LLMLAB_LAUNCH_CHECK("rope_kv_write");
  return 0;
}

// The same from a q/k/v product that was left in pieces along its inner size
// (float32 parts[s][row][ld], s < splits): one block per (row, head) sums the pieces in
// their order, adds the bias, rotates q and k heads and writes q to q_out [rows, ldq] and
// k and v into their cache pages (skipped without a cache).  One rounding, as in the
// product kernels that have this epilogue.  For some rows of a large matrix: cut along
// K the product spreads over the chip, which a head per block does not.
__global__ __launch_bounds__(256) void qkv_from_pieces_kernel(
    const float* __restrict__ parts, int splits, size_t part_stride, int ld, const void* __restrict__ bias,
    int bias_bf16, int nq, int nkv, int d, const float* __restrict__ inv_freq,
    const int* __restrict__ positions, const int* __restrict__ row_req, const int* __restrict__ table,
    int table_stride, int page_size, bf16_t* __restrict__ kcache, bf16_t* __restrict__ vcache,
    bf16_t* __restrict__ q_out, int ldq) {
  const int r = blockIdx.x, head = blockIdx.y;
  if (head >= nq && !kcache) return;
  const int pos = positions[r];
  size_t page = 0;
  int off = 0;
  if (head >= nq) {
    page = (size_t)table[(size_t)row_req[r] * table_stride + pos / page_size];
    off = pos % page_size;
  }
  const int half = d >> 1;
  const float* src = parts + (size_t)r * ld + (size_t)head * d;
  for (int i = threadIdx.x; i < half; i += blockDim.x) {
    float lo = bias ? load_vec(bias, bias_bf16, head * d + i) : 0.f;
    float hi = bias ? load_vec(bias, bias_bf16, head * d + i + half) : 0.f;
    // four pieces at a time, loads unconditional (past the last piece: the last one again,
    // not added), so that they travel together
    for (int s0 = 0; s0 < splits; s0 += 4) {
      float pl[4], ph[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float* ps = src + (size_t)min(s0 + j, splits - 1) * part_stride;
        pl[j] = ps[i];
        ph[j] = ps[i + half];
      }
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (s0 + j < splits) {
          lo += pl[j];
          hi += ph[j];
        }
    }
    if (inv_freq && head < nq + nkv) {
      float sn, cs;
      rope_sincos<bf16_t>((float)pos * inv_freq[i], &sn, &cs);
      const float nlo = lo * cs - hi * sn, nhi = hi * cs + lo * sn;
      lo = nlo;
      hi = nhi;
    }
    if (head < nq) {
      bf16_t* dst = q_out + (size_t)r * ldq + (size_t)head * d;
      dst[i] = (bf16_t)lo;
      dst[i + half] = (bf16_t)hi;
    } else if (head < nq + nkv) {
      bf16_t* kdst = kcache + (page * nkv + (head - nq)) * (size_t)page_size * d;
      kdst[kcache_index(off, i, d)] = (bf16_t)lo;
      kdst[kcache_index(off, i + half, d)] = (bf16_t)hi;
    } else {
      bf16_t* vdst = vcache + (page * nkv + (head - nq - nkv)) * (size_t)d * page_size;
      vdst[vcache_index(off, i, d)] = (bf16_t)lo;
      vdst[vcache_index(off, i + half, d)] = (bf16_t)hi;
    }
  }
}

extern "C" int llmlab_qkv_from_pieces(const float* parts, int splits, size_t part_stride, int ld,
                                      const void* bias, int bias_dtype, int rows, int nq, int nkv, int d,
                                      const float* inv_freq, const int* positions, const int* row_req,
                                      const int* table, int table_stride, int page_size, void* kcache,
                                      void* vcache, void* q_out, int ldq, hipStream_t stream) {
  LLMLAB_REQUIRE(rows >= 0 && nq > 0 && nkv >= 0 && d > 0 && d % 2 == 0 && nq + 2 * nkv <= 65535,
                 "qkv_from_pieces: bad sizes rows=%d nq=%d nkv=%d d=%d", rows, nq, nkv, d);
  LLMLAB_REQUIRE(splits >= 1 && ld >= (nq + 2 * nkv) * d && part_stride >= (size_t)rows * ld && ldq >= nq * d,
                 "qkv_from_pieces: %d pieces, row strides %d and %d", splits, ld, ldq);
  LLMLAB_REQUIRE((kcache == nullptr) == (vcache == nullptr), "qkv_from_pieces: need both caches or none");
  LLMLAB_REQUIRE(positions != nullptr && (kcache == nullptr || (table != nullptr && row_req != nullptr && page_size > 0)),
                 "qkv_from_pieces: positions and, for a cache write, a block table are needed");
  if (rows == 0) return 0;
  const int half = d / 2;
  dim3 grid(rows, nq + 2 * nkv), block(half >= 256 ? 256 : (half + 63) / 64 * 64);
  hipLaunchKernelGGL(qkv_from_pieces_kernel, grid, block, 0, stream, parts, splits, part_stride, ld, bias,
                     bias_dtype == DT_BF16, nq, nkv, d, inv_freq, positions, row_req, table, table_stride,
                     page_size, (bf16_t*)kcache, (bf16_t*)vcache, (bf16_t*)q_out, ldq);
  LLMLAB_LAUNCH_CHECK("qkv_from_pieces");
  return 0;
}

// Rotation alone, of x[rows, heads, d] with arbitrary row and head strides.
template <typename T>
__global__ void rope_inplace_kernel(T* __restrict__ x, long row_stride, long head_stride, int d,
                                    const float* __restrict__ inv_freq,
                                    const int* __restrict__ positions) {
  const int r = blockIdx.x, head = blockIdx.y;
  const int pos = positions[r];
  T* base = x + (size_t)r * row_stride + (size_t)head * head_stride;
  const int half = d >> 1;
  for (int i = threadIdx.x; i < half; i += blockDim.x) {
    const float lo = to_float(base[i]), hi = to_float(base[i + half]);
    float s, c;
    rope_sincos<T>((float)pos * inv_freq[i], &s, &c);
    base[i] = from_float<T>(lo * c - hi * s);
    base[i + half] = from_float<T>(hi * c + lo * s);
  }
}

extern "C" int llmlab_rope_inplace(void* x, int dtype, int rows, int heads, int d, long row_stride,
                                   long head_stride, const float* inv_freq, const int* positions,
                                   hipStream_t stream) {
  LLMLAB_REQUIRE(rows >= 0 && heads > 0 && d > 0 && d % 2 == 0, "rope_inplace: bad sizes");
  if (rows == 0) return 0;
  dim3 grid(rows, heads), block(64);
  if (dtype == DT_BF16)
    hipLaunchKernelGGL(rope_inplace_kernel<bf16_t>, grid, block, 0, stream, (bf16_t*)x, row_stride,
                       head_stride, d, inv_freq, positions);
  else
    hipLaunchKernelGGL(rope_inplace_kernel<float>, grid, block, 0, stream, (float*)x, row_stride,
                       head_stride, d, inv_freq, positions);
  LLMLAB_LAUNCH_CHECK("rope_inplace");
  return 0;
}

// ------------------------------------------------------------- token feedback
// dst[dst_index[i]] = src[src_index[i]]: tokens chosen by the previous step go
// straight into this step's input rows without a trip through the host.
__global__ void gather_tokens_kernel(int* __restrict__ dst, const int* __restrict__ dst_index,
                                     const int* __restrict__ src, const int* __restrict__ src_index,
                                     int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[dst_index[i]] = src[src_index[i]];
}

extern "C" int llmlab_gather_tokens(int* dst, const int* dst_index, const int* src, const int* src_index,
                                    int n, hipStream_t stream) {
  LLMLAB_REQUIRE(n >= 0, "gather_tokens: negative count");
  if (n == 0) return 0;
  hipLaunchKernelGGL(gather_tokens_kernel, dim3((n + 63) / 64), dim3(64), 0, stream, dst, dst_index, src,
                     src_index, n);
  LLMLAB_LAUNCH_CHECK("gather_tokens");
  return 0;
}

// ------------------------------------------------------------ weight packing
// A bfloat16 matrix W [N, K] in MFMA fragment order: strips of 16 rows, each strip
// a run of K/32 tiles (K padded to a multiple of 32, N to a multiple of 16, with
// zeros); a tile is the B operand of one v_mfma_f32_16x16x32_bf16, 1 KB, lane l
// (row l % 16 of the strip, columns 8 * (l / 16) .. + 7 of the tile) owning bytes
// 16 l .. 16 l + 15.  Every product kernel reads W in this order, one or two
// contiguous KB per wave instruction, instead of 16 rows of 64 bytes each.
__global__ __launch_bounds__(256) void pack_weight_kernel(const bf16_t* __restrict__ src,
                                                           bf16_t* __restrict__ dst, int N, int K,
                                                           int tiles_per_strip, long chunks) {
  const long idx = (long)blockIdx.x * 256 + threadIdx.x;
  if (idx >= chunks) return;
  const long tile = idx >> 6;
  const int l = (int)(idx & 63), c = l & 15, g = l >> 4;
  const int n = (int)(tile / tiles_per_strip) * 16 + c;
  const int k = (int)(tile % tiles_per_strip) * 32 + g * 8;
  const bf16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
  *(bf16x8*)(dst + idx * 8) = (n < N && k < K) ? *(const bf16x8*)(src + (size_t)n * K + k) : zero;
}

extern "C" long llmlab_packed_elements(int N, int K) {
  return (long)((N + 15) / 16) * ((K + 31) / 32) * 512;
}

extern "C" int llmlab_pack_weight(const void* src, void* dst, int N, int K, hipStream_t stream) {
  LLMLAB_REQUIRE(N > 0 && K > 0 && K % 8 == 0, "pack_weight: bad sizes N=%d K=%d (K must be a multiple of 8)", N, K);
  LLMLAB_REQUIRE(((uintptr_t)src % 16 == 0) && ((uintptr_t)dst % 16 == 0), "pack_weight: operands must be 16-byte aligned");
  const int tiles = (K + 31) / 32;
  const long chunks = (long)((N + 15) / 16) * tiles * 64;
  hipLaunchKernelGGL(pack_weight_kernel, dim3((unsigned)((chunks + 255) / 256)), dim3(256), 0, stream,
                     (const bf16_t*)src, (bf16_t*)dst, N, K, tiles, chunks);
  LLMLAB_LAUNCH_CHECK("pack_weight");
  return 0;
}

// ------------------------------------------------------------ pending sums
// x[r, :] += sum_s pend[s][r, :], s in order: folds what a product left in pieces
// into the float32 residual stream (for consumers that cannot add it on the fly).
__global__ __launch_bounds__(256) void add_pending_kernel(float* __restrict__ x, const float* __restrict__ pend,
                                                           int splits, size_t stride, long count) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= count) return;
  float v = x[i];
  for (int s = 0; s < splits; ++s) v += pend[s * stride + i];
  x[i] = v;
}

extern "C" int llmlab_add_pending(float* x, const float* pend, int splits, size_t stride, int rows,
                                  int width, hipStream_t stream) {
  LLMLAB_REQUIRE(rows >= 0 && width > 0 && splits >= 0 && stride >= (size_t)rows * width,
                 "add_pending: bad sizes rows=%d width=%d splits=%d", rows, width, splits);
  if (rows == 0 || splits == 0) return 0;
  const long count = (long)rows * width;
  hipLaunchKernelGGL(add_pending_kernel, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, stream, x, pend,
                     splits, stride, count);
  LLMLAB_LAUNCH_CHECK("add_pending");
  return 0;
}

// ------------------------------------------------------------- layer norm
// y = (x - mean(x)) * rsqrt(var(x) + eps) * w with var the mean of the squared
// deviations (taken about the mean, in a pass of its own over registers), no bias; all in float32.
// ADD false: out[i, :] = T(y) for x row rows[i] (or i).  ADD true: the float32 stream
// resid[i, :] += y, and, if copy is given, copy[i, :] = T(resid[i, :]) after the sum: what
// the next reader of the stream multiplies with.  x may be a result that a product left in
// pieces: row i is the sum of x[s][i, :], s < splits, in their order.
//
// A thread keeps its first KEEP groups of W numbers (of the row, the weight and the stream) in
// registers, all asked for at once, so that a row costs one trip to memory; what lies beyond is
// read again.  Few rows are bound by that trip: a row is spread over as many threads as it has
// groups of four, its pieces come G at a time (G = 0: it is whole), the first G with the row, the weights and the stream,
// without a branch (16 rows of 2048 in two pieces, back to back: in three strided passes of 256 threads 6.2 us, 3.2 with
// the loads of a group under a branch, 2.7 so).  Many rows are bound by the memory rate:
// ONE_WAVE, a wave a row and no barrier at all (with the stream's copy, 1,900 rows of 896 7.1 -> 5.2 us by that, 4.5 by
// loads that travel together; in two pieces 5.9 -> 5.1; 2,048 of 2048 14.3 -> 9.9 -> 8.8).
template <typename T, bool ADD, bool VEC, bool ONE_WAVE, int KEEP, int G>
__global__ __launch_bounds__(ONE_WAVE ? 256 : 1024) void layernorm_kernel(
    const float* __restrict__ x, int splits, size_t stride, const void* __restrict__ w, int w_bf16, float eps,
    T* __restrict__ out, float* __restrict__ resid, T* __restrict__ copy, const int* __restrict__ rows, int n_rows,
    int hidden) {
  constexpr int W = VEC ? 4 : 1;
  __shared__ float red[ONE_WAVE ? 1 : 32];
  const int i = ONE_WAVE ? (int)blockIdx.x * 4 + ((int)threadIdx.x >> 6) : (int)blockIdx.x;
  if (ONE_WAVE && i >= n_rows) return;                     // (a wave's row is its own: no barrier below)
  const int t = ONE_WAVE ? (int)threadIdx.x & 63 : (int)threadIdx.x, step = (ONE_WAVE ? 64 : (int)blockDim.x) * W;
  const float* src = x + (size_t)(rows ? rows[i] : i) * hidden;
  struct alignas(4 * W) Group {
    float v[W];
  };
  auto get = [](const float* p) {
    Group g;
    if constexpr (VEC) *(floatx4*)g.v = *(const floatx4*)p;
    else g.v[0] = *p;
    return g;
  };
  // The whole values of N groups from element c on, `step` apart (loads unconditional: past the last piece the last one
  // again, not added; past the row's end its last group again, not counted).
  auto fetch = [&](auto count, int c, Group* g) {
    constexpr int N = decltype(count)::value;
    auto at = [&](int j) { return min(c + j * step, hidden - W); };
#pragma unroll
    for (int j = 0; j < N; ++j) g[j] = get(src + at(j));
    if constexpr (G > 0) {
      auto pieces = [&](int s0) {
        Group p[N][G];
#pragma unroll
        for (int j = 0; j < N; ++j)
#pragma unroll
          for (int q = 0; q < G; ++q) p[j][q] = get(src + min(s0 + q, splits - 1) * stride + at(j));
#pragma unroll
        for (int j = 0; j < N; ++j)
#pragma unroll
          for (int q = 0; q < G; ++q)
#pragma unroll
            for (int e = 0; e < W; ++e) g[j].v[e] += s0 + q < splits ? p[j][q].v[e] : 0.f;
      };
      pieces(1);
      for (int s0 = 1 + G; s0 < splits; s0 += G) pieces(s0);
    }
  };
  auto whole = [&](int c) {
    Group g;
    fetch(std::integral_constant<int, 1>{}, c, &g);
    return g;
  };
  auto weights = [&](int c) { return ask_for_weights<W>(w, w_bf16, c); };
  auto total = [&](float v, int which) {
    v = full_wave_sum(v);      // (whole waves, all of whose threads come here)
    if constexpr (!ONE_WAVE) {
      if ((threadIdx.x & 63) == 0) red[which * 16 + (threadIdx.x >> 6)] = v;
      __syncthreads();
      v = 0.f;
      for (int k = 0; k < (int)(blockDim.x >> 6); ++k) v += red[which * 16 + k];
    }
    return v;
  };
  Group keep[KEEP], old[KEEP];
  RawWeights<W> wk[KEEP];
  float s = 0.f;
#pragma unroll
  for (int j = 0; j < KEEP; ++j) {
    const int c = min(t * W + j * step, hidden - W);
    wk[j] = weights(c);
    if (ADD) old[j] = get(resid + (size_t)i * hidden + c);
  }
  fetch(std::integral_constant<int, KEEP>{}, t * W, keep);
#pragma unroll
  for (int j = 0; j < KEEP; ++j)
#pragma unroll
    for (int e = 0; e < W; ++e) s += t * W + j * step < hidden ? keep[j].v[e] : 0.f;
  for (int c = t * W + KEEP * step; c < hidden; c += step) {
    const Group g = whole(c);
#pragma unroll
    for (int e = 0; e < W; ++e) s += g.v[e];
  }
  const float mean = total(s, 0) / (float)hidden;
  float v = 0.f;
  // (the roundings fixed, and the same in all instances: see rmsnorm_kernel)
  auto deviate = [&](const Group& g, bool first) {
    float d[W];
#pragma unroll
    for (int e = 0; e < W; ++e) d[e] = g.v[e] - mean;
    if constexpr (W == 4) {
      v = first ? fmaf(d[0], d[0], d[1] * d[1]) : fmaf(d[1], d[1], fmaf(d[0], d[0], v));
      v = fmaf(d[3], d[3], fmaf(d[2], d[2], v));
    } else {
      v = fmaf(d[0], d[0], v);
    }
  };
#pragma unroll
  for (int j = 0; j < KEEP; ++j)
    if (t * W + j * step < hidden) deviate(keep[j], j == 0);
  for (int c = t * W + KEEP * step; c < hidden; c += step) deviate(whole(c), false);
  const float inv = 1.0f / sqrtf(total(v, 1) / (float)hidden + eps);
  auto put = [&](int c, const Group& g, const RawWeights<W>& wg, const Group& og) {
    typedef T Out __attribute__((ext_vector_type(W)));
    Group y;
    Out o;
#pragma unroll
    for (int e = 0; e < W; ++e) {
      y.v[e] = (g.v[e] - mean) * inv * wg.value(e, w_bf16);
      if (ADD) y.v[e] += og.v[e];
      o[e] = from_float<T>(y.v[e]);
    }
    if (ADD) {
      float* dst = resid + (size_t)i * hidden + c;
      if constexpr (VEC) *(floatx4*)dst = *(const floatx4*)y.v;
      else *dst = y.v[0];
      if (copy) *(Out*)(copy + (size_t)i * hidden + c) = o;
    } else {
      *(Out*)(out + (size_t)i * hidden + c) = o;
    }
  };
#pragma unroll
  for (int j = 0; j < KEEP; ++j) {
    const int c = t * W + j * step;
    if (c < hidden) put(c, keep[j], wk[j], old[j]);
  }
  for (int c = t * W + KEEP * step; c < hidden; c += step)
    put(c, whole(c), weights(c), ADD ? get(resid + (size_t)i * hidden + c) : Group{});
}

template <typename T, bool ADD>
static void launch_layernorm(const float* x, int splits, size_t stride, const void* w, int w_bf16, float eps, T* out,
                             float* resid, T* copy, const int* rows, int n_rows, int hidden, hipStream_t stream) {
  const bool vec = hidden % 4 == 0 && stride % 4 == 0 && (((uintptr_t)x | (uintptr_t)resid) & 15) == 0 &&
                   (((uintptr_t)out | (uintptr_t)copy) & (4 * sizeof(T) - 1)) == 0 &&
                   ((uintptr_t)w & (w_bf16 ? 7 : 15)) == 0;
  // A wave a row where the rows fill the chip and a row fits a wave's registers; else a block, whose
  // threads cover the row in one group each, or in two to four where 1,024 threads (256 for more than 128 rows) do not.
#define LLMLAB_LAYERNORM(VEC, ONE_WAVE, KEEP, G, grid, threads)                                                     \
  hipLaunchKernelGGL((layernorm_kernel<T, ADD, VEC, ONE_WAVE, KEEP, G>), dim3(grid), dim3(threads), 0, stream, x,   \
                     splits, stride, w, w_bf16, eps, out, resid, copy, rows, n_rows, hidden)
  if (vec && n_rows > 512 && hidden <= 2048) {
    const int blocks = (n_rows + 3) / 4;
    if (hidden <= 1024 && splits == 1) LLMLAB_LAYERNORM(true, true, 4, 0, blocks, 256);
    else if (hidden <= 1024) LLMLAB_LAYERNORM(true, true, 4, 1, blocks, 256);
    else if (splits == 1) LLMLAB_LAYERNORM(true, true, 8, 0, blocks, 256);
    else LLMLAB_LAYERNORM(true, true, 8, 1, blocks, 256);
    return;
  }
  int threads = 64;
  while (threads < 1024 && threads * (vec ? 4 : 1) < hidden) threads += 64;
  if (n_rows > 128 && threads > 256) threads = 256;
  if (vec && threads * 4 >= hidden && splits == 1) LLMLAB_LAYERNORM(true, false, 1, 0, n_rows, threads);
  else if (vec && threads * 4 >= hidden) LLMLAB_LAYERNORM(true, false, 1, 4, n_rows, threads);
  else if (vec && threads * 8 >= hidden && splits == 1) LLMLAB_LAYERNORM(true, false, 2, 0, n_rows, threads);
  else if (vec && threads * 8 >= hidden) LLMLAB_LAYERNORM(true, false, 2, 2, n_rows, threads);
  else if (vec && threads * 12 >= hidden && splits == 1) LLMLAB_LAYERNORM(true, false, 3, 0, n_rows, threads);
  else if (vec && threads * 12 >= hidden) LLMLAB_LAYERNORM(true, false, 3, 2, n_rows, threads);
  else if (vec && splits == 1) LLMLAB_LAYERNORM(true, false, 4, 0, n_rows, threads);
  else if (vec) LLMLAB_LAYERNORM(true, false, 4, 2, n_rows, threads);
  else LLMLAB_LAYERNORM(false, false, 4, 4, n_rows, threads);
#undef LLMLAB_LAYERNORM
}

// out: n_out rows of the compute dtype; rows: which rows of x (null: all in order).
extern "C" int llmlab_layernorm(const float* x, const void* w, int w_dtype, float eps, void* out, int out_dtype,
                                const int* rows, int n_out, int hidden, hipStream_t stream) {
  LLMLAB_REQUIRE(n_out >= 0 && hidden > 0, "layernorm: bad sizes n=%d hidden=%d", n_out, hidden);
  if (n_out == 0) return 0;
  if (out_dtype == DT_BF16)
    launch_layernorm<bf16_t, false>(x, 1, 0, w, w_dtype == DT_BF16, eps, (bf16_t*)out, nullptr, nullptr, rows, n_out,
                                    hidden, stream);
  else
    launch_layernorm<float, false>(x, 1, 0, w, w_dtype == DT_BF16, eps, (float*)out, nullptr, nullptr, rows, n_out,
                                   hidden, stream);
  LLMLAB_LAUNCH_CHECK("layernorm");
  return 0;
}

// resid += layernorm(y), y the sum of `splits` pieces `stride` numbers apart; copy (may be null, of copy_dtype)
// receives the new rows of resid.
extern "C" int llmlab_layernorm_add(const float* y, int splits, size_t stride, const void* w, int w_dtype, float eps,
                                    float* resid, void* copy, int copy_dtype, int n_rows, int hidden,
                                    hipStream_t stream) {
  LLMLAB_REQUIRE(n_rows >= 0 && hidden > 0, "layernorm_add: bad sizes n=%d hidden=%d", n_rows, hidden);
  LLMLAB_REQUIRE(y != resid, "layernorm_add: the sublayer's output and the stream are two buffers");
  LLMLAB_REQUIRE(splits == 1 || (splits > 1 && stride >= (size_t)n_rows * hidden),
                 "layernorm_add: %d pieces do not follow each other", splits);
  if (n_rows == 0) return 0;
  if (copy_dtype == DT_BF16)
    launch_layernorm<bf16_t, true>(y, splits, stride, w, w_dtype == DT_BF16, eps, nullptr, resid, (bf16_t*)copy, nullptr,
                                   n_rows, hidden, stream);
  else
    launch_layernorm<float, true>(y, splits, stride, w, w_dtype == DT_BF16, eps, nullptr, resid, (float*)copy, nullptr,
                                  n_rows, hidden, stream);
  LLMLAB_LAUNCH_CHECK("layernorm_add");
  return 0;
}

// ------------------------------------------------- activations on float32 sums
#define ACT_CAST 0        // out = T(x)
#define ACT_RELU2 1       // out = T(max(x, 0)^2)
#define ACT_ZERO 2        // out = 0
template <typename T, int ACT>
__global__ void activation_kernel(const float* __restrict__ x, T* __restrict__ out, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    float v = ACT == ACT_ZERO ? 0.f : x[i];
    if (ACT == ACT_RELU2) {
      v = fmaxf(v, 0.f);
      v = v * v;
    }
    out[i] = from_float<T>(v);
  }
}

// The float32 output of a product becomes the next product's input (compute dtype) through
// an activation.  In float32 ``out`` may be ``x`` itself.
extern "C" int llmlab_activation(const float* x, void* out, int out_dtype, int act, long n, hipStream_t stream) {
  LLMLAB_REQUIRE(n >= 0 && act >= ACT_CAST && act <= ACT_ZERO, "activation: bad arguments n=%ld act=%d", n, act);
  if (n == 0) return 0;
  const int blocks = (int)((n + 255) / 256 < 65535 ? (n + 255) / 256 : 65535);
#define LLMLAB_ACT(T, A) hipLaunchKernelGGL((activation_kernel<T, A>), dim3(blocks), dim3(256), 0, stream, x, (T*)out, (size_t)n)
  if (out_dtype == DT_BF16) {
    if (act == ACT_RELU2) LLMLAB_ACT(bf16_t, ACT_RELU2); else if (act == ACT_ZERO) LLMLAB_ACT(bf16_t, ACT_ZERO); else LLMLAB_ACT(bf16_t, ACT_CAST);
  } else {
    if (act == ACT_RELU2) LLMLAB_ACT(float, ACT_RELU2); else if (act == ACT_ZERO) LLMLAB_ACT(float, ACT_ZERO); else LLMLAB_ACT(float, ACT_CAST);
  }
#undef LLMLAB_ACT
  LLMLAB_LAUNCH_CHECK("activation");
  return 0;
}

// ------------------------------------------------- one gate per head on a mixer's output
// out[r, h, :] *= sigmoid(gate[r, h]): the sigmoid and the product in float32, one rounding.
template <typename T>
__global__ void gate_heads_kernel(T* __restrict__ out, const float* __restrict__ gate, int heads, int head_dim,
                                  size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    const float g = gate[i / head_dim];          // (rows of heads * head_dim numbers, gates [rows, heads])
    out[i] = from_float<T>(to_float(out[i]) / (1.f + __expf(-g)));
  }
}

extern "C" int llmlab_gate_heads(void* out, int dtype, const float* gate, int rows, int heads, int head_dim,
                                 hipStream_t stream) {
  LLMLAB_REQUIRE(rows >= 0 && heads > 0 && head_dim > 0, "gate_heads: bad sizes rows=%d heads=%d head_dim=%d", rows,
                 heads, head_dim);
  const size_t n = (size_t)rows * heads * head_dim;
  if (n == 0) return 0;
  const int blocks = (int)((n + 255) / 256 < 65535 ? (n + 255) / 256 : 65535);
  if (dtype == DT_BF16)
    hipLaunchKernelGGL(gate_heads_kernel<bf16_t>, dim3(blocks), dim3(256), 0, stream, (bf16_t*)out, gate, heads,
                       head_dim, n);
  else
    hipLaunchKernelGGL(gate_heads_kernel<float>, dim3(blocks), dim3(256), 0, stream, (float*)out, gate, heads,
                       head_dim, n);
  LLMLAB_LAUNCH_CHECK("gate_heads");
  return 0;
}

// ------------------------------------------------- one vector added to every row of the stream
__global__ void add_row_vector_kernel(float* __restrict__ x, const float* __restrict__ v, int hidden, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    x[i] += v[i % hidden];
}

extern "C" int llmlab_add_row_vector(float* x, const float* v, int rows, int hidden, hipStream_t stream) {
  LLMLAB_REQUIRE(rows >= 0 && hidden > 0, "add_row_vector: bad sizes rows=%d hidden=%d", rows, hidden);
  const size_t n = (size_t)rows * hidden;
  if (n == 0) return 0;
  const int blocks = (int)((n + 255) / 256 < 65535 ? (n + 255) / 256 : 65535);
  hipLaunchKernelGGL(add_row_vector_kernel, dim3(blocks), dim3(256), 0, stream, x, v, hidden, n);
  LLMLAB_LAUNCH_CHECK("add_row_vector");
  return 0;
}
