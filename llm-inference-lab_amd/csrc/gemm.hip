// Matrix products  out = x . W^T  (x [M, K] K-contiguous; W [N, K], in bfloat16
// packed in MFMA fragment order by llmlab_pack_weight, in float32 K-contiguous)
// for gfx950, with the epilogues the model needs fused in.
//
//   bfloat16:  v_mfma_f32_16x16x32_bf16 everywhere.
//     * small products: 64x64, four waves 2x2, both operands loaded from global memory straight
//       into a ring of three stages of LDS (gemm_bf16_ring); 128x128, 128x192 and 192x128 with eight waves 4x2 in the same
//       way where their blocks find a unit each, or two of them one.
//     * tiled kernel: 256 threads = 4 waves, block tile 64x128 or
//       128x128 (waves 1x4, side by side along the columns), or 512 threads = 8 waves on
//       128x256 (1x8; widths of 96 to 224 with a wave per 32 columns; 64x64 with waves 2x2 for grouped
//       products only), K step 64; x staged through
//       three stages of LDS (rows padded to 80 elements: a wave's 16-byte fragment reads
//       then take 8.4 clocks, as lane-contiguous ones do; 9.5 with 72, 16 unpadded), its
//       fragments read into registers half a tile ahead of their products, the fragments
//       of W read straight from the packed matrix into registers; three or four tiles
//       are on their way from memory in a ring of register buffers while one is
//       multiplied.  With the waves 1x4 every
//       fragment of W is read by one wave only and all four share the rows of x in LDS:
//       5 to 35 % faster than 2x2 waves with W staged through LDS too (which was the
//       large tile before).  Also measured and not adopted: 256x128 tiles with eight
//       64x64 or four 128x64 wave tiles, K steps of 128, 128x256, 64x256, 128x64 and
//       32x128 tiles with 1x4 waves (the second as good as 128x128, no better), eight
//       waves 2x4 on 128x128 and 64x128, a 64x256 tile with eight waves 1x8 for few rows of a wide
//       matrix (as fast as 64x128, no faster), and 256x256 tiles with four 128x128 wave tiles (half the LDS traffic
//       per product, one wave per SIMD: 833 against 793 TF/s on the largest product
//       tried, slower on the rest).  Counters of the 128x128 tile on a product of
//       2048 x 37888 x 3584 (900 TF/s; two blocks share a compute unit, the clock is at
//       2.0 GHz under this load): matrix pipes busy 40 % of the time, LDS 52 % (and
//       counted in bank conflicts for another 21 %), the texture address units 56 %: no
//       unit is the limit alone, the waves wait for one another's turns at three of them.
//     * the largest products (from 1024 rows on, where its blocks fill the chip): a 256x256
//       tile whose eight waves form two groups that alternate between reading LDS and
//       issuing MFMAs, both operands loaded from global memory straight into LDS
//       (gemm_bf16_pingpong): 1.1 to 1.25 PF/s where the tiles above reach 0.9 to 0.97.
//     (products of few rows, as in decode steps, have kernels of their own in decode.hip)
//   float32: numbers split into three bfloat16 parts (W in one where its numbers are bfloat16 ones) for the matrix
//     cores, 32-bit products and sums as exact as plain FMAs (gemm_f32_split_kernel); a plain FMA kernel beside it as its
//     reference (tiles of 64x64 to 128x128, 4x4 to 8x8 outputs per thread); for up to 64 rows one in
//     which a wave owns four rows of W and its lanes split the inner size.
//
// Fragment layout of the 16x16x32 MFMA (wave of 64 lanes, lane l):
//   A operand: row l%16, k = 8*(l/16) .. +7      B operand: column l%16, same k
//   result element i (0..3): row 4*(l/16)+i, column l%16
//
// Epilogues: STORE  out[M,N] (T) = acc (+bias)            RESID  out[M,N] (f32) += acc (+bias)
//            F32    out[M,N] (f32) = acc                   SWIGLU out[M,N/2] (T) = silu(g)*u
//            PART   out[z][M,N] (f32) = acc over the K range of group z
//            QKV    q (T) = rotate(acc + bias); rotated k and v of the rows go to their cache pages
// For SWIGLU the rows of W alternate in runs of 16: gate rows of 16 outputs, then
// the up rows of the same 16 outputs, so fragments j and j+1 hold gate and up of
// the same outputs in the same lanes.
#include <type_traits>

#include "common.h"

enum { EPI_STORE = 0, EPI_RESID = 1, EPI_F32 = 2, EPI_SWIGLU = 3, EPI_QKV = 4, EPI_PART = 5 };

struct EpiArgs {
  void* out;         // T or float, see above
  const void* bias;  // may be null
  int bias_bf16;
  int ldo;    // row stride of out in elements
  int n_out;  // logical output columns (SWIGLU: intermediate size; else N)
  // PART: the inner size is cut over the blocks of grid z, kt_per_split K tiles each; group z
  // leaves its sums (float32, bias in group 0) in out + z * part_stride: the product without
  // the final sum, which the next reader of those rows does
  int kt_per_split;
  size_t part_stride;
  // QKV: the columns are [q heads | k heads | v heads] of size d; q and k are rotated by
  // their row's position, q goes to out [M, ldo], k and v into the cache pages of the row's
  // request (skipped when no cache is given).  A head must lie within one tile (BN % d == 0).
  const float* inv_freq;   // [d/2] or null (no rotation)
  const int* positions;    // [M]
  const int* row_req;      // [M]
  const int* table;        // block table
  bf16_t* kcache;
  bf16_t* vcache;
  int table_stride, page_size, nq, nkv, d;
  // STORE: 1 = the sum goes through max(z, 0)^2 (in float32) before it is rounded;
  // SWIGLU: 2 = the gate goes through gelu (tanh form) instead of silu; 3 = the clamped pair (below)
  int act;
  // Grouped products (several matrices of equal shape, one below the other in W; every tile of
  // rows belongs to one of them): g_tile[tile of rows] is the tile's matrix (-1: the tile is
  // empty), g_w_stride the packed elements of one matrix, g_rows (may be null) the row of x that
  // row m of the product reads (-1: none; such rows' results land in rows nobody reads).
  const int* g_tile;
  const int* g_rows;
  size_t g_w_stride;
  float limit, slope, shift;      // constants of the clamped pair
};

__device__ __forceinline__ float relu2_f(float z) {
  z = fmaxf(z, 0.f);
  return z * z;
}

// (the function of the few-row kernel, to the bit)
__device__ __forceinline__ float silu_f(float z) { return z / (1.f + __expf(-z)); }

// tanh form of gelu: 0.5 z (1 + tanh(sqrt(2/pi) (z + 0.044715 z^3))), as z * sigmoid(2 t)
__device__ __forceinline__ float gelu_tanh_f(float z) {
  const float t = 0.7978845608028654f * (z + 0.044715f * z * z * z);
  return z / (1.f + __expf(-2.f * t));
}
__device__ __forceinline__ float gelu_tanh_exact_f(float z) {
  const float t = 0.7978845608028654f * (z + 0.044715f * z * z * z);
  return 0.5f * z * (1.f + tanhf(t));
}
// the gate of a paired product: act 2 = gelu (tanh form), else silu
__device__ __forceinline__ float gate_act_f(float z, int act) { return act == 2 ? gelu_tanh_f(z) : silu_f(z); }
__device__ __forceinline__ float gate_act_exact_f(float z, int act) {
  return act == 2 ? gelu_tanh_exact_f(z) : z / (1.f + expf(-z));
}

// A gated pair: act(gate) * up; act 3, the clamped pair: with g = min(gate, limit) and u = up held within
// -limit .. limit, g * sigmoid(slope * g) * (u + shift).
__device__ __forceinline__ float pair_f(float g, float u, int act, const EpiArgs& e) {
  if (act != 3) return gate_act_f(g, act) * u;
  g = fminf(g, e.limit);
  return g / (1.f + __expf(-e.slope * g)) * (fminf(fmaxf(u, -e.limit), e.limit) + e.shift);
}
__device__ __forceinline__ float pair_exact_f(float g, float u, const EpiArgs& e) {
  if (e.act != 3) return gate_act_exact_f(g, e.act) * u;
  g = fminf(g, e.limit);
  return g / (1.f + expf(-e.slope * g)) * (fminf(fmaxf(u, -e.limit), e.limit) + e.shift);
}

// One output element (non-SWIGLU).
template <typename T, int EPI>
__device__ __forceinline__ void epi_store(const EpiArgs& e, int m, int n, float acc) {
  if (e.bias) acc += load_vec(e.bias, e.bias_bf16, n);
  const size_t at = (size_t)m * e.ldo + n;
  if (EPI == EPI_STORE)
    ((T*)e.out)[at] = from_float<T>(e.act ? relu2_f(acc) : acc);
  else if (EPI == EPI_RESID)
    ((float*)e.out)[at] += acc;
  else
    ((float*)e.out)[at] = acc;
}

// The epilogue of a wave's sums where they are: lane (c, g) holds, of the 16 x 16 block (i, j), row m0 + 16 i + c and
// the columns n0 + 16 j + 4 g .. + 3 (products taken transposed, W x^T).  Sums of 32 bits are written, and the residual
// read, 16 bytes a lane, a row of blocks on its way while the one before is added; two blocks of bfloat16 results are
// exchanged between neighbouring groups of lanes so that a lane writes 16 bytes too.  By way of LDS, where a thread found
// the activation anew for each number, a tile alone on its unit spent 14 us so with a residual (192 x 256, a trip to memory
// behind the other) and 11 with paired results (256 x 256); here 7, at the rate of memory for what all units then want
// at once, and 2.3 with the hardware's reciprocal in place of the activation's division, which takes 2 more (192 x
// 256: gate and up of 2,048 rows of the 0.5B shape, two rounds, 54 us by way of LDS, 43 and 47).
template <int TM, int TN, int EPI>
__device__ __forceinline__ void register_epilogue(const floatx4 (&acc)[TM][TN], const EpiArgs& e, int m0, int n0, int M,
                                                  int N, int c, int g) {
  static_assert(TN % 2 == 0 && (TN % 4 == 0 || TM % 2 == 0 || EPI != EPI_SWIGLU), "blocks in pairs");
  // eight neighbouring results a lane out of four of block a and four of block b: lane groups 0 and 2 get a's, 1 and
  // 3 b's, the lower half of the block's columns in groups 0 and 1
  auto exchange = [](const bf16x4& a, const bf16x4& b) {
    typedef __attribute__((__vector_size__(2 * sizeof(uint32_t)))) uint32_t u32x2;
    typedef __attribute__((__vector_size__(4 * sizeof(uint32_t)))) uint32_t u32x4;
    const u32x2 x = __builtin_bit_cast(u32x2, a), y = __builtin_bit_cast(u32x2, b);
    const auto r0 = __builtin_amdgcn_permlane16_swap(x[0], y[0], false, false);
    const auto r1 = __builtin_amdgcn_permlane16_swap(x[1], y[1], false, false);
    return __builtin_bit_cast(bf16x8, u32x4{(uint32_t)r0[0], (uint32_t)r1[0], (uint32_t)r0[1], (uint32_t)r1[1]});
  };
  if constexpr (EPI == EPI_SWIGLU) {
    // columns alternate in runs of 16: gate, up of the same 16 outputs
    bf16_t* out = (bf16_t*)e.out;
    const int o0 = n0 >> 1;
    const bool whole = (e.ldo & 7) == 0 && ((uintptr_t)out & 15) == 0 && o0 + TN * 8 <= e.n_out;
    auto put = [&](int m, int col, const bf16x4& v) {      // (unaligned, or past the last output)
      if (m < M)
#pragma unroll
        for (int x = 0; x < 4; ++x)
          if (o0 + col + x < e.n_out) out[(size_t)m * e.ldo + o0 + col + x] = v[x];
    };
    // (two runs of outputs of a row where a wave has them, else the same run of two rows)
    constexpr int DI = TN % 4 == 0 ? 1 : 2, DJ = TN % 4 == 0 ? 2 : 1;
    auto results = [&](auto act) {      // (the activation a constant: no branch a number)
      auto pair = [&](int i, int jp) {
        bf16x4 v;
#pragma unroll
        for (int x = 0; x < 4; ++x) v[x] = (bf16_t)pair_f(acc[i][2 * jp][x], acc[i][2 * jp + 1][x], decltype(act)::value, e);
        return v;
      };
#pragma unroll
      for (int i = 0; i < TM; i += DI)
#pragma unroll
        for (int jp = 0; jp < TN / 2; jp += DJ) {
          const int i1 = i + DI - 1, jp1 = jp + DJ - 1;
          const bf16x4 a = pair(i, jp), b = pair(i1, jp1);
          if (whole) {
            const bf16x8 v = exchange(a, b);
            const int m = m0 + 16 * ((g & 1) ? i1 : i) + c, col = 16 * ((g & 1) ? jp1 : jp) + (g >> 1) * 8;
            if (m < M) *(bf16x8*)(out + (size_t)m * e.ldo + o0 + col) = v;
          } else {
            put(m0 + 16 * i + c, 16 * jp + 4 * g, a);
            put(m0 + 16 * i1 + c, 16 * jp1 + 4 * g, b);
          }
        }
    };
    if (e.act == 3) results(std::integral_constant<int, 3>{});
    else if (e.act == 2) results(std::integral_constant<int, 2>{});
    else results(std::integral_constant<int, 0>{});
  } else if constexpr (EPI != EPI_QKV) {
    constexpr bool OUT32 = EPI != EPI_STORE;
    const bool whole = (e.ldo & (OUT32 ? 3 : 7)) == 0 && ((uintptr_t)e.out & 15) == 0 && n0 + TN * 16 <= N;
    floatx4 bias[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) bias[j] = floatx4{0.f, 0.f, 0.f, 0.f};
    if (e.bias) {
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int x = 0; x < 4; ++x) bias[j][x] = load_vec(e.bias, e.bias_bf16, min(n0 + 16 * j + 4 * g + x, N - 1));
    }
    if (!whole) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const int m = m0 + 16 * i + c;
#pragma unroll
          for (int x = 0; x < 4; ++x) {
            const int n = n0 + 16 * j + 4 * g + x;
            if (m >= M || n >= N) continue;
            const size_t at = (size_t)m * e.ldo + n;
            float v = acc[i][j][x] + bias[j][x];
            if constexpr (EPI == EPI_STORE) {
              if (e.act) v = relu2_f(v);
              ((bf16_t*)e.out)[at] = (bf16_t)v;
            } else {
              ((float*)e.out)[at] = (EPI == EPI_RESID ? ((float*)e.out)[at] : 0.f) + v;
            }
          }
        }
    } else if constexpr (EPI == EPI_STORE) {
      auto rounded = [&](int i, int j) {
        floatx4 v = acc[i][j] + bias[j];
        if (e.act)
#pragma unroll
          for (int x = 0; x < 4; ++x) v[x] = relu2_f(v[x]);
        return bf16x4{(bf16_t)v[0], (bf16_t)v[1], (bf16_t)v[2], (bf16_t)v[3]};
      };
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; j += 2) {
          const bf16x8 v = exchange(rounded(i, j), rounded(i, j + 1));
          const int m = m0 + 16 * i + c;
          if (m < M) *(bf16x8*)((bf16_t*)e.out + (size_t)m * e.ldo + n0 + 16 * (j + (g & 1)) + (g >> 1) * 8) = v;
        }
    } else {
      // neighbouring lanes have neighbouring rows: one takes both halves' columns of the even row's 32, the other of
      // the odd one's, so that an instruction touches eight rows by 128 bytes and not sixteen by 64
      const bool odd = c & 1;
      float* const out = (float*)e.out + n0 + (odd ? 16 : 0) + 4 * g;
      auto row = [&](int i, int h) { return out + (size_t)min(m0 + 16 * i + (c & ~1) + h, M - 1) * e.ldo; };
      floatx4 old[2][2][TN / 2];
      auto ask = [&](int i) {
        if constexpr (EPI == EPI_RESID) {
#pragma unroll
          for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int jp = 0; jp < TN / 2; ++jp) old[i & 1][h][jp] = *(const floatx4*)(row(i, h) + 32 * jp);
        }
      };
      ask(0);
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        if (i + 1 < TM) ask(i + 1);
#pragma unroll
        for (int jp = 0; jp < TN / 2; ++jp) {
          const floatx4 a = acc[i][2 * jp] + bias[2 * jp], b = acc[i][2 * jp + 1] + bias[2 * jp + 1];
          floatx4 v[2];
#pragma unroll
          for (int x = 0; x < 4; ++x) {
            const float a1 = dpp_move<0xB1>(a[x]), b1 = dpp_move<0xB1>(b[x]);      // the neighbour's
            v[0][x] = odd ? b1 : a[x];
            v[1][x] = odd ? b[x] : a1;
          }
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            if constexpr (EPI == EPI_RESID) v[h] = old[i & 1][h][jp] + v[h];
            if (m0 + 16 * i + (c & ~1) + h < M) *(floatx4*)(row(i, h) + 32 * jp) = v[h];
          }
        }
      }
    }
  }
}

// The epilogue of a q/k/v tile of BM x BN sums that lies in LDS (rows of BN + 4 floats), by the NT
// threads of the block: global memory is written in pieces of 16 bytes, consecutive lanes next to
// each other.  s_pos, s_page, s_freq and s_bias are what the QKV
// epilogue fetched per row and per column of the tile before the product.
template <int BM, int BN, int NT, int EPI>
__device__ __forceinline__ void tile_epilogue(const float* Cs, const EpiArgs& e, int m0, int n0, int M, int N,
                                              int tid, const int* s_pos, const int* s_page, const float* s_freq,
                                              const float* s_bias) {
  constexpr int C_STRIDE = BN + 4;
  if constexpr (EPI == EPI_QKV) {
    // q and k heads.  A unit of work: eight pairs (i .. i+7, and those + d/2) of one head of
    // one row, rotated and stored 16 bytes at a time (eight neighbours of one octet of d lie
    // next to each other in the key order too).
    const int d = e.d, dh = d >> 1, heads = BN / d, cpl = dh >> 3, head0 = n0 / d;
    const int units = BM * heads * cpl;
    const bool vec = (e.ldo & 7) == 0 && ((uintptr_t)e.out & 15) == 0;
    for (int u = tid; u < units; u += NT) {
      const int jc = u % cpl, t = u / cpl, hh = t % heads, row = t / heads;
      const int m = m0 + row, head = head0 + hh, i = jc * 8;
      if (m >= M || head >= e.nq + e.nkv) continue;          // (values: below)
      const bool is_q = head < e.nq;
      if (!is_q && !e.kcache) continue;
      const float* src = Cs + row * C_STRIDE + hh * d + i;
      float lo[8], hi[8];
#pragma unroll
      for (int q = 0; q < 8; q += 4) {
        const floatx4 l4 = *(const floatx4*)(src + q), h4 = *(const floatx4*)(src + dh + q);
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          lo[q + x] = l4[x] + s_bias[hh * d + i + q + x];
          hi[q + x] = h4[x] + s_bias[hh * d + dh + i + q + x];
        }
      }
      const int pos = s_pos[row];
      if (e.inv_freq) {
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          // the hardware sine and cosine of r = frac(angle / 2 pi)
          float r = (float)pos * s_freq[i + q] * 0.15915494309189535f;
          r -= floorf(r);
          const float sn = __builtin_amdgcn_sinf(r), cs = __builtin_amdgcn_cosf(r);
          const float nlo = lo[q] * cs - hi[q] * sn, nhi = hi[q] * cs + lo[q] * sn;
          lo[q] = nlo;
          hi[q] = nhi;
        }
      }
      bf16x8 blo, bhi;
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        blo[q] = (bf16_t)lo[q];
        bhi[q] = (bf16_t)hi[q];
      }
      if (is_q) {
        bf16_t* dst = (bf16_t*)e.out + (size_t)m * e.ldo + (size_t)head * d + i;
        if (vec) {
          *(bf16x8*)dst = blo;
          *(bf16x8*)(dst + dh) = bhi;
        } else {
          for (int q = 0; q < 8; ++q) {
            dst[q] = blo[q];
            dst[dh + q] = bhi[q];
          }
        }
      } else {
        bf16_t* dst = e.kcache + ((size_t)s_page[row] * e.nkv + (head - e.nq)) * (size_t)e.page_size * d;
        const int off = pos % e.page_size;
        *(bf16x8*)(dst + kcache_index(off, i, d)) = blo;
        *(bf16x8*)(dst + kcache_index(off, i + dh, d)) = bhi;
      }
    }
    // v heads.  In the value order four consecutive keys of one number of d lie next to each
    // other, and the numbers of a 16-wide block of d after one another: four rows that are
    // four consecutive positions of one request, the first a multiple of four, put four
    // numbers of a head into 32 consecutive bytes of the page.  The rows of the tile are
    // taken in fours from the first row on whose position is a multiple of four if the tile
    // continues as its first row begins (a prompt from its start does; so does a portion
    // that follows the rows of decoding requests, from its second tile on); a unit of work
    // is such a group of rows by four numbers.  Groups that are not four positions in a row
    // of one request (and the rows before the first group and after the last) store number
    // by number: 2 bytes each, which memory has to merge into what it holds; a tile of
    // value heads stored so finished long after the others.
    const int hv0 = max(0, e.nq + e.nkv - head0), hv1 = min(heads, e.nq + 2 * e.nkv - head0);
    if (e.vcache && hv1 > hv0) {
      const int nv = hv1 - hv0, chunks = d >> 2;
      const int shift = (4 - (s_pos[0] & 3)) & 3;
      const size_t per_page = (size_t)e.page_size * d;
      for (int u = tid; u < (BM / 4 + 1) * nv * chunks; u += NT) {
        const int jc = u % chunks, t = u / chunks, hh = hv0 + t % nv, r0 = shift - 4 + 4 * (t / nv);
        const int dd0 = jc * 4, head = head0 + hh;
        const float* bias = s_bias + hh * d + dd0;
        bool together = r0 >= 0 && r0 + 3 < BM && m0 + r0 + 3 < M;
        if (together) {
          const int pos0 = s_pos[r0];
          together = (pos0 & 3) == 0;
#pragma unroll
          for (int k = 1; k < 4; ++k) together = together && s_pos[r0 + k] == pos0 + k && s_page[r0 + k] == s_page[r0];
        }
        if (together) {
          bf16x8 w0, w1;
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const floatx4 v4 = *(const floatx4*)(Cs + (r0 + k) * C_STRIDE + hh * d + dd0);
            w0[k] = (bf16_t)(v4[0] + bias[0]);
            w0[4 + k] = (bf16_t)(v4[1] + bias[1]);
            w1[k] = (bf16_t)(v4[2] + bias[2]);
            w1[4 + k] = (bf16_t)(v4[3] + bias[3]);
          }
          bf16_t* dst = e.vcache + ((size_t)s_page[r0] * e.nkv + (head - e.nq - e.nkv)) * per_page +
                        vcache_index(s_pos[r0] % e.page_size, dd0, d);
          *(bf16x8*)dst = w0;
          *(bf16x8*)(dst + 8) = w1;
        } else {
          for (int k = 0; k < 4; ++k) {
            const int row = r0 + k;
            if (row < 0 || row >= BM || m0 + row >= M) continue;
            const floatx4 v4 = *(const floatx4*)(Cs + row * C_STRIDE + hh * d + dd0);
            bf16_t* dst = e.vcache + ((size_t)s_page[row] * e.nkv + (head - e.nq - e.nkv)) * per_page;
            const int off = s_pos[row] % e.page_size;
#pragma unroll
            for (int x = 0; x < 4; ++x) dst[vcache_index(off, dd0 + x, d)] = (bf16_t)(v4[x] + bias[x]);
          }
        }
      }
    }
  }
}

// QKV: what the epilogue needs from global memory per row of the tile (position, and the page of that
// position for the tiles that hold k or v heads) and per column (bias, rotary frequencies).  `ask`, before
// the product's first loads: the position, the request and the vectors; `page`, behind those loads: the
// page, which needs the two; `put`, after the product: into LDS.  Nothing waits for a trip to memory
// before the product's own first tiles are on their way (put into LDS at once, position, request and page
// were two trips in a row before them: 512 rows of 1152 x 896 13.5 us, 12.6 now).  The tiles of two groups of waves
// alone ask for the page before their first loads: one trip that their products of 50 us and more do not show (700 to 2,560
// rows of 4608 x 3584, 2560 x 2048, 1152 x 896 and 6144 x 4096 the other way round: the same within 1 %).
template <int BM, int BN, int NT>
struct QkvRows {
  static_assert(BM <= NT && BN <= 2 * NT && NT >= 128, "a row, two columns and a frequency a thread");
  int pos, at, page_no;
  float freq, bias[2];
  __device__ __forceinline__ void ask(const EpiArgs& e, int m0, int n0, int M, int N, int tid) {
    const int m = min(m0 + min(tid, BM - 1), M - 1);
    pos = e.positions[m];
    at = e.kcache && n0 + BN > e.nq * e.d ? e.row_req[m] : -1;
    freq = e.inv_freq && tid < (e.d >> 1) ? e.inv_freq[tid] : 0.f;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int n = n0 + tid + i * NT;
      bias[i] = e.bias && tid + i * NT < BN && n < N ? load_vec(e.bias, e.bias_bf16, n) : 0.f;
    }
  }
  __device__ __forceinline__ void page(const EpiArgs& e) {
    page_no = at >= 0 ? e.table[(size_t)at * e.table_stride + pos / e.page_size] : 0;
  }
  __device__ __forceinline__ void put(int tid, int* s_pos, int* s_page, float* s_freq, float* s_bias) const {
    if (tid < BM) {
      s_pos[tid] = pos;
      s_page[tid] = page_no;
    }
    if (tid < 128) s_freq[tid] = freq;
#pragma unroll
    for (int i = 0; i < 2; ++i)
      if (tid + i * NT < BN) s_bias[tid + i * NT] = bias[i];
  }
};

// ============================================================ bf16, tiled
template <int BM, int BN, int BK, int WM, int WN, int EPI, bool GROUPED = false>
__global__ __launch_bounds__(64 * WM * WN) void gemm_bf16_tiled(const bf16_t* __restrict__ A,
                                                        const bf16_t* __restrict__ W, EpiArgs e, int M,
                                                        int N, int K) {
  constexpr int LDS_STRIDE = BK + 16;        // padded rows: the fragment reads of a wave spread evenly over the banks
  constexpr int NT = 64 * WM * WN;           // threads: WM x WN waves
  constexpr int WTM = BM / WM, WTN = BN / WN;  // wave tile
  constexpr int TM = WTM / 16, TN = WTN / 16;
  constexpr int KCH = BK / 8;                // 16-byte chunks in a row of a tile
  constexpr int A_CHUNKS = (BM * KCH + NT - 1) / NT;    // chunks of x per thread (past the tile's last: that one again)
  constexpr bool EVEN = BM * KCH % NT == 0;
  static_assert(BM * KCH >= NT, "tile too small");
  // three stages of LDS for x: the tile after the next is put in while this one is
  // multiplied and the next one's fragments are read, one barrier per tile
  constexpr int A_STAGE = BM * LDS_STRIDE;
  // (one array: after the last tile it holds the block's results for the epilogue)
  constexpr int C_STRIDE = BN + 4;           // floats per row of the result tile in LDS
  constexpr size_t STAGE_BYTES = (size_t)(3 * A_STAGE) * sizeof(bf16_t);
  constexpr size_t C_BYTES = (size_t)BM * C_STRIDE * sizeof(float);
  __shared__ __attribute__((aligned(16))) char smem[EPI != EPI_QKV || STAGE_BYTES > C_BYTES ? STAGE_BYTES : C_BYTES];
  bf16_t* As2 = (bf16_t*)smem;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave / WN, wn = wave % WN;
  // Blocks are handed to the 8 dies (each with an L2 of its own) in turn.  Give
  // every die a band of neighbouring column tiles, rows running fastest, so that
  // what its blocks read at one time is a few column tiles of W and the rows of x.
  int bx = blockIdx.x, by = blockIdx.y;
  {
    const int gx = gridDim.x, gy = gridDim.y, total = gx * gy;
    const int lin = by * gx + bx;
    const int whole = total & ~7;            // the last few blocks (total % 8) keep their place
    const int mapped = lin < whole ? (lin & 7) * (whole >> 3) + (lin >> 3) : lin;
    bx = mapped / gy;
    by = mapped - bx * gy;
  }
  const int m0 = by * BM, n0 = bx * BN;
  const int c = lane & 15, g = lane >> 4;
  if constexpr (GROUPED) {
    const int member = e.g_tile[by];       // (the same for the whole block: all leave together)
    if (member < 0) return;
    W += (size_t)member * e.g_w_stride;
  }

  constexpr bool QKV = EPI == EPI_QKV;
  __shared__ int s_pos[QKV ? BM : 1], s_page[QKV ? BM : 1];
  __shared__ float s_freq[QKV ? 128 : 1], s_bias[QKV ? BN : 1];
  QkvRows<QKV ? BM : 64, QKV ? BN : 64, QKV ? NT : 128> rows;
  if constexpr (QKV) rows.ask(e, m0, n0, M, N, tid);

  floatx4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

  // Memory latency is several times the time a tile takes to multiply, so PD tiles
  // are on their way at any time: a ring of register buffers, refilled as soon as a
  // buffer has been put into LDS.
  constexpr int PD = (A_CHUNKS + BN * KCH / NT) <= 4 ? 4 : 3;
  bf16x8 ra[PD][A_CHUNKS];
  // every wave reads the B fragments of its columns straight from the packed W into
  // registers; only x goes through LDS
  bf16x8 rbd[PD][BK / 32][TN];
  const bf16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};

  // Loads are unconditional (a load under a branch makes the compiler wait for every
  // load in flight where the branch ends).  Rows of x past M and pieces past K read
  // a valid piece instead: they meet zeros of the padded W or land in rows nobody
  // stores.  W is packed in fragment order: the 64 columns of a strip of 16 rows
  // are consecutive memory (1 KB per 32 columns), a thread reading 16 bytes of it.
  const int T = (K + 31) >> 5, nstrips = (N + 15) >> 4;
  int gathered[GROUPED ? A_CHUNKS : 1];      // GROUPED: the rows of x this thread's pieces come from
  if constexpr (GROUPED) {
#pragma unroll
    for (int i = 0; i < A_CHUNKS; ++i) {
      const int m = min(m0 + (EVEN ? tid + i * NT : min(tid + i * NT, BM * KCH - 1)) / KCH, M - 1);
      gathered[i] = e.g_rows ? max(e.g_rows[m], 0) : m;
    }
  }
  auto fetch = [&](int slot, int k0) {
#pragma unroll
    for (int i = 0; i < A_CHUNKS; ++i) {
      const int ch = EVEN ? tid + i * NT : min(tid + i * NT, BM * KCH - 1), row = ch / KCH, kc = (ch % KCH) * 8;
      const int m = GROUPED ? gathered[i] : min(m0 + row, M - 1), k = min(k0 + kc, K - 8);
      ra[slot][i] = *(const bf16x8*)(A + (size_t)m * K + k);
    }
  };
  auto fetch_b = [&](int slot, int k0) {
#pragma unroll
    for (int ks = 0; ks < BK / 32; ++ks)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int step = (k0 >> 5) + ks;
        const int strip = min(((n0 + wn * WTN) >> 4) + j, nstrips - 1);
        const bf16x8 v = *(const bf16x8*)(W + ((size_t)strip * T + min(step, T - 1)) * 512 + lane * 8);
        rbd[slot][ks][j] = step < T ? v : zero;
      }
  };
  auto stash = [&](int slot, int stage) {
    bf16_t* As = As2 + stage * A_STAGE;
#pragma unroll
    for (int i = 0; i < A_CHUNKS; ++i) {
      const int ch = EVEN ? tid + i * NT : min(tid + i * NT, BM * KCH - 1), row = ch / KCH, kc = (ch % KCH) * 8;
      *(bf16x8*)(As + row * LDS_STRIDE + kc) = ra[slot][i];
    }
  };

  // this block's K tiles: all of them, or (PART) its group's share starting at tile kt0
  // (tiles past the share are fetched like any other and never multiplied)
  int nk = (K + BK - 1) / BK, kt0 = 0;
  if constexpr (EPI == EPI_PART) {
    kt0 = (int)blockIdx.z * e.kt_per_split;
    nk = max(0, min(nk - kt0, e.kt_per_split));
    e.out = (float*)e.out + (size_t)blockIdx.z * e.part_stride;
    if (blockIdx.z > 0) e.bias = nullptr;
  }
  const int kbase = kt0 * BK;
#pragma unroll
  for (int p = 0; p < PD; ++p) {      // past K: zeros for W
    fetch(p, kbase + p * BK);
    fetch_b(p, kbase + p * BK);
  }
  if constexpr (QKV) rows.page(e);
  // Tile t lies in stage t % 3.  It is put there during tile t - 2, and its fragments are
  // read into registers half a tile ahead of their products (those of its first 32
  // columns of K during the second half of tile t - 1), so that the reads of LDS pass
  // behind the matrix instructions of the half before: with one wave on a SIMD nothing
  // else would hide them.  One barrier per tile: what is overwritten during tile t (stage
  // (t + 2) % 3) was last read during tile t - 1.
  auto frags = [&](bf16x8 (&a)[TM], int stage, int ks) {
    const bf16_t* As = As2 + stage * A_STAGE;
#pragma unroll
    for (int i = 0; i < TM; ++i)
      a[i] = *(const bf16x8*)(As + (wm * WTM + i * 16 + c) * LDS_STRIDE + ks * 32 + g * 8);
  };
  static_assert(BK == 64, "two half tiles");
  bf16x8 a0[TM], a1[TM];
  stash(0, 0);
  fetch(0, kbase + PD * BK);
  if (nk > 1) stash(1 % PD, 1);
  fetch(1 % PD, kbase + (PD + 1) * BK);
  __syncthreads();
  frags(a0, 0, 0);
  int stage = 0;                                 // t % 3
  for (int kt = 0; kt < nk; kt += PD) {
#pragma unroll
    for (int p = 0; p < PD; ++p) {
      const int t = kt + p;
      const bool live = t < nk;
      const int p2 = (p + 2) % PD;              // ring slot of tile t + 2 (a constant once unrolled)
      const int stage1 = stage == 2 ? 0 : stage + 1, stage2 = stage1 == 2 ? 0 : stage1 + 1;
      if (live) {
        frags(a1, stage, 1);
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(rbd[p][0][j], a0[i], acc[i][j], 0, 0, 0);
        frags(a0, stage1, 0);
        if (t + 2 < nk) stash(p2, stage2);
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(rbd[p][1][j], a1[i], acc[i][j], 0, 0, 0);
        __syncthreads();
      }
      // (outside the branch, like every load of the loop: see above)
      fetch(p2, kbase + (t + 2 + PD) * BK);
      fetch_b(p, kbase + (t + PD) * BK);
      stage = stage1;
    }
  }

  // ---- epilogue
  if constexpr (QKV) {      // through LDS, where a thread finds both halves of its pairs
    // (every live tile ended with a barrier, so the stages are free)
    float* Cs = (float*)smem;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
        *(floatx4*)(Cs + (wm * WTM + i * 16 + c) * C_STRIDE + wn * WTN + j * 16 + g * 4) = acc[i][j];
    rows.put(tid, s_pos, s_page, s_freq, s_bias);
    __syncthreads();
    tile_epilogue<BM, BN, NT, EPI>(Cs, e, m0, n0, M, N, tid, s_pos, s_page, s_freq, s_bias);
  } else {
    register_epilogue<TM, TN, EPI>(acc, e, m0 + wm * WTM, n0 + wn * WTN, M, N, c, g);
  }
}

// ============================================================ bf16, 256 x 256 by two groups of waves
// The largest products.  Eight waves, each with a 128 x 64 part of a 256 x 256 tile; both
// operands come by direct loads from global memory into LDS (no registers in between).  The
// waves form two groups with a wave on every SIMD each, half a step (32 of the inner size)
// apart: between two barriers one group reads its twelve fragments and issues its
// loads while the other issues its 32 MFMAs, then they change roles, so that the reads of
// LDS and the matrix instructions of a compute unit overlap by construction and not by
// the luck of the scheduler (all eight waves in step: 975 TF/s on 8192 x 37888 x 3584,
// the groups apart: 1065; the 128 x 256 tile of the kernel above: 966).  A block fills a
// compute unit; the q/k/v epilogue takes the two halves of the rows through LDS one after the other.
//
// What bounds it is the way of x to the compute units, line by line: with 1 KB of consecutive
// memory a load in place of rows the same loop is 20 % faster.  W has such tiles (packed:
// one load, one fragment, in a ring of four steps).  A load of x takes 8 rows of 128 bytes, two
// steps of the inner size, neighbouring lanes in the same row, so that a load touches eight lines
// and takes them whole; with one fragment a load (16 rows of 64 bytes, neighbouring lanes in
// different rows) it touched 16 half lines, each by four lanes far apart, and 2367 rows of 37888 x 3584 took 597 us instead of 522,
// of 3584 x 18944 322 instead of 286, 2048 of 22016 x 2048 191 instead of 169, of 3584 x 18944
// 317 instead of 273 (16 rows of 64 bytes with neighbouring lanes in one row: 539, 280, 178, 319).
// A piece of x is half of the tile's rows of two steps: NG of them in a ring, one fetched a step,
// each by the step NG - 2 later at the latest.  Six make the 256 x 256 tile's LDS full; the tile
// that writes the cache needs room for positions and biases and has five.
// In LDS a row of a load lies as 128 bytes, its eight pieces of 16 bytes exchanged by the row's
// number: a fragment read, 16 rows of one piece each, then meets every bank once.
// A ring of five or six steps of W instead of four, or blocks that begin at different steps of the
// inner size (to spread the channels of memory), change nothing; four waves of 128 x 128, whose
// fragments for the next step are read between this one's MFMAs, are as fast and no faster.
//
// The direct loads are written in assembly: the compiler then knows nothing of them, the
// waits (vmcnt) are placed by hand, and the loop holds no other load that it would count.
//
// BM = 192 is the same with 96 x 64 a wave, for steps whose rows fill tiles of 192 better
// than tiles of 256 (576 rows: three tiles instead of three of which one is a quarter full).
template <int BM, int EPI>
__global__ __launch_bounds__(512) void gemm_bf16_pingpong(const bf16_t* __restrict__ A,
                                                          const bf16_t* __restrict__ W, EpiArgs e, int M,
                                                          int N, int K) {
  static_assert(BM == 256 || BM == 192, "a wave has 128 or 96 rows");
  constexpr int BN = 256, NT = 512, HALF = 128;
  constexpr int TM = BM / 32;                           // blocks of 16 rows of a wave
  constexpr int NG = BM == 256 && EPI == EPI_QKV ? 5 : 6;      // pieces of x in LDS
  constexpr int PIECE = BM / 2 * 128;                   // bytes: half of the rows, two steps
  constexpr int W_AT = NG * PIECE, W_STEP = (BN / 16) * 1024;
  constexpr int C_STRIDE = BN + 4;
  constexpr size_t C_BYTES = (size_t)HALF * C_STRIDE * sizeof(float);
  __shared__ __attribute__((aligned(1024))) char smem[EPI == EPI_QKV && C_BYTES > W_AT + 4 * W_STEP ? C_BYTES : W_AT + 4 * W_STEP];

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = wave >> 2;                             // waves 0-3 and 4-7: one of each on every SIMD
  const int wm = wave & 1, wn = ((wave >> 1) & 1) | (grp << 1);   // rows wm * BM / 2, columns wn * 64
  int bx = blockIdx.x, by = blockIdx.y;
  {                                                      // a band of column tiles per die, as above
    const int gx = gridDim.x, gy = gridDim.y, total = gx * gy;
    const int lin = by * gx + bx;
    const int whole = total & ~7;
    const int mapped = lin < whole ? (lin & 7) * (whole >> 3) + (lin >> 3) : lin;
    bx = mapped / gy;
    by = mapped - bx * gy;
  }
  const int m0 = by * BM, n0 = bx * BN;
  const int c = lane & 15, g = lane >> 4;

  constexpr bool QKV = EPI == EPI_QKV;
  __shared__ int s_pos[QKV ? BM : 1], s_page[QKV ? BM : 1];
  __shared__ float s_freq[QKV ? 128 : 1], s_bias[QKV ? BN : 1];
  QkvRows<QKV ? BM : 64, QKV ? BN : 64, QKV ? NT : 128> rows;
  if constexpr (QKV) rows.ask(e, m0, n0, M, N, tid);

  // Per step a wave fetches four times 1 KB (three times of x with BM = 192): the even waves of x,
  // the odd ones of W (so that both groups fetch both).  Rows past M, strips past N and numbers past K read a
  // valid place instead: they land in rows and columns that nobody stores, or meet the
  // zeros of the padded W.
  const int T = (K + 31) >> 5, nstrips = (N + 15) >> 4;
  const bool fetches_x = (wave & 1) == 0;
  const int quarter = wave >> 1;
  constexpr int NFX = BM / 64;                          // loads of a piece of x by each of its four waves
  unsigned off[2][4];                                   // bytes from the tile's rows of x (by half) or of W
  int shift[4];                                         // (of x) the numbers of k that `off` holds
  unsigned dst[4];
  const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (fetches_x) {
      const int b = min(quarter * NFX + i, BM / 16 - 1);
      shift[i] = ((lane & 7) ^ (((b & 1) << 2) | (lane >> 4))) * 8;
#pragma unroll
      for (int h = 0; h < 2; ++h)
        off[h][i] = ((unsigned)(min(m0 + h * (BM / 2) + b * 8 + (lane >> 3), M - 1) - m0) * (unsigned)K + shift[i]) * 2u;
      dst[i] = lds0 + b * 1024;
    } else {
      const int f = quarter * 4 + i;
      off[0][i] = (unsigned)(min((n0 >> 4) + f, nstrips - 1) - (n0 >> 4)) * (unsigned)T * 1024u + lane * 16u;
      dst[i] = lds0 + W_AT + f * 1024;
    }
  }
  const char* const xbase = (const char*)(A + (size_t)m0 * K);
  const char* const wbase = (const char*)(W + (size_t)(n0 >> 4) * T * 512);
  auto load_to_lds = [&](unsigned at, const char* base, unsigned to) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                 :
                 : "v"(at), "s"(base), "s"(to)
                 : "memory", "m0");
  };
  // this block's steps: all of them, or (PART) its group's share of the inner size from
  // step `first` on, whose sums go to the group's own piece of the output
  int first = 0, nk = T;
  if constexpr (EPI == EPI_PART) {
    first = (int)blockIdx.z * e.kt_per_split * 2;
    nk = max(0, min(T - first, e.kt_per_split * 2));
    e.out = (float*)e.out + (size_t)blockIdx.z * e.part_stride;
    if (blockIdx.z > 0) e.bias = nullptr;
  }
  // piece q of x: half q % 2 (given as a constant) of the rows, steps q and q + 1 of an even q
  auto fetch_x = [&](int q, int half, unsigned slot) {
    const int k = (first + (q & ~1)) * 32;
    if (k + 64 <= K) {
      const char* base = xbase + (size_t)k * 2;
#pragma unroll
      for (int i = 0; i < NFX; ++i) load_to_lds(off[half][i], base, dst[i] + slot);
    } else {
#pragma unroll
      for (int i = 0; i < NFX; ++i)
        load_to_lds(off[half][i] + (unsigned)(min(k + shift[i], K - 8) - shift[i]) * 2u, xbase, dst[i] + slot);
    }
  };
  auto fetch_w = [&](int stage, int step) {
    const char* base = wbase + (size_t)min(first + step, T - 1) * 1024;
#pragma unroll
    for (int i = 0; i < 4; ++i) load_to_lds(off[0][i], base, dst[i] + stage * W_STEP);
  };
  // What a wave waits for before a barrier: its reads of LDS, and of its loads those that the next
  // step reads: of W all but two steps; of x, before an even step, all but the pieces
  // after that step's two (an odd step reads the same pieces as the step before).
  auto wait_loads = [&](bool even_next) {
    if (!fetches_x) __builtin_amdgcn_s_waitcnt(0x0070 | 8);
    else if (even_next) __builtin_amdgcn_s_waitcnt(0x0070 | ((NG - 4) * NFX));
    else __builtin_amdgcn_s_waitcnt(0x0070 | 15);
  };

  floatx4 acc[TM][4];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  bf16x8 a[TM], b[4];

  // every wave passes the same barriers; nothing may move across one
  auto barrier = [&]() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
  };
  // Step t of W lies in stage t % 4, piece q of x in slot q % NG.  A wave's memory phase of step t reads its
  // fragments, issues its loads of W of step t + 3 (into the stage that both groups read last in
  // step t - 1, at least one barrier ago) or of piece t + NG - 2 of x (into the slot of piece t - 2, read
  // last in step t - 1 or t - 2) and waits for its own loads of step t + 1; the
  // barrier after the other group's same phase then says that step t + 1 is whole.
  if constexpr (QKV) rows.page(e);
  if (fetches_x) {
#pragma unroll
    for (int q = 0; q < NG - 2; ++q) fetch_x(q, q & 1, q * PIECE);
  } else {
#pragma unroll
    for (int q = 0; q < 3; ++q) fetch_w(q, q);
  }
  wait_loads(true);
  barrier();
  if (grp == 1) barrier();                               // the second group runs half a step behind
  unsigned read_at = wm * PIECE, write_at = (NG - 2) * PIECE;
  const int even_at = c * 128 + ((g ^ (c >> 1)) << 4), odd_at = c * 128 + (((4 + g) ^ (c >> 1)) << 4);
  for (int t0 = 0; t0 < nk; t0 += 4) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int t = t0 + u;
      if (t < nk) {                                      // (the same for every wave of the block)
        const char* ws = smem + W_AT + u * W_STEP;
        const char* xs = smem + read_at + ((u & 1) ? odd_at : even_at);
#pragma unroll
        for (int j = 0; j < 4; ++j) b[j] = *(const bf16x8*)(ws + (wn * 4 + j) * 1024 + lane * 16);
#pragma unroll
        for (int i = 0; i < TM; ++i) a[i] = *(const bf16x8*)(xs + i * 2048);
        if (fetches_x) fetch_x(t + NG - 2, (u + NG) & 1, write_at);
        else fetch_w((u + 3) & 3, t + 3);
        write_at = write_at == (NG - 1) * PIECE ? 0 : write_at + PIECE;
        if (u & 1) {
          read_at += 2 * PIECE;
          if (read_at >= NG * PIECE) read_at -= NG * PIECE;
        }
        wait_loads(u & 1);
        barrier();
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[j], a[i], acc[i][j], 0, 0, 0);
        barrier();
      }
    }
  }
  if (grp == 0) barrier();
  __builtin_amdgcn_s_waitcnt(0x0070);                    // the last loads (past K, never read) are in
  barrier();

  // ---- epilogue
  if constexpr (QKV) {      // the rows 0-127 of the tile through LDS, then the rest
    float* Cs = (float*)smem;
    rows.put(tid, s_pos, s_page, s_freq, s_bias);
    auto to_lds = [&](int part) {
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int row = wm * (BM / 2) + i * 16;             // of the tile
        if (row / HALF == part) {
#pragma unroll
          for (int j = 0; j < 4; ++j) *(floatx4*)(Cs + (row % HALF + c) * C_STRIDE + wn * 64 + j * 16 + g * 4) = acc[i][j];
        }
      }
      __syncthreads();
    };
    to_lds(0);
    tile_epilogue<HALF, BN, NT, EPI>(Cs, e, m0, n0, M, N, tid, s_pos, s_page, s_freq, s_bias);
    __syncthreads();
    to_lds(1);
    tile_epilogue<BM - HALF, BN, NT, EPI>(Cs, e, m0 + HALF, n0, M, N, tid, s_pos + HALF, s_page + HALF, s_freq, s_bias);
  } else {
    register_epilogue<TM, 4, EPI>(acc, e, m0 + wm * (BM / 2), n0 + wn * 64, M, N, c, g);
  }
}

// ============================================================ bf16, small tiles by direct loads
// Small products: four waves 2 x 2 on a tile of 64 x 64, both operands by direct loads into LDS as in the kernel
// above (x 8 rows of 128 bytes a load, W by fragments), in stages of 64 of the inner size, three of them.  What
// bounds such a product is its few blocks' way through launch, first trip to memory, K tiles and epilogue; here no
// operand passes through registers on its way, every stage but one is on its way at any time, a stage
// takes one barrier, and three blocks of the 64 x 64 tile (48 KB) share a unit.  Against the same tile with x by way of registers and W
// straight into them, over 182 products of 24 to 2,048 rows whole and in pieces: 18 % less; 512 rows of 896 x 896 8.9 -> 7.8 us,
// 2,048 11.7 -> 9.2, 512 of 896 x 4864 in four pieces 15.6 -> 12.6, 64 of 3584 x 18944 in eight 39.6 -> 30.8.  Four and five stages (two blocks a
// unit): 4 % slower.  Larger tiles of this kind with four waves: 64 x 128 (three stages) is slower than the tile above with many
// rows (512 of 9728 x 896 24.8 against 21.4) and faster in pieces of few rows only (64 of 3584 x 18944 28.2 against 32.4), 128 x 160
// and 128 x 256 as fast as theirs (128 of 37888 x 3584 71.8 against 73.7): not kept.
// With eight waves, 4 x 2: 128 x 128 and 128 x 192 in three stages (one block a unit) and 192 x 128 in two (two blocks a
// unit, the end of one behind the loop of the other); which product takes them and what they measure: direct_tile.  What bounds
// them is LDS (128 x 192: 128 KB of fragments a stage, 1,024 clocks beside 768 of matrix instructions) and, of 16 us
// that 512 rows of 9728 x 896 take, the half that launch, first trip to memory and epilogue are.
template <int EPI, int BM = 64, int BN = 64, int NST = 3, int WM = 2, int WN = 2, int WAVES = 1>
__global__ __launch_bounds__(64 * WM * WN, WAVES) void gemm_bf16_ring(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W,
                                                                      EpiArgs e, int M, int N, int K) {
  constexpr int NW = WM * WN, NT = 64 * NW, WTM = BM / WM, WTN = BN / WN, TM = WTM / 16, TN = WTN / 16;
  constexpr int XL = BM / 8, WL = BN / 8, NL = (XL + WL) / NW;     // loads of 1 KB of a stage: of x, of W, of one wave
  static_assert((XL + WL) % NW == 0 && WTM % 16 == 0 && WTN % 16 == 0 && NL * (NST - 2) < 64, "shape");
  constexpr int STAGE = (XL + WL) * 1024, W_AT = XL * 1024;
  constexpr int C_STRIDE = BN + 4;
  constexpr size_t C_BYTES = (size_t)BM * C_STRIDE * sizeof(float);
  __shared__ __attribute__((aligned(1024))) char smem[EPI == EPI_QKV && C_BYTES > NST * STAGE ? C_BYTES : NST * STAGE];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % WM, wn = wave / WM;
  int bx = blockIdx.x, by = blockIdx.y;
  {                                                      // a band of column tiles per die, as above
    const int gx = gridDim.x, gy = gridDim.y, total = gx * gy;
    const int lin = by * gx + bx;
    const int whole = total & ~7;
    const int mapped = lin < whole ? (lin & 7) * (whole >> 3) + (lin >> 3) : lin;
    bx = mapped / gy;
    by = mapped - bx * gy;
  }
  const int m0 = by * BM, n0 = bx * BN;
  const int c = lane & 15, g = lane >> 4;
  constexpr bool QKV = EPI == EPI_QKV;
  __shared__ int s_pos[QKV ? BM : 1], s_page[QKV ? BM : 1];
  __shared__ float s_freq[QKV ? 128 : 1], s_bias[QKV ? BN : 1];
  QkvRows<QKV ? BM : 64, QKV ? BN : 64, NT> rows;
  if constexpr (QKV) rows.ask(e, m0, n0, M, N, tid);
  const int T = (K + 31) >> 5, nstrips = (N + 15) >> 4;
  unsigned off[NL];
  int shift[NL];
  const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
  // Load i of a wave is number wave + NW i of the stage: the first XL take 8 rows of x each, the others a step
  // of a strip of W.  Rows past M, strips past N and numbers past K read a valid place instead.
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    const int b = wave + NW * i;
    if (NW * i < XL) {                    // (XL % NW == 0: the same for all waves)
      shift[i] = ((lane & 7) ^ (((b & 1) << 2) | (lane >> 4))) * 8;
      off[i] = ((unsigned)(min(m0 + b * 8 + (lane >> 3), M - 1) - m0) * (unsigned)K + shift[i]) * 2u;
    } else {
      const int f = (b - XL) >> 1;
      shift[i] = (b - XL) & 1;
      off[i] = (unsigned)(min((n0 >> 4) + f, nstrips - 1) - (n0 >> 4)) * (unsigned)T * 1024u + lane * 16u;
    }
  }
  static_assert(XL % NW == 0, "x first");
  const char* const xbase = (const char*)(A + (size_t)m0 * K);
  const char* const wbase = (const char*)(W + (size_t)(n0 >> 4) * T * 512);
  auto load_to_lds = [&](unsigned at, const char* base, unsigned to) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(at), "s"(base), "s"(to) : "memory", "m0");
  };
  int first = 0, nk = T;
  if constexpr (EPI == EPI_PART) {
    first = (int)blockIdx.z * e.kt_per_split * 2;
    nk = max(0, min(T - first, e.kt_per_split * 2));
    e.out = (float*)e.out + (size_t)blockIdx.z * e.part_stride;
    if (blockIdx.z > 0) e.bias = nullptr;
  }
  auto fetch = [&](int stage, unsigned slot) {
    const int t = first + 2 * stage, k = t * 32;
    const bool whole = k + 64 <= K;
    const char* xb = whole ? xbase + (size_t)k * 2 : xbase;
    const char* w0 = wbase + (size_t)min(t, T - 1) * 1024;
    const char* w1 = wbase + (size_t)min(t + 1, T - 1) * 1024;
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const unsigned to = lds0 + slot + (wave + NW * i) * 1024;
      if (NW * i < XL) {
        if (whole) load_to_lds(off[i], xb, to);
        else load_to_lds(off[i] + (unsigned)(min(k + shift[i], K - 8) - shift[i]) * 2u, xb, to);
      } else {
        load_to_lds(off[i], ((wave + NW * i - XL) & 1) ? w1 : w0, to);
      }
    }
  };
  auto barrier = [&]() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
  };
  constexpr int VM = NL * (NST - 2);
  auto wait_loads = [&]() { __builtin_amdgcn_s_waitcnt(0x0070 | (VM & 15) | ((VM >> 4) << 14)); };
  floatx4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  bf16x8 a[2][TM], b[2][TN];
  const int at[2] = {c * 128 + ((g ^ (c >> 1)) << 4), c * 128 + (((4 + g) ^ (c >> 1)) << 4)};
  auto frags = [&](int h, unsigned slot) {
    const char* xs = smem + slot + wm * WTM * 128 + at[h];
    const char* ws = smem + slot + W_AT + (wn * TN * 2 + h) * 1024 + lane * 16;
#pragma unroll
    for (int j = 0; j < TN; ++j) b[h][j] = *(const bf16x8*)(ws + j * 2048);
#pragma unroll
    for (int i = 0; i < TM; ++i) a[h][i] = *(const bf16x8*)(xs + i * 2048);
  };
  auto products = [&](int h) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[h][j], a[h][i], acc[i][j], 0, 0, 0);
  };
  fetch(0, 0);
  if constexpr (QKV) rows.page(e);      // (waits for the first stage too, which has to come first in any case)
#pragma unroll
  for (int s = 1; s < NST; ++s) fetch(s, s * STAGE);
  asm volatile("s_waitcnt vmcnt(%0)" :: "n"(NL * (NST - 1)) : "memory");
  barrier();
  // Stage s (steps 2 s and 2 s + 1) lies in slot s % NST.  Its first half's fragments are read during the stage
  // before, its second half's while the first is multiplied; behind the one barrier of a stage it has been
  // read by all, the next one is there, and stage s + NST is asked for into its place.
  unsigned slot = 0;
  frags(0, 0);
  for (int t = 0; t < nk; t += 2) {
    const unsigned next = slot == (NST - 1) * STAGE ? 0 : slot + STAGE;
    frags(1, slot);
    products(0);
    wait_loads();                       // stage t / 2 + 1 is there, this stage is read
    barrier();
    fetch((t >> 1) + NST, slot);
    frags(0, next);
    if (t + 1 < nk) products(1);
    slot = next;
  }
  __builtin_amdgcn_s_waitcnt(0x0070);                    // the last loads (past K, never read) are in
  barrier();
  if constexpr (QKV) {
    float* Cs = (float*)smem;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
        *(floatx4*)(Cs + (wm * WTM + i * 16 + c) * C_STRIDE + wn * WTN + j * 16 + g * 4) = acc[i][j];
    rows.put(tid, s_pos, s_page, s_freq, s_bias);
    __syncthreads();
    tile_epilogue<BM, BN, NT, EPI>(Cs, e, m0, n0, M, N, tid, s_pos, s_page, s_freq, s_bias);
  } else {
    register_epilogue<TM, TN, EPI>(acc, e, m0 + wm * WTM, n0 + wn * WTN, M, N, c, g);
  }
}

// ================================================================ float32
// Debug interface: 1 = products of many rows by the plain FMA kernel instead of the matrix
// cores (tests compare the two).
static int g_f32_fma = 0;
extern "C" void llmlab_debug_f32_fma(int on) { g_f32_fma = on; }

// BM x BN outputs per block of 256 threads (16 x 16); thread (ty, tx) owns the TM = BM/16
// rows ty*TM + i and the TN = BN/16 columns tx + 16*j, so for SWIGLU columns j = 0, 2, ..
// are gate and j = 1, 3, .. the up values of the same outputs.  K steps of 8 through LDS
// (both operands transposed, so that a thread reads its TM rows as vectors); the next
// step's numbers are on their way from memory while this one is multiplied.  Plain FMAs.
template <int EPI, int BM, int BN>
__global__ __launch_bounds__(256) void gemm_f32_kernel(const float* __restrict__ A,
                                                        const float* __restrict__ W, EpiArgs e, int M,
                                                        int N, int K, int vec) {
  constexpr int BK = 8, TM = BM / 16, TN = BN / 16;
  constexpr int LA = BM * BK / 256, LB = BN * BK / 256;      // numbers per thread and step: 2 or 4
  __shared__ __attribute__((aligned(16))) float As[BK][BM + 4];
  __shared__ __attribute__((aligned(16))) float Bs[BK][BN + 4];
  const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  float acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = 0.f;
  // a thread fetches LA (LB) consecutive k of one row of x (of W)
  const int arow = tid / (BK / LA), ak = (tid % (BK / LA)) * LA;
  const int brow = tid / (BK / LB), bk = (tid % (BK / LB)) * LB;
  const float* ap = A + (size_t)min(m0 + arow, M - 1) * K;
  const float* bp = W + (size_t)min(n0 + brow, N - 1) * K;
  float ra[LA], rb[LB];
  auto fetch = [&](int k0) {
    if (vec && k0 + BK <= K) {
      if constexpr (LA == 4) {
        const floatx4 v = *(const floatx4*)(ap + k0 + ak);
        ra[0] = v[0]; ra[1] = v[1]; ra[2] = v[2]; ra[3] = v[3];
      } else {
        ra[0] = ap[k0 + ak]; ra[1] = ap[k0 + ak + 1];
      }
      if constexpr (LB == 4) {
        const floatx4 v = *(const floatx4*)(bp + k0 + bk);
        rb[0] = v[0]; rb[1] = v[1]; rb[2] = v[2]; rb[3] = v[3];
      } else {
        rb[0] = bp[k0 + bk]; rb[1] = bp[k0 + bk + 1];
      }
    } else {
#pragma unroll
      for (int x = 0; x < LA; ++x) ra[x] = k0 + ak + x < K ? ap[k0 + ak + x] : 0.f;
#pragma unroll
      for (int x = 0; x < LB; ++x) rb[x] = k0 + bk + x < K ? bp[k0 + bk + x] : 0.f;
    }
  };
  fetch(0);
  for (int k0 = 0; k0 < K; k0 += BK) {
    __syncthreads();
#pragma unroll
    for (int x = 0; x < LA; ++x) As[ak + x][arow] = ra[x];
#pragma unroll
    for (int x = 0; x < LB; ++x) Bs[bk + x][brow] = rb[x];
    __syncthreads();
    if (k0 + BK < K) fetch(k0 + BK);
#pragma unroll
    for (int kk = 0; kk < BK; ++kk) {
      float a[TM], b[TN];
#pragma unroll
      for (int i = 0; i < TM; i += 4) {
        const floatx4 v = *(const floatx4*)&As[kk][ty * TM + i];
        a[i] = v[0]; a[i + 1] = v[1]; a[i + 2] = v[2]; a[i + 3] = v[3];
      }
#pragma unroll
      for (int j = 0; j < TN; ++j) b[j] = Bs[kk][tx + 16 * j];
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
    }
  }
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int m = m0 + ty * TM + i;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      if constexpr (EPI == EPI_SWIGLU) {
        if (j & 1) continue;
        const int nb = n0 + 16 * j;
        const int o = (nb >> 5) * 16 + tx;
        if (o < e.n_out) ((float*)e.out)[(size_t)m * e.ldo + o] = pair_exact_f(acc[i][j], acc[i][j + 1], e);
      } else {
        const int n = n0 + tx + 16 * j;
        if (n < N) epi_store<float, EPI>(e, m, n, acc[i][j]);
      }
    }
  }
}

// Many rows in float32: the products are taken by the bfloat16 matrix instructions without giving
// up a bit of the operands.  A float32 number of 2^-110 to 3.39e38 is the sum of three bfloat16 numbers, x = h + m + l (h =
// x rounded to nearest, m = x - h rounded, l the rest: 24 bits of significand in three times 8, the
// differences exact), and x w = h_x h_w + h_x m_w + m_x h_w + m_x m_w + h_x l_w + l_x h_w up to terms below
// 2^-24 of |x w|, less than what one rounding of a 32-bit sum costs (three of the nine part products are left out: about
// 2^-26 of a product, so that a product by itself is within two roundings, not one).  Every bfloat16 product is
// exact in float32 and the sums are float32; an instruction adds 32 of them where
// v_mfma_f32_32x32x2_f32 adds 2, so fewer roundings meet in a sum (relative error of a product of
// normal numbers against 64 bits: inner size 896 4.5e-7, 5.4e-7 with the float32 instructions; 4,864 1.1e-6
// and 1.25e-6, 6e-7 in three pieces).
//
// Where all numbers of W are bfloat16 numbers, as in checkpoints that were trained and kept in bfloat16, m_w and l_w are
// zero and with them three of the six products.  A block takes W for such until it meets another number, and all parts from
// that step on: a thread that puts such a number down leaves its step in LDS, where every wave looks before it multiplies a
// step.  Nothing is kept between calls, and both ways give the same sums to the bit (the
// terms left out are zeros).  (Relative error of a prompt's logits, 1,531 tokens of the 0.5B shape, mean of eight seeds:
// 2.13e-6; 2.63e-6 before the small products had sums of their own.  1,531 rows of 9728 x 896 with such a number in the last
// step 95 us, without one 91, of such numbers 146; when the block found out at the end and started over 209.)
//
// BM x BN outputs per block of WM x WN waves, steps of 32 of the inner size.  A thread
// fetches eight numbers of a row as they lie in memory, two steps ahead (four neighbouring lanes 64 consecutive bytes: with
// neighbouring lanes in different rows the way of the loads to the compute unit bounded the small tile, 1,531 rows
// of 1152 x 896 34 us against 23), splits them in registers and puts the parts down in LDS in fragment order, [16
// rows][part][64 places][8], where lane (c, g) of a fragment holds the numbers 4 g .. 4 g + 3 and 16 + 4 g .. of its row's 32
// (the order inside a step is free, both operands share it).  Two stages of LDS: the next step is put down
// in this one.  With eight waves they form two groups, a wave of each on every SIMD, half a step apart: between two barriers
// one group reads its fragments and splits and puts down its pieces while the other issues its matrix instructions
// (128 x 256, one part: 2,550 clocks a step where all waves in step took 4,000; not with three parts in the 128 x 128
// tile, whose splitting takes longer than its products: 3,100 against 2,900).  The product is taken transposed, C^T = W
// x^T, so that a lane holds four neighbouring columns of a row, and for SWIGLU the gate and the up
// value of an output.
//
// What bounds it: LDS (128 x 256, one part: 128 KB of reads and 40 of writes a step, 1,850 clocks at the rates of LDS,
// 1,630 of matrix instructions).  Back to back, with one / three parts (by one loop for all numbers, whose loads had
// neighbouring lanes in different rows): 1,531 rows of 9728 x 896 91 / 146 us (166 / 174), 293 / 183 TFLOP/s of 32-bit products; of 896 x 4864 in three
// pieces 57 / 78 (77 / 80), of 1152 x 896 25 / 35 (38 / 38), 4,000 of 9728 x 896 227 / 371 (415 / 447).
//
// Two ranges have no such parts.  Of numbers below 2^-110 the last bits fall under bfloat16's smallest number, 2^-133
// (the sum of the parts is then off by 2.4e-7 of the number at 2^-112, 9.5e-4 at 2^-124): it shows in what the third
// part is rounded from, whose lower half is not zero.  And numbers that bfloat16 rounds to infinity (3.396e38 and above,
// infinity itself), like products of parts that overflow where the whole product does not, or overflow with both
// signs, leave an output that is not finite.  A block that meets either takes its outputs again on
// v_mfma_f32_16x16x4_f32, operands straight from memory: true 32-bit products over the whole range (1,531 rows of 9728 x
// 896 with such a number in every block 654 us).  (The split is the one of Henry, Tang and Heinecke, "Leveraging the
// bfloat16 artificial intelligence datatype for higher-precision computations", 2019.)
template <int EPI, int BM, int BN, int WM, int WN, bool VEC>
__global__ __launch_bounds__(64 * WM * WN, 2) void gemm_f32_split_kernel(const float* __restrict__ A,
                                                                const float* __restrict__ W, EpiArgs e, int M,
                                                                int N, int K) {
  constexpr int BK = 32, NW = WM * WN;
  constexpr bool GROUPS = NW == 8;
  constexpr int TM = BM / 16 / WM, TN = BN / 16 / WN;    // 16 x 16 tiles per wave along m and n
  constexpr int LA = BM / 16 / NW, LB = BN / 16 / NW;    // pieces of eight numbers per thread and step
  static_assert(LA >= 1 && LB >= 1 && LA * NW * 16 == BM && LB * NW * 16 == BN && TN % 2 == 0, "pieces");
  constexpr int STAGE = (BM + BN) / 16 * 3072;
  __shared__ __attribute__((aligned(1024))) char smem[2 * STAGE];
  __shared__ int s_again;
  __shared__ int s_other;      // where the first step begins that holds a number of W of more than one part, of those put down
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % WM, wn = wave / WM;
  int bx = blockIdx.x, by = blockIdx.y;
  {                                                      // a band of column tiles per die, as above
    const int gx = gridDim.x, gy = gridDim.y, total = gx * gy;
    const int lin = by * gx + bx;
    const int whole = total & ~7;
    const int mapped = lin < whole ? (lin & 7) * (whole >> 3) + (lin >> 3) : lin;
    bx = mapped / gy;
    by = mapped - bx * gy;
  }
  const int m0 = by * BM, n0 = bx * BN;
  const int c = lane & 15, g = lane >> 4;
  // this block's range of the inner size (PART: its group's share, whole steps)
  int k_begin = 0, k_end = K;
  if constexpr (EPI == EPI_PART) {
    k_begin = min(K, (int)blockIdx.z * e.kt_per_split * BK);
    k_end = min(K, k_begin + e.kt_per_split * BK);
    e.out = (float*)e.out + (size_t)blockIdx.z * e.part_stride;
    if (blockIdx.z > 0) e.bias = nullptr;
  }
  if (tid == 0) {
    s_again = 0;
    s_other = 0x7fffffff;
  }

  // (the small products in sums of their own where there are registers for them: a sum is rounded at its own size, once
  // a step and not three or six times; a product of 1,531 rows of 896 x 896 then is 1.9e-7 off 64 bits, 3.1e-7 in one sum)
  constexpr bool APART = TN * TM <= 8;
  floatx4 acc[TN][TM], small[APART ? TN : 1][APART ? TM : 1];
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      acc[j][i] = floatx4{0.f, 0.f, 0.f, 0.f};
      if constexpr (APART) small[j][i] = floatx4{0.f, 0.f, 0.f, 0.f};
    }

  // piece x of a thread: row (wave + NW x) * 16 + sr of the tile, numbers 4 sg .. and 16 + 4 sg .. of the step (four
  // neighbouring lanes read 64 consecutive bytes)
  const int sr = lane >> 2, sg = lane & 3;
  const char* const abase = (const char*)(A + (size_t)m0 * K);
  const char* const bbase = (const char*)(W + (size_t)n0 * K);
  using Offset = std::conditional_t<VEC, uint32_t, size_t>;
  Offset aoff[LA], boff[LB];     // bytes from the tile's first row of x and of W
#pragma unroll
  for (int x = 0; x < LA; ++x) aoff[x] = (Offset)(min(m0 + (wave + NW * x) * 16 + sr, M - 1) - m0) * K * 4;
#pragma unroll
  for (int x = 0; x < LB; ++x) boff[x] = (Offset)(min(n0 + (wave + NW * x) * 16 + sr, N - 1) - n0) * K * 4;
  struct Pieces {
    floatx4 a[LA][2], b[LB][2];
  };
  // Past the range other numbers of the rows are read; stash() puts zeros down for those of x.  Every load is
  // unconditional and their number the same each time: the compiler then counts what is on its way instead of
  // waiting for all of it.
  auto guarded = [&](const float* row, int k) {      // (rows that are not 16-byte aligned)
    floatx4 v;
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = row[min(k + q, k_end - 1)];
    return v;
  };
  auto fetch = [&](Pieces& r, int k0) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int k = k0 + 16 * h + 4 * sg;
      if constexpr (VEC) {
        const uint32_t kb = (uint32_t)min(k, k_end - 4) * 4u;
#pragma unroll
        for (int x = 0; x < LA; ++x) r.a[x][h] = *(const floatx4*)(abase + (aoff[x] + kb));
#pragma unroll
        for (int x = 0; x < LB; ++x) r.b[x][h] = *(const floatx4*)(bbase + (boff[x] + kb));
      } else {
#pragma unroll
        for (int x = 0; x < LA; ++x) r.a[x][h] = guarded((const float*)(abase + aoff[x]), k);
#pragma unroll
        for (int x = 0; x < LB; ++x) r.b[x][h] = guarded((const float*)(bbase + boff[x]), k);
      }
    }
  };
  // Where row r of a fragment has what lane group q of it holds: 16 bytes, with the rows of a group exchanged by the
  // group's number, so that eight neighbouring lanes of a write (two rows, four groups) and of a read (one group, eight rows)
  // meet different banks.
  auto place = [](int r, int q) { return (q * 16 + (r ^ (2 * q))) * 16; };
  const int mine = place(c, g);
  unsigned rest = 0;             // of the numbers of x, what the third part is rounded from
  auto split = [&](const floatx4 (&v)[2], char* to, int k0) {      // (of x the numbers from k0 on; W: k0 < 0)
    uint32_t part[3][4];
    float num[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) num[q] = v[q >> 2][q & 3];
    if (k0 + BK > k_end) {
#pragma unroll
      for (int q = 0; q < 8; ++q) num[q] = k0 + (q >> 2) * 16 + 4 * sg + (q & 3) < k_end ? num[q] : 0.f;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {      // two numbers at a time
      float x0 = num[2 * q], x1 = num[2 * q + 1];
#pragma unroll
      for (int p = 0; p < 3; ++p) {
        typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2;
        const bf16x2 both = {(bf16_t)x0, (bf16_t)x1};
        part[p][q] = __builtin_bit_cast(uint32_t, both);
        if (p < 2) {
          x0 -= __uint_as_float(part[p][q] << 16);
          x1 -= __uint_as_float(part[p][q] & 0xffff0000u);
        }
      }
      rest |= __float_as_uint(x0) | __float_as_uint(x1);      // (their lower halves are zero where bfloat16 holds them)
    }
#pragma unroll
    for (int p = 0; p < 3; ++p)
      *(bf16x8*)(to + p * 1024) = __builtin_bit_cast(bf16x8, floatx4{__uint_as_float(part[p][0]), __uint_as_float(part[p][1]),
                                                                     __uint_as_float(part[p][2]), __uint_as_float(part[p][3])});
  };
  auto upper_halves = [&](const floatx4 (&v)[2], char* to) {      // and what they leave out, zero where bfloat16 holds the numbers
    uint32_t h[4], out = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint32_t a = __float_as_uint(v[q >> 1][(q & 1) * 2]), b = __float_as_uint(v[q >> 1][(q & 1) * 2 + 1]);
      h[q] = __builtin_amdgcn_perm(b, a, 0x07060302);
      out |= a | b;
    }
    *(bf16x8*)to = __builtin_bit_cast(bf16x8, floatx4{__uint_as_float(h[0]), __uint_as_float(h[1]), __uint_as_float(h[2]),
                                                      __uint_as_float(h[3])});
    return out & 0xffffu;
  };
  // The step from k0 on to `stage`.  ONE: one part of every number of W is taken, else three
  auto stash = [&](auto one, const Pieces& r, int k0, int stage) {
    constexpr bool ONE = decltype(one)::value;
    char* to = smem + stage * STAGE + place(sr, sg);
    uint32_t other = 0;
#pragma unroll
    for (int x = 0; x < LA; ++x) split(r.a[x], to + (wave + NW * x) * 3072, k0);
#pragma unroll
    for (int x = 0; x < LB; ++x) {
      if constexpr (ONE) other |= upper_halves(r.b[x], to + BM / 16 * 3072 + (wave + NW * x) * 1024);
      else split(r.b[x], to + (BM / 16 + wave + NW * x) * 3072, -BK);
    }
    if constexpr (ONE)
      if (__ballot(other != 0) != 0 && other != 0) atomicMin(&s_other, k0);      // (no branch by lanes where there is none)
  };
  // the parts of step `t` as a wave multiplies them, and their products, the small ones first
  // (ONE: the order of the general sum, without its terms that are zero)
  auto x_part = [&](bf16x8 (&xf)[TM], int stage, int p) {
    const char* xs = smem + stage * STAGE + mine;
#pragma unroll
    for (int i = 0; i < TM; ++i) xf[i] = *(const bf16x8*)(xs + ((wm * TM + i) * 3 + p) * 1024);
  };
  auto w_part = [&](auto one, bf16x8 (&wf)[TN], int stage, int p) {
    constexpr int PW = decltype(one)::value ? 1 : 3;
    const char* ws = smem + stage * STAGE + BM / 16 * 3072 + mine;
#pragma unroll
    for (int j = 0; j < TN; ++j) wf[j] = *(const bf16x8*)(ws + ((wn * TN + j) * PW + p) * 1024);
  };
  auto products = [&](auto large, const bf16x8 (&wf)[TN], const bf16x8 (&xf)[TM]) {
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        floatx4& sum = APART && !decltype(large)::value ? small[APART ? j : 0][APART ? i : 0] : acc[j][i];
        sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[j], xf[i], sum, 0, 0, 0);
      }
  };
  auto barrier = [&]() {      // (nothing moves across; a wave's reads and writes of LDS are done)
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0xc07f);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };

  // The steps from k0 on; with one part of W up to the first that holds a number of more.  Returns where it left off.
  auto walk = [&](auto one, int k0) -> int {
    constexpr bool ONE = decltype(one)::value;
    constexpr int PW = ONE ? 1 : 3;
    // (what a wave finds in s_other in its step from k0 on: every piece of that step was put down before the barrier it came
    // through; what others put down meanwhile is of a later step)
    // (a relaxed atomic load: of a volatile one each would be waited for at once)
    auto other_from = [&]() {
      return ONE ? __hip_atomic_load(&s_other, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) : 0x7fffffff;
    };
    auto before = [&](int other) { return ONE && __builtin_amdgcn_readfirstlane(other) <= k0; };
    Pieces r0, r1;
    fetch(r0, k0);
    fetch(r1, k0 + BK);
    if constexpr (ONE) barrier();      // (s_other is set)
    stash(one, r0, k0, 0);
    fetch(r0, k0 + 2 * BK);
    __syncthreads();
    if (before(other_from())) return k0;
    // A step is put down during the one before, from registers that were asked for two steps before that.
    bf16x8 xf[3][TM], wf[PW][TN];
    auto read = [&](int stage) {
#pragma unroll
      for (int p = 0; p < 3; ++p) x_part(xf[p], stage, p);
#pragma unroll
      for (int p = 0; p < PW; ++p) w_part(one, wf[p], stage, p);
    };
    auto multiply = [&]() {
      const std::false_type part;
      if constexpr (ONE) {
        products(part, wf[0], xf[1]);
        products(part, wf[0], xf[2]);
      } else {
        products(part, wf[1], xf[1]);            // m_w m_x
        products(part, wf[1], xf[0]);
        products(part, wf[0], xf[1]);
        products(part, wf[2], xf[0]);
        products(part, wf[0], xf[2]);
      }
      products(std::true_type{}, wf[0], xf[0]);  // h_w h_x
    };
    // (r: the next step's numbers)
    if constexpr (GROUPS && (ONE || TN > 2)) {
      if (wave >= NW / 2) barrier();       // the second group runs half a step behind
      auto step = [&](int stage, Pieces& r) -> bool {
        const int other = other_from();
        read(stage);
        stash(one, r, k0 + BK, stage ^ 1);
        barrier();
        if (before(other)) return false;
        fetch(r, k0 + 3 * BK);
        multiply();
        // (the loads and what they take to address between the matrix instructions)
#pragma unroll
        for (int n = 0; n < 2 * (LA + LB); ++n) {
          __builtin_amdgcn_sched_group_barrier(0x8, 3, 0);      // matrix instructions
          __builtin_amdgcn_sched_group_barrier(0x2, 4, 0);      // vector instructions
          __builtin_amdgcn_sched_group_barrier(0x20, 1, 0);     // a load
        }
        barrier();
        k0 += BK;
        return k0 < k_end;
      };
      // (both groups leave at the same step, and the first waits for the second's reads of it)
      while (step(0, r1) && step(1, r0)) {}
      if (wave < NW / 2) barrier();
    } else {
      auto step = [&](int stage, Pieces& r) -> bool {
        const int other = other_from();
        read(stage);
        if (before(other)) return false;
        stash(one, r, k0 + BK, stage ^ 1);
        multiply();
        fetch(r, k0 + 3 * BK);
        __syncthreads();
        k0 += BK;
        return k0 < k_end;
      };
      while (step(0, r1) && step(1, r0)) {}
    }
    return k0;
  };
  if (k_begin < k_end) {
    const int left_off = walk(std::true_type{}, k_begin);
    if (left_off < k_end) walk(std::false_type{}, left_off);
  }
  if constexpr (APART) {
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int i = 0; i < TM; ++i) acc[j][i] += small[j][i];
  }
  bool again = (rest & 0xffffu) != 0;
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int x = 0; x < 4; ++x) again |= !(fabsf(acc[j][i][x]) < __builtin_inff());
  if (again) s_again = 1;      // (any thread's; the same value from all)
  __syncthreads();
  if (s_again) {
    auto checked = [&](const float* row, int k) {
      floatx4 v = guarded(row, k);
#pragma unroll
      for (int q = 0; q < 4; ++q) v[q] = k + q < k_end ? v[q] : 0.f;
      return v;
    };
    // lane (c, g) holds the numbers 4 g .. 4 g + 3 of 16 of its row; an instruction contracts one of each group
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int i = 0; i < TM; ++i) acc[j][i] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int k0 = k_begin; k0 < k_end; k0 += 16) {
      const int k = k0 + 4 * g;
      const bool whole = VEC && k0 + 16 <= k_end;
      floatx4 xf[TM], wf[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const float* row = A + (size_t)min(m0 + (wm * TM + i) * 16 + c, M - 1) * K;
        xf[i] = whole ? *(const floatx4*)(row + k) : checked(row, k);
      }
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const float* row = W + (size_t)min(n0 + (wn * TN + j) * 16 + c, N - 1) * K;
        wf[j] = whole ? *(const floatx4*)(row + k) : checked(row, k);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int i = 0; i < TM; ++i)
            acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[j][e], xf[i][e], acc[j][i], 0, 0, 0);
    }
  }
  // lane (c, g) holds, of every 16 x 16 tile, output row m = c and the columns n = 4 g .. 4 g + 3
  const bool whole_pieces = (e.ldo & 3) == 0 && ((uintptr_t)e.out & 15) == 0;
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int m = m0 + (wm * TM + i) * 16 + c;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int nb = n0 + (wn * TN + j) * 16;
      if constexpr (EPI == EPI_SWIGLU) {
        // tiles of columns alternate: gate, up of the same 16 outputs
        if (j & 1) continue;
        const int o = (nb >> 5) * 16 + 4 * g;
        floatx4 v;
#pragma unroll
        for (int x = 0; x < 4; ++x) v[x] = pair_exact_f(acc[j][i][x], acc[j + 1][i][x], e);
        float* dst = (float*)e.out + (size_t)m * e.ldo + o;
        if (whole_pieces && o + 4 <= e.n_out) *(floatx4*)dst = v;
        else
#pragma unroll
          for (int x = 0; x < 4; ++x)
            if (o + x < e.n_out) dst[x] = v[x];
      } else {
        const int n = nb + 4 * g;
        floatx4 v = acc[j][i];
        if (e.bias)
#pragma unroll
          for (int x = 0; x < 4; ++x) v[x] += load_vec(e.bias, e.bias_bf16, min(n + x, N - 1));
        if (EPI == EPI_STORE && e.act)
#pragma unroll
          for (int x = 0; x < 4; ++x) v[x] = relu2_f(v[x]);
        float* dst = (float*)e.out + (size_t)m * e.ldo + n;
        if (whole_pieces && n + 4 <= N) {
          if (EPI == EPI_RESID) v += *(const floatx4*)dst;
          *(floatx4*)dst = v;
        } else {
#pragma unroll
          for (int x = 0; x < 4; ++x)
            if (n + x < N) dst[x] = (EPI == EPI_RESID ? dst[x] : 0.f) + v[x];
        }
      }
    }
  }
}

// The tiles of the products of many rows (what the numbers are: below, where a bfloat16 product is given its tile).
enum { TILE_64 = 0, TILE_64x128 = 1, TILE_128 = 2, TILE_128x256 = 3, TILE_256 = 4, TILE_192 = 5, TILE_KINDS = 6,
       // chosen by their own rule (one_round_tile) for whole products
       TILE_64x96 = 6, TILE_64x160 = 7, TILE_64x224 = 8, TILE_128x160 = 9,
       // by direct loads, eight waves: in place of other tiles where direct_tile says so
       TILE_DIRECT_128 = 10, TILE_DIRECT_128x192 = 11, TILE_DIRECT_192x128 = 12, TILE_ALL = 13 };
struct TileModel {
  int bm, bn;
  double L, f, tk, resident, stream;
  int whole_rounds;
};
// (the 64 x 64 row was fitted to a kernel that took x by way of registers, slower by 18 %; in the range of
// few_blocks_cost that decides)
static const TileModel TILE_MODELS[TILE_ALL] = {{64, 64, 6.39, 0.79, 0.289, 1.0, 20e3, 0},
                                                  {64, 128, 6.54, 0.71, 0.5, 1.5, 27e3, 0},
                                                  {128, 128, 8.0, 0.48, 0.66, 1.0, 24e3, 0},
                                                  {128, 256, 0.0, 6.16, 0.945, 1.0, 24e3, 1},
                                                  {256, 256, 0.0, 12.8, 1.34, 1.0, 24e3, 1},
                                                  {192, 256, 0.0, 10.2, 1.08, 1.0, 24e3, 1},
                                                  {64, 96}, {64, 160}, {64, 224}, {128, 160},
                                                  {128, 128}, {128, 192}, {192, 128}};

// The tile of a float32 product of many rows, and into how many pieces along the inner size one that adds
// into the stream is cut.
struct F32Plan {
  int tile, pieces;      // TILE_64, TILE_128 or TILE_128x256
};
static F32Plan f32_plan(int M, int N, int K, int num_cus, int max_pieces, int min_steps);

// The tiles by direct loads address a tile's rows by 32 bits of bytes, which hold 255 rows (and 15 strips of
// W) of this inner size; beyond, the 64 x 128 tile, whose addresses have 64.
constexpr int DIRECT_MAX_INNER = 1 << 22;

template <int EPI>
static void launch_f32_split(int tile, const float* A, const float* W, const EpiArgs& e, int M, int N, int K, int pieces,
                             hipStream_t stream) {
  // (whole loads of 16 bytes, and 32 bits of offset within 256 rows)
  const bool vec = (K % 4 == 0) && ((uintptr_t)A % 16 == 0) && ((uintptr_t)W % 16 == 0) && K <= DIRECT_MAX_INNER;
  if (!vec && tile == TILE_128x256) tile = TILE_128;
  const int bm = TILE_MODELS[tile].bm, bn = TILE_MODELS[tile].bn;
  const dim3 grid((N + bn - 1) / bn, (M + bm - 1) / bm, pieces);
  if (tile == TILE_128x256)
    hipLaunchKernelGGL((gemm_f32_split_kernel<EPI, 128, 256, 2, 4, true>), grid, dim3(512), 0, stream, A, W, e, M, N, K);
  else if (tile == TILE_128 && vec)
    hipLaunchKernelGGL((gemm_f32_split_kernel<EPI, 128, 128, 2, 4, true>), grid, dim3(512), 0, stream, A, W, e, M, N, K);
  else if (tile == TILE_128)
    hipLaunchKernelGGL((gemm_f32_split_kernel<EPI, 128, 128, 2, 4, false>), grid, dim3(512), 0, stream, A, W, e, M, N, K);
  else if (vec)
    hipLaunchKernelGGL((gemm_f32_split_kernel<EPI, 64, 64, 2, 2, true>), grid, dim3(256), 0, stream, A, W, e, M, N, K);
  else
    hipLaunchKernelGGL((gemm_f32_split_kernel<EPI, 64, 64, 2, 2, false>), grid, dim3(256), 0, stream, A, W, e, M, N, K);
}

// Products of many rows in float32: the matrix cores, or (debug) the plain FMA kernel, their reference, with
// the largest tile that still gives every compute unit a block.
template <int EPI>
static void launch_f32_tiled(const float* A, const float* W, const EpiArgs& e, int M, int N, int K,
                             int num_cus, hipStream_t stream) {
  const int vec = (K % 4 == 0) && ((uintptr_t)A % 16 == 0) && ((uintptr_t)W % 16 == 0);
  auto blocks = [&](int bm, int bn) { return (long)((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
  if (g_f32_fma == 0) {
    launch_f32_split<EPI>(f32_plan(M, N, K, num_cus, 1, 1).tile, A, W, e, M, N, K, 1, stream);
    return;
  }
  if (blocks(128, 128) >= num_cus)
    hipLaunchKernelGGL((gemm_f32_kernel<EPI, 128, 128>), dim3((N + 127) / 128, (M + 127) / 128), dim3(256), 0,
                       stream, A, W, e, M, N, K, vec);
  else if (blocks(128, 64) >= num_cus)
    hipLaunchKernelGGL((gemm_f32_kernel<EPI, 128, 64>), dim3((N + 63) / 64, (M + 127) / 128), dim3(256), 0,
                       stream, A, W, e, M, N, K, vec);
  else
    hipLaunchKernelGGL((gemm_f32_kernel<EPI, 64, 64>), dim3((N + 63) / 64, (M + 63) / 64), dim3(256), 0,
                       stream, A, W, e, M, N, K, vec);
}

// Few rows in float32 (decode steps, short portions): a block owns NB = 4 rows of W, its KW
// waves split the inner size, and a wave's lanes split its share, four numbers a lane and
// step, so that a wave instruction reads 1 KB of a row of W in a row (any inner size: one
// number at a time where rows are not 16-byte aligned).  Two steps are on their way from
// memory at a time.  MB rows of x go with them (they stay in the caches); the MB x NB sums
// meet by lane shuffles and, across the waves, in LDS in a fixed order.  For SWIGLU the four
// rows are two gate rows and the up rows of the same two outputs.  Still plain FMAs in 32
// bits.  (One wave per block left a narrow output, 224 blocks of the down product, with one
// wave per compute unit walking 19 steps one after the other: 26 us for 17 MB.)
template <int EPI, int MB, int KW>
__global__ __launch_bounds__(64 * KW) void gemm_f32_rows_kernel(const float* __restrict__ A,
                                                                 const float* __restrict__ W, EpiArgs e, int M,
                                                                 int N, int K, int vec) {
  constexpr int NB = 4;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int m0 = blockIdx.y * MB;
  int rows_w[NB];
  if constexpr (EPI == EPI_SWIGLU) {
    const int n = (blockIdx.x >> 3) * 32 + (blockIdx.x & 7) * 2;     // two gate rows; their up rows 16 on
    rows_w[0] = n; rows_w[1] = n + 1; rows_w[2] = n + 16; rows_w[3] = n + 17;
  } else {
#pragma unroll
    for (int j = 0; j < NB; ++j) rows_w[j] = blockIdx.x * NB + j;
  }
  const float* wp[NB];
  const float* xp[MB];
#pragma unroll
  for (int j = 0; j < NB; ++j) wp[j] = W + (size_t)min(rows_w[j], N - 1) * K;   // clamped: read, never stored
#pragma unroll
  for (int i = 0; i < MB; ++i) xp[i] = A + (size_t)min(m0 + i, M - 1) * K;
  float acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = 0.f;
  if (vec) {
    constexpr int STEP = 256 * KW;
    auto mac = [&](const floatx4 (&w4)[NB], const floatx4 (&x4)[MB]) {
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
          for (int c = 0; c < 4; ++c) acc[i][j] = fmaf(x4[i][c], w4[j][c], acc[i][j]);
    };
    int k = (wave * 64 + lane) * 4;
    for (; k + STEP < K; k += 2 * STEP) {            // two steps at a time
      floatx4 w4[2][NB], x4[2][MB];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
#pragma unroll
        for (int j = 0; j < NB; ++j) w4[u][j] = *(const floatx4*)(wp[j] + k + u * STEP);
#pragma unroll
        for (int i = 0; i < MB; ++i) x4[u][i] = *(const floatx4*)(xp[i] + k + u * STEP);
      }
      mac(w4[0], x4[0]);
      mac(w4[1], x4[1]);
    }
    for (; k < K; k += STEP) {
      floatx4 w4[NB], x4[MB];
#pragma unroll
      for (int j = 0; j < NB; ++j) w4[j] = *(const floatx4*)(wp[j] + k);
#pragma unroll
      for (int i = 0; i < MB; ++i) x4[i] = *(const floatx4*)(xp[i] + k);
      mac(w4, x4);
    }
  } else {
    for (int k = wave * 64 + lane; k < K; k += 64 * KW) {
      float w1[NB], x1[MB];
#pragma unroll
      for (int j = 0; j < NB; ++j) w1[j] = wp[j][k];
#pragma unroll
      for (int i = 0; i < MB; ++i) x1[i] = xp[i][k];
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = fmaf(x1[i], w1[j], acc[i][j]);
    }
  }
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = wave_sum(acc[i][j]);
  if constexpr (KW > 1) {
    __shared__ float red[KW][MB][NB];
    if (lane == 0) {
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) red[wave][i][j] = acc[i][j];
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        float t = red[0][i][j];
#pragma unroll
        for (int w = 1; w < KW; ++w) t += red[w][i][j];
        acc[i][j] = t;
      }
  } else {
    if (lane != 0) return;
  }
#pragma unroll
  for (int i = 0; i < MB; ++i) {
    const int m = m0 + i;
    if (m >= M) continue;
    if constexpr (EPI == EPI_SWIGLU) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int o = (rows_w[j] >> 5) * 16 + (rows_w[j] & 15);
        if (o < e.n_out) ((float*)e.out)[(size_t)m * e.ldo + o] = pair_exact_f(acc[i][j], acc[i][j + 2], e);
      }
    } else {
#pragma unroll
      for (int j = 0; j < NB; ++j)
        if (rows_w[j] < N) epi_store<float, EPI>(e, m, rows_w[j], acc[i][j]);
    }
  }
}

template <int EPI, int KW>
static void launch_f32_rows_kw(const float* A, const float* W, const EpiArgs& e, int M, int N, int K, int vec,
                               unsigned groups, hipStream_t stream) {
  if (M == 1)
    hipLaunchKernelGGL((gemm_f32_rows_kernel<EPI, 1, KW>), dim3(groups, 1), dim3(64 * KW), 0, stream, A, W, e, M, N, K, vec);
  else if (M == 2)
    hipLaunchKernelGGL((gemm_f32_rows_kernel<EPI, 2, KW>), dim3(groups, 1), dim3(64 * KW), 0, stream, A, W, e, M, N, K, vec);
  else if (M <= 4)
    hipLaunchKernelGGL((gemm_f32_rows_kernel<EPI, 4, KW>), dim3(groups, 1), dim3(64 * KW), 0, stream, A, W, e, M, N, K, vec);
  else
    hipLaunchKernelGGL((gemm_f32_rows_kernel<EPI, 8, KW>), dim3(groups, (M + 7) / 8), dim3(64 * KW), 0, stream, A, W, e,
                       M, N, K, vec);
}

// Waves per block: as many as give every wave at least two steps of its own, up to 8, fewer
// where the blocks alone already put several waves on every compute unit.
template <int EPI>
static void launch_f32_rows(const float* A, const float* W, const EpiArgs& e, int M, int N, int K, int num_cus,
                            hipStream_t stream) {
  const int vec = (K % 4 == 0) && ((uintptr_t)A % 16 == 0) && ((uintptr_t)W % 16 == 0);
  const unsigned groups = EPI == EPI_SWIGLU ? (unsigned)(N / 32) * 8 : (unsigned)((N + 3) / 4);
  const long blocks = (long)groups * ((M + 7) / 8);
  const int steps = (K + 255) / 256;
  int kw = 1;
  while (kw < 8 && steps >= 4 * kw && blocks * kw < 8L * num_cus) kw *= 2;
  if (kw >= 8) launch_f32_rows_kw<EPI, 8>(A, W, e, M, N, K, vec, groups, stream);
  else if (kw == 4) launch_f32_rows_kw<EPI, 4>(A, W, e, M, N, K, vec, groups, stream);
  else if (kw == 2) launch_f32_rows_kw<EPI, 2>(A, W, e, M, N, K, vec, groups, stream);
  else launch_f32_rows_kw<EPI, 1>(A, W, e, M, N, K, vec, groups, stream);
}
constexpr int F32_ROWS_MAX = 64;     // up to here the few-row kernel (the tiled one would run on N / 64 blocks)

// ================================================================ dispatch
// The 64 x 64 tile of gemm_bf16_ring for small products; three tile shapes with x through LDS and W straight
// from the packed matrix, 64 x 128 and 128 x 128 with four waves and 128 x 256
// with eight, side by side along the columns (1 x 4, 1 x 8), so that every fragment of W
// is read by one wave only and the rows of x in LDS are shared by all of them; and the
// 256 x 256 and 192 x 256 tiles of gemm_bf16_pingpong for the largest products.  The shape
// is picked by an estimate of the time, fitted to sweeps of the four products of a layer
// at three model shapes and 576 to 8192 rows, when all epilogues went through LDS (its picks then cost
// 0.8 % over the best shape there; now, over shapes of 0.5B to 7B at 256 to 3,000 rows, 1.2 % for gate and up, 3.4 for output
// and 3.6 for down products, and constants lowered to what the epilogues take lose more on single output products):
//   time = L + rounds * (f + K tiles * tk),  rounds = max(1, blocks / (units * resident)).
// One block of the 128 x 256 tile fills a compute unit (eight waves of 220 registers a lane), so
// its rounds are whole: ceil(blocks / units).  Where its blocks fill their rounds it is
// the fastest by 5 to 20 % (2048 rows, 3584 x 18944: 301 us against 337 with 128 x 128;
// 8192 rows, 37888 x 3584: 2320 against 2577), where the last round is nearly empty the
// slowest (2048 rows, 5120 x 27648: 852 against 731).
// With few rows the product is bound by the read of W instead: a block draws `stream`
// bytes a microsecond, the chip 5.3e6 at most (one tile of rows, 17 to 64 of them, of
// matrices from 9 to 283 MB, in 4 or 8 pieces: the estimate is within 2 us of the
// measurement).
constexpr double CHIP_STREAM = 5.3e6;     // bytes a microsecond

// The tiles of the two groups of waves: whole rounds of one block a unit; with 256 rows a
// step of 32 of the inner size takes 0.67 us in a full round and from 0.41 us in a round of
// few blocks (the chip clocks higher), and 12.8 us were to pass before and after the loop; with 192
// rows 0.54, 0.37 and 10.2 us (epilogues by way of LDS, as above; fitted to a sweep of 14 matrices of four model shapes at 512 to 8192
// rows, inner sizes from 896 to 18944: 7 and 5 % rms).
static double pingpong_cost(int bm, int M, int N, int K, int num_cus, int pieces) {
  const double rounds = (double)((M + bm - 1) / bm) * ((N + 255) / 256) * pieces / num_cus;
  const double whole = floor(rounds + 1e-9), last = rounds - whole;
  const int steps = pieces > 1 ? 2 * (((K + 63) / 64 + pieces - 1) / pieces) : (K + 31) / 32;
  const double before_after = bm == 256 ? 12.8 : 10.2, full = bm == 256 ? 0.67 : 0.544, few = bm == 256 ? 0.414 : 0.371;
  double t = whole * (before_after + steps * full);
  if (last > 1e-9) t += before_after + steps * (few + (full - few) * last);
  return t;
}

static double tile_cost(int kind, int M, int N, int K, int num_cus, int pieces) {
  if (kind == TILE_256 || kind == TILE_192) return pingpong_cost(TILE_MODELS[kind].bm, M, N, K, num_cus, pieces);
  const TileModel& t = TILE_MODELS[kind];
  const double blocks = (double)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn) * pieces;
  double rounds = blocks / (num_cus * t.resident);
  // (the 64 x 64 tile beyond 64 rows: measured, a block more than the units hold costs a whole
  // round: 256 rows of 4608 x 3584, 288 blocks, 32 us against 29 with 144 blocks of 64 x 128,
  // and 192 rows, 216 blocks, 26 against 29)
  if (t.whole_rounds || (kind == TILE_64 && M > 64)) rounds = ceil(rounds - 1e-9);
  const int nk = ((K + 63) / 64 + pieces - 1) / pieces;
  const double compute = (rounds > 1.0 ? rounds : 1.0) * (t.f + nk * t.tk);
  const double rate = blocks * t.stream < CHIP_STREAM ? blocks * t.stream : CHIP_STREAM;
  const double read = (double)N * K * 2.0 / rate;
  return t.L + (compute > read ? compute : read);
}

// Debug interface (kernels/debug.py): a tile can be forced, for tests and measurements
// (0 = choose; 64, 130 = 64 x 128, 129 = 128 x 128, 131 = 128 x 256, 132 = 256 x 256, 133 =
// 192 x 256, 134 / 135 / 136 = 64 x 96 / 160 / 224, 137 = 128 x 160, 138 / 139 / 140 = 128 x 128, 128 x 192 and 192 x 128 by direct loads; -131 = choose among the first three; -256 and below: the tiles of two groups
// of waves from so many rows on).
static int g_force_tile = 0, g_without_wide = 0, g_pp_min_rows = 512;
// The 128 x 256 tile is weighed from so many rows on.  (By the product alone it would pay from
// 768: 1,536 rows of 5120 x 27648 447 us against 543; inside prefill steps of 768 to 1,536
// tokens of five shapes that is between 1.4 % faster and 1.3 % slower than from 2,048 on.)
constexpr int WIDE_TILE_MIN_ROWS = 2048;
constexpr int PP_MIN_INNER = 896;      // the shortest inner size the estimates of those tiles were fitted to
static int addressable(int kind, int K) {
  return K > DIRECT_MAX_INNER && (kind == TILE_64 || kind == TILE_256 || kind == TILE_192) ? TILE_64x128 : kind;
}
extern "C" void llmlab_debug_gemm_tile(int tile) {
  g_force_tile = tile > 0 ? tile : 0;
  g_without_wide = tile == -131;
  g_pp_min_rows = tile <= -256 ? -tile : 512;
}

// Up to 128 rows of a wide matrix: the product is bound by the read of W, every compute unit draws its
// share at the same rate, and what matters is that all of them draw until the end: one round of
// blocks that nearly fills the chip, each wave with 32 columns of its own.  The width that does that,
// 32 times 3, 4, 5 or 7, is the narrowest whose blocks find a unit each (-1: none does, or the round would
// leave a fifth of the units, of the narrowest tile three tenths, without a block).
// Measured against the best of the other tiles / the estimates' pick: 64 rows of 37888 x 3584 (160 columns,
// 237 blocks) 57 us against 70 / 70, of 22016 x 2048 (96, 230) 26.2 / 27.2 / 27.8, of 17920 x 1536 (96, 187)
// 19.6 / 20.9 / 22.9, of 27648 x 5120 (128, 216) 62 / 62 / 69, of 55296 x 5120 (224, 247) 105 / 109 / 109; 17 rows
// the same.  Short inner sizes: 17 / 64 rows of 24448 x 1024 (96) 15.3 / 16.8 against 15.9 / 16.8 by the estimates, of
// 37888 x 1024 (160) 20.3 / 21.8 against 21.6 / 24.2; 128 columns lose at 1,024 (28672: 16.9 / 18.4 against 16.2 / 17.3)
// and not at 1,152 (18.6 / 19.9 and 18.8 / 20.9); 224 lose until 2,048 (49152 x 1152: 26.9 / 28.5 against 25.3 / 28.5, x
// 2048: 40.3 / 42.2 and 38.7 / 42.5) and not at 3,072 (56.1 / 60.7 and 56.8 / 62.5).  128 rows of 37888 x 3584 in one tile of rows (160) 70 / 78 / 79, of 17920 x 1536 in two (2 x 112
// blocks) 23.9 / 27.1 / 27.3.
static int one_round_tile(int M, int N, int K, int num_cus) {
  if (M > 128 || K < 1024) return -1;
  auto fills = [&](int width, int tiles, double least) {
    const long blocks = (long)((N + width - 1) / width) * tiles;
    return blocks <= num_cus && blocks >= least * num_cus;
  };
  if (M > 64) {
    if (fills(160, 1, 0.8)) return TILE_128x160;
    return fills(160, 2, 0.8) ? TILE_64x160 : -1;
  }
  if (fills(96, 1, 0.7)) return TILE_64x96;
  if (fills(128, 1, 0.8)) return K >= 1152 ? TILE_64x128 : -1;
  if (fills(160, 1, 0.8)) return TILE_64x160;
  return K >= 3072 && fills(224, 1, 0.8) ? TILE_64x224 : -1;
}

// By an estimate of the time, fitted to a sweep of eight matrices of three model shapes at 65 to 4,096 rows
// whole and in up to eight pieces, each with W's numbers of one part and of three (948 times; 4 to 9 % rms about the
// geometric mean of the two, since W's numbers are not known here; the picks lose 0.6 % whole and 2.3 % in pieces to the
// best of the sweep; before the bound below).  Against the tiles and picks before (64 x 64 and 128 x 128, one loop for all numbers, a load of 16
// rows with neighbouring lanes in different ones) they take 0.60 of the time whole and 0.72 with the fold of their
// pieces where W has one part, 0.87 and 0.94 where it has three (9 % more at worst, of a product in fewer pieces than
// before).  A block of the 128 x 128 and 128 x 256 tiles is alone on its unit, rounds are whole; of the 64 x 64 tile
// three share one, whose first is slow by itself.
//
// How many steps a sum may add where the product may be cut: a sum is rounded at its own size once a product and step, so that
// its error grows as the root of its steps.  The bound is what the estimate of the first kernels gave (64 x 64 and
// 128 x 128, everything in one sum): the 128 x 256 tile, which adds everything in one sum, holds to it (and to 64 steps: 7,041
// rows of 896 x 4864 whole were 7.4e-7 off 64 bits and a decode step behind such prompts 1.68e-6, in three pieces 4.3e-7 and
// 1.44e-6); the others, whose small products have sums of their own and whose error at the same steps is 0.55 of
// that, may add three times as many.  (Without the bound 4,040 rows of 1536 x 1536 whole 4.2e-7 / 6.0e-7 off 64 bits with one part of
// W and with three, in two pieces 2.9e-7 / 4.2e-7; 2,312 of 2048 x 2048 4.9e-7 / 7.0e-7 and 3.4e-7 / 4.9e-7; 3,336 of 896 x
// 4864 by 128 x 128 whole 4.3e-7, in four pieces, as planned with it, 2.1e-7, by the first kernel in four 3.7e-7.)
constexpr int F32_WIDE_STEPS = 64;
static int f32_sum_steps(int M, int N, int steps, int num_cus, int max_pieces, int min_steps) {
  int most = steps;
  double least = 1e30;
  for (int bm = 64; bm <= 128; bm += 64) {
    for (int pieces = 1; pieces <= max_pieces; ++pieces) {
      const int s = (steps + pieces - 1) / pieces;
      if (pieces > 1 && s < min_steps) break;
      const double share = (double)((M + bm - 1) / bm) * ((N + bm - 1) / bm) * pieces / num_cus;
      const double whole = ceil(share - 1e-9);
      double t = whole * (5.4 + s * (1.31 + 0.12 * (share < 1.0 ? share : 1.0)));
      if (bm == 64) {
        const double shared = (share <= 3.0 ? whole : share) * (1.0 + 0.58 * s);
        t = 2.0 + 0.863 * s;
        if (shared > t && whole > 1.0) t = shared;
      }
      if (pieces > 1) t += pieces * ((double)M * N * 2.2e-6 + 0.3);
      if (t < least) {
        least = t;
        most = s;
      }
    }
  }
  return most;
}
static F32Plan f32_plan(int M, int N, int K, int num_cus, int max_pieces, int min_steps) {
  const int steps = (K + 31) / 32;
  const int sum_steps = f32_sum_steps(M, N, steps, num_cus, max_pieces, min_steps);
  F32Plan best{-1, 1};
  double least = 0.0;
  for (const int tile : {TILE_64, TILE_128, TILE_128x256}) {
    if (g_force_tile == 64 && tile != TILE_64) continue;
    if ((g_force_tile == 128 || g_force_tile == 129) && tile != TILE_128) continue;
    if (g_force_tile == 131 && tile != TILE_128x256) continue;
    const int bm = TILE_MODELS[tile].bm, bn = TILE_MODELS[tile].bn;
    for (int pieces = 1; pieces <= max_pieces; ++pieces) {
      const int s = (steps + pieces - 1) / pieces;
      if (pieces > 1 && s < min_steps) break;
      const int most = tile == TILE_128x256 ? (sum_steps < F32_WIDE_STEPS ? sum_steps : F32_WIDE_STEPS) : 3 * sum_steps;
      const bool finer = pieces < max_pieces && (steps + pieces) / (pieces + 1) >= min_steps;      // (there are more pieces to be had)
      if (s > most && finer) continue;
      const double share = (double)((M + bm - 1) / bm) * ((N + bn - 1) / bn) * pieces / num_cus;
      const double whole = ceil(share - 1e-9);
      double t;
      if (tile == TILE_128x256) {
        t = 1.65 + whole * (8.9 + s * (1.475 + 0.377 * (share < 1.0 ? share : 1.0)));
      } else if (tile == TILE_128) {
        t = 1.4 + whole * (5.9 + s * (0.945 + 0.22 * (share < 1.0 ? share : 1.0)));
      } else {
        const double shared = (share <= 3.0 ? whole : share) * (1.25 + 0.394 * s);
        t = 5.7 + 0.504 * s;
        if (shared > t && whole > 1.0) t = shared;
      }
      if (pieces > 1) t += pieces * ((double)M * N * 2.2e-6 + 0.3);      // (their way through memory to the next reader)
      if (best.tile < 0 || t < least) {
        least = t;
        best = F32Plan{tile, pieces};
      }
    }
  }
  return best;
}

static int estimated_tile(int M, int N, int K, int num_cus) {
  if (g_force_tile == 64) return addressable(TILE_64, K);
  if (g_force_tile == 130) return TILE_64x128;
  if (g_force_tile == 129 || g_force_tile == 128) return TILE_128;
  if (g_force_tile == 131) return TILE_128x256;
  if (g_force_tile == 132) return addressable(TILE_256, K);
  if (g_force_tile == 133) return addressable(TILE_192, K);
  // One or two tiles of rows of a wide matrix (the head, gate and up at larger shapes):
  // bound by the read of W, which the wider tiles stream better than the estimate
  // knows, and the 128-row tile reads W once where two 64-row tiles read it twice
  // (64 rows, 152064 x 3584: 220 us against 250 with the 64 x 64 tile; 128 rows,
  // 55296 x 5120: 127 against 157).
  const long wide = (N + 127) / 128;
  if (M <= 64 && wide >= num_cus) return TILE_64x128;
  // ... and of a matrix of 32,768 to 65,536 rows the 128 x 256 tile (96 / 128 rows of 37888 x
  // 3584: 81 / 77 us against 83 / 84, and 70 in the one round of one_round_tile, which whole products ask first; of 59136 x 8192: 195 / 201 against 200 / 209; a decode
  // step of 128 requests of the 7B shape 6.99 -> 6.86 ms, of the 32B shape 24.8 -> 24.4; a
  // vocabulary of 152,064 gains nothing from it)
  if (M > 64 && M <= 128 && N >= 32768 && N <= 65536 && K >= 1024 && !g_without_wide) return TILE_128x256;
  if (M > 64 && M <= 128 && wide >= 3L * num_cus / 2) return TILE_128;
  // The 128 x 256 tile from 2048 rows on: with 576 and 1024 rows it wins or loses a few
  // percent by the product alone, and a prefill step of 1024 tokens as a whole is 1 to
  // 2 % slower with it than without (steps of 2048: from 0.6 % slower to 3 % faster by
  // the shape of the model, of 4096 and 8192: 3 to 7 % faster at the larger shapes), and
  // an inner size of 1024 on: with 896 its one block per unit shows its start and its
  // epilogue, and steps of 4096 are 1.7 % slower with it.
  const int kinds = M >= WIDE_TILE_MIN_ROWS && K >= 1024 && !g_without_wide ? TILE_256 : TILE_128x256;
  double cost[TILE_KINDS];
  int best = 0;
  for (int kind = 0; kind < kinds; ++kind) {
    cost[kind] = tile_cost(kind, M, N, K, num_cus, 1);
    if (cost[kind] < cost[best]) best = kind;
  }
  // Enough 128 x 128 tiles for four rounds of blocks: a large tile, whatever the
  // estimate makes of the rows it pads (576 rows, 37888 x 3584: 206 us against 221 with
  // 64 x 128; 1024 rows: 324 against 370).  Which of the two, the estimates cannot tell
  // here (they err by 10 % in opposite directions): the 128 x 256 tile unless its last
  // round is less than half full and one of few (2048 rows, 37888 x 3584, 9.25 rounds:
  // 640 us against 588 inside a prefill step; 18.5 rounds: 1246 against 1273; 37: 2302
  // against 2517; 3.5 rounds, 7168 x 5120: 359 against 379).
  if (((long)(M + 127) / 128) * wide >= 4L * num_cus) {
    best = TILE_128;
    if (kinds > TILE_128x256) {
      const double rounds = (double)((M + 127) / 128) * ((N + 255) / 256) / num_cus;
      const double last = rounds - floor(rounds);
      if (last < 1e-9 || last >= 0.5 || rounds >= 16.0) best = TILE_128x256;
    }
  }
  // The tiles of the two groups of waves where the estimate of one is the lowest (over the
  // sweeps the 256 x 256 tile is then 10 to 30 % faster than the best of the others: 2048
  // rows, 37888 x 3584: 460 us against 607; with a quarter
  // of a round of blocks it is twice as slow; the 192 x 256 tile where its blocks fill
  // their rounds better: 2048 rows, 4608 x 3584: 66 us against 74 with 256 rows).
  // From 512 rows on (prefill steps of 512 to 960 tokens as a whole: 2.4 to 6.8 % faster at
  // the 7B shape, 3 to 4.6 % at the 32B shape; from 256 rows a step of 384 tokens would be
  // 13 % slower at the 7B shape: the estimates are not fitted there) and an inner size of
  // 896, the shortest measured (steps of 1024 / 4096 / 8192 tokens of the 0.5B shape: 5.8 /
  // 3.5 / 5.8 % faster, 576 and 2048 unchanged).  (The same two groups of waves on a 128 x
  // 256 tile, 64 x 64 a wave, are as fast as the 128 x 256 tile above and no faster: a wave
  // then reads as many bytes from LDS per MFMA as there, and LDS is the limit of both.)
  // ... and from 129 rows on for a wide matrix, where one or two tiles of rows already fill the
  // chip (192 / 256 / 384 rows of 55296 x 5120: 153 / 171 / 261 us against 187 / 199 / 274 with the
  // best of the others; of 59136 x 8192: 229 / 263 / 392 against 305 / 316 / 437)
  const bool pp_rows = M >= g_pp_min_rows || (g_pp_min_rows == 512 && M > 128 && N >= 16384);
  if (pp_rows && K >= PP_MIN_INNER && K <= DIRECT_MAX_INNER && !g_without_wide) {
    // (the estimates of the other tiles, fitted at shorter inner sizes, are up to a quarter low from
    // 3,584 on (and 512 rows): 4096 rows of 1536 x 8960 129 us against 147 with their pick, 2048 of 3584 x 18944 268 against 301,
    // 2367 of 2048 x 11008 154 against 181.  Not where the blocks of the 64 x 128 tile nearly find the three places
    // a unit that they have, until an inner size of 8,192: 1400 rows of 3584 x 3584 70 us with it against 76, 768 of 6144 x 4096 64 against 70)
    const bool low = M >= 512 && K >= 3584 && (K >= 8192 || 10 * (long)((M + 63) / 64) * wide > 27L * num_cus);
    double least = tile_cost(best, M, N, K, num_cus, 1) * (low ? 1.25 : 1.0);
    for (int kind = TILE_256; kind <= TILE_192; ++kind) {
      const double c = tile_cost(kind, M, N, K, num_cus, 1);
      if (c < least) {
        least = c;
        best = kind;
      }
    }
  }
  return addressable(best, K);
}

// Few blocks: the estimates above count a block that has its unit to itself, whose chain of K tiles is the time,
// like one of several that share it, and lose 10 % on average (up to 42 %).  Here a unit holds `resident` blocks at a
// time; a round of them takes what the unit needs for all of them (f + K tiles x tk each), or the chain of one (K
// tiles x chain), whichever is more; a block more than the places of a round is a round of its own.  (Counted as a
// share of one, 1400 rows of 2304 x 768 went to 64 x 64, 792 blocks on 768 places, 19.4 us against 15.2 with 64 x
// 128, and 700 of 5632 x 1024 to 128 x 128, 264 blocks, 23.7 against 18.2.)  Fitted to 12,000 products: the four of a layer of 14
// model shapes, 512 to 4096 wide, 65 to 3,000 rows, whole and in two to eight pieces (7, 7 and 6 % rms).  Over 1,200 of them
// the picks lose 1 % to the best tile of gate and up, and with the fold of the pieces 2 and 3 % of the output and down
// product: 512 rows of 896 x 4864 with the norm 17.8 us (64 x 64 in four pieces) against 24.7 (64 x 128 in six, the
// estimates'), 700 of 2048 x 2048 15.8 against 22.5, 100 of 4608 x 3584 17.5 against 22.4.
// Where they are asked (2): up to 1,024 rows of a matrix of less than 32 MB (128 rows: 64 MB) where the blocks of the 64 x 128
// tile find two places a unit; with more, 512 rows of 9728 x 896, the estimates choose as well.  Up to 2,560 rows of
// less than 16 MB and inner sizes to 2,048 (1) a whole product weighs the 64 x 64 tile against the estimates' (2048 rows of
// 1152 x 896 12.0 against 13.7, of 896 x 896 9.4 against 10.6), one in pieces the two of 64 rows; 2048 rows of 896 x 4864 would be taken
// whole, 33.3 us by itself against 39.9 in two pieces with their fold, and inside a prompt's step be slower by 4 us a
// layer.  Beyond that (0) the estimates above.
static int few_blocks_range(int M, int N, int K, int num_cus) {
  const double bytes = (double)N * K * 2.0;
  if (g_force_tile != 0 || (long)((M + 63) / 64) * ((N + 127) / 128) > 2L * num_cus) return 0;
  if ((M <= 1024 && bytes < 32e6) || (M <= 128 && bytes < 64e6)) return 2;
  return M <= 2560 && K <= 2048 && bytes < 16e6 ? 1 : 0;
}
static double few_blocks_cost(int kind, int M, int N, int K, int num_cus, int pieces) {
  static const struct {
    double L, chain, f, tk;
    int resident;
  } fit[3] = {{4.78, 0.357, 0.09, 0.234, 3}, {5.87, 0.5, 0.5, 0.327, 3}, {6.89, 0.735, 1.25, 0.478, 2}};
  const auto& p = fit[kind];
  const double blocks = (double)((M + TILE_MODELS[kind].bm - 1) / TILE_MODELS[kind].bm) *
                        ((N + TILE_MODELS[kind].bn - 1) / TILE_MODELS[kind].bn) * pieces;
  const int nk = ((K + 63) / 64 + pieces - 1) / pieces;
  auto round_of = [&](double share) {           // share: blocks a unit
    const double together = share * (p.f + nk * p.tk), alone = nk * p.chain;
    return together > alone ? together : alone;
  };
  const double share = blocks / num_cus, rounds = floor(share / p.resident + 1e-9);
  const double last = share - rounds * p.resident;
  double t = rounds * round_of(p.resident);
  if (last > 1e-6) t += round_of(ceil(last - 1e-9));
  const double read = (double)N * K * 2.0 / CHIP_STREAM;
  return p.L + (t > read ? t : read);
}

static int choose_tile(int M, int N, int K, int num_cus) {
  int kind = estimated_tile(M, N, K, num_cus);
  const int range = kind <= TILE_128 ? few_blocks_range(M, N, K, num_cus) : 0;
  if (range)
    for (int other = TILE_64; other <= (range == 2 ? TILE_128 : TILE_64); ++other)
      if (few_blocks_cost(other, M, N, K, num_cus, 1) < few_blocks_cost(kind, M, N, K, num_cus, 1)) kind = other;
  return addressable(kind, K);
}

// The tile of a product that is written into the cache by heads of d: that, or where no head fits it the
// estimates' (a head of 128 in a tile of 128 columns saves the kernel that rotates and writes).
static int heads_tile(int M, int N, int K, int d, int num_cus) {
  const int kind = choose_tile(M, N, K, num_cus);
  return TILE_MODELS[kind].bn % d == 0 ? kind : estimated_tile(M, N, K, num_cus);
}

// The tile of a product that is neither cut into pieces nor written into the cache by heads (those need a
// width that heads divide): the rule for few rows of a wide matrix, else the estimates.
static int plain_tile(int M, int N, int K, int num_cus) {
  if (g_force_tile >= 134 && g_force_tile <= 137) return TILE_64x96 + (g_force_tile - 134);
  const int one_round = g_force_tile == 0 && !g_without_wide ? one_round_tile(M, N, K, num_cus) : -1;
  if (one_round >= 0) return one_round;
  return choose_tile(M, N, K, num_cus);
}
// The tiles of eight waves by direct loads in place of the tile that the estimates, the plan or a rule above named, whose prices
// and answers are those of the tiles that they choose among; these are faster where all their blocks find a place at once.
// Every sum keeps its order, so the results are the same to the bit.
//   128 x 128, a block a unit, in place of 64 x 128 and 128 x 128 in one round, whole or in pieces (beyond 64 rows; us
//   before / with it): 384 rows of 9728 x 896 13.6 / 11.8, 256 of 11008 x 2048 24.3 / 21.1, 2,048 of 896 x 4864 in two pieces
//   32.0 / 26.8, 384 of 2048 x 11008 in four 34.5 / 27.5, 457 of 3584 x 18944 in two 114 / 84.  Beyond one round it loses (512 of
//   9728 x 896, 304 blocks, 17.6 / 21.2), and where the blocks of 64 x 128 find a unit each, whose chains are half as long,
//   as long as the matrix is small (656 of 2048 x 1536, 176 blocks, as q/k/v 16.0 / 17.2, 762 of 2560 x 2048 19.8 / 21.3, 1,384 of 896 x 4864
//   36.4 / 37.6; from 24 MB on W read once a tile of rows counts for more: 154 of 4608 x 3584, 108, 25.1 / 22.8, 520 of 2048 x 11008, 144, 90.9 / 81.8).
//   Over 376 products drawn at random 0.83 of the time, 1.04 at most.
//   192 x 128, two blocks a unit, in place of a 64 x 128 tile of more than two blocks a unit where its own find a unit each: 512 rows
//   of 9728 x 896 17.6 / 15.0, 1,024 of 4864 x 896 18.2 / 15.2, 384 of 11008 x 2048 32.5 / 28.5; and of 192 x 256 whose last round is
//   less than half full, of up to three, at inner sizes to 2,048: 1,900 of 9728 x 896 43.8 / 39.0, 900 of 17920 x 1536 63.4 / 56.1, 1,536
//   of 11008 x 2048 77.9 / 74.2 (not 1,024 of 17920 x 1536, 1.64 rounds, 66.8 / 69.2; 384 of 37888 x 3584 137 / 141).
//   128 x 192, a block a unit, where 192 x 128 has more than units: 640 of 9728 x 896 18.7 / 16.7, 256 of 17920 x 1536 26.8 / 23.3,
//   512 of 11008 x 2048 34.2 / 32.0.
// (Weights from memory and not from the caches.)
static int direct_tile(int kind, int M, int N, int K, int pieces, bool heads, int num_cus) {
  const long UNITS = num_cus;
  if (K > DIRECT_MAX_INNER) return kind;
  if (g_force_tile >= 138 && g_force_tile <= 140) {
    const int forced = TILE_DIRECT_128 + (g_force_tile - 138);
    // (heads: columns that they divide, as they divide those of the tile that was named)
    return heads && (forced != TILE_DIRECT_128 || TILE_MODELS[kind].bn > 128) ? kind : forced;
  }
  if (g_force_tile != 0 || g_without_wide || M <= 64) return kind;
  auto blocks = [&](int bm, int bn) { return (long)((M + bm - 1) / bm) * ((N + bn - 1) / bn) * pieces; };
  if ((kind == TILE_128 || (kind == TILE_64x128 && (blocks(64, 128) > UNITS || (double)N * K * 2.0 >= 24e6))) &&
      blocks(128, 128) <= UNITS)
    return TILE_DIRECT_128;
  if (heads) return kind;
  if (kind == TILE_64x128 && blocks(64, 128) > 2 * UNITS) {
    if (blocks(192, 128) <= UNITS) return TILE_DIRECT_192x128;
    if (blocks(128, 192) <= UNITS) return TILE_DIRECT_128x192;
  }
  const long large = blocks(192, 256), last = large % UNITS;
  if (kind == TILE_192 && pieces == 1 && K <= 2048 && large > UNITS && large < 3 * UNITS && last > 0 && 2 * last <= UNITS)
    return TILE_DIRECT_192x128;
  return kind;
}
// ... its code above (for tests; -1: the tile stays)
extern "C" int llmlab_direct_tile(int kind, int M, int N, int K, int pieces, int heads, int num_cus) {
  const int tile = direct_tile(kind, M, N, K, pieces, heads != 0, num_cus > 0 ? num_cus : 256);
  return tile == kind ? -1 : tile;
}

// The width of the tile that such a product is launched with (for tests).
extern "C" int llmlab_plain_tile(int M, int N, int K, int num_cus) {
  if (num_cus <= 0) num_cus = 256;
  return TILE_MODELS[direct_tile(addressable(plain_tile(M, N, K, num_cus), K), M, N, K, 1, false, num_cus)].bn;
}

template <int EPI>
static void launch_tile(int kind, const bf16_t* A, const bf16_t* W, const EpiArgs& e, int M, int N, int K,
                        int pieces, int num_cus, hipStream_t stream) {
  kind = direct_tile(addressable(kind, K), M, N, K, pieces, EPI == EPI_QKV, num_cus);      // (a tile that the caller names)
  const TileModel& t = TILE_MODELS[kind];
  dim3 grid((N + t.bn - 1) / t.bn, (M + t.bm - 1) / t.bm, pieces);
  if (kind == TILE_64)
    hipLaunchKernelGGL((gemm_bf16_ring<EPI>), grid, dim3(256), 0, stream, A, W, e, M, N, K);
  else if (kind == TILE_64x128)
    hipLaunchKernelGGL((gemm_bf16_tiled<64, 128, 64, 1, 4, EPI>), grid, dim3(256), 0, stream, A, W, e, M, N, K);
  else if (kind == TILE_128)
    hipLaunchKernelGGL((gemm_bf16_tiled<128, 128, 64, 1, 4, EPI>), grid, dim3(256), 0, stream, A, W, e, M, N, K);
  else if (kind == TILE_128x256)
    hipLaunchKernelGGL((gemm_bf16_tiled<128, 256, 64, 1, 8, EPI>), grid, dim3(512), 0, stream, A, W, e, M, N, K);
  else if (kind == TILE_256)
    hipLaunchKernelGGL((gemm_bf16_pingpong<256, EPI>), grid, dim3(512), 0, stream, A, W, e, M, N, K);
  else if (kind == TILE_192)
    hipLaunchKernelGGL((gemm_bf16_pingpong<192, EPI>), grid, dim3(512), 0, stream, A, W, e, M, N, K);
  else if (kind == TILE_DIRECT_128)
    hipLaunchKernelGGL((gemm_bf16_ring<EPI, 128, 128, 3, 4, 2, 2>), grid, dim3(512), 0, stream, A, W, e, M, N, K);
  if constexpr (EPI != EPI_QKV) {
    if (kind == TILE_DIRECT_128x192)
      hipLaunchKernelGGL((gemm_bf16_ring<EPI, 128, 192, 3, 4, 2, 2>), grid, dim3(512), 0, stream, A, W, e, M, N, K);
    else if (kind == TILE_DIRECT_192x128)
      hipLaunchKernelGGL((gemm_bf16_ring<EPI, 192, 128, 2, 4, 2, 4>), grid, dim3(512), 0, stream, A, W, e, M, N, K);
  }
  if constexpr (EPI != EPI_QKV && EPI != EPI_PART) {      // (plain_tile: whole products only)
    if (kind == TILE_64x96)
      hipLaunchKernelGGL((gemm_bf16_tiled<64, 96, 64, 1, 3, EPI>), grid, dim3(192), 0, stream, A, W, e, M, N, K);
    else if (kind == TILE_64x160)
      hipLaunchKernelGGL((gemm_bf16_tiled<64, 160, 64, 1, 5, EPI>), grid, dim3(320), 0, stream, A, W, e, M, N, K);
    else if (kind == TILE_64x224)
      hipLaunchKernelGGL((gemm_bf16_tiled<64, 224, 64, 1, 7, EPI>), grid, dim3(448), 0, stream, A, W, e, M, N, K);
    else if (kind == TILE_128x160)
      hipLaunchKernelGGL((gemm_bf16_tiled<128, 160, 64, 1, 5, EPI>), grid, dim3(320), 0, stream, A, W, e, M, N, K);
  }
}

// Grouped products: `members` matrices [N, K] of equal shape lie one below the other in the packed
// W (every member whole strips of 16 rows: N % 16 == 0); tile t of bm rows of the product belongs
// to member tile_member[t] (-1: empty, its block leaves at once); row m reads row rows_index[m]
// of x (null: row m).  out has M rows (a multiple of bm).  Epilogues: SWIGLU, F32, and STORE
// (compute dtype; epilogue 6: through max(z, 0)^2 first; epilogue 8: SWIGLU as the clamped pair).
extern "C" int llmlab_linear_grouped(const void* x, const void* w, int epilogue, void* out, int M, int N, int K,
                                     int ldo, int n_out, const int* tile_member, const int* rows_index, int bm,
                                     int wide, float limit, float slope, float shift, hipStream_t stream) {
  LLMLAB_REQUIRE(M >= 0 && N > 0 && K > 0 && K % 8 == 0 && N % 16 == 0, "linear_grouped: bad sizes M=%d N=%d K=%d", M,
                 N, K);
  LLMLAB_REQUIRE((bm == 64 || bm == 128) && M % bm == 0, "linear_grouped: %d rows in tiles of %d", M, bm);
  if (g_force_tile == 129) wide = 0;
  if (g_force_tile == 131) wide = 1;
  const int act = epilogue == 6 ? 1 : epilogue == 8 ? 3 : 0;
  if (act == 1) epilogue = EPI_STORE;
  if (act == 3) epilogue = EPI_SWIGLU;
  LLMLAB_REQUIRE(epilogue == EPI_SWIGLU || epilogue == EPI_F32 || epilogue == EPI_STORE, "linear_grouped: epilogue %d",
                 epilogue);
  if (epilogue == EPI_SWIGLU)
    LLMLAB_REQUIRE(N % 32 == 0 && n_out > 0 && 2 * ((n_out + 15) / 16 * 16) == N,
                   "linear_grouped(swiglu): %d weight rows do not interleave %d outputs", N, n_out);
  else
    LLMLAB_REQUIRE(n_out <= N && n_out > N - 16, "linear_grouped: n_out %d, N %d", n_out, N);
  LLMLAB_REQUIRE(ldo >= n_out && tile_member != nullptr, "linear_grouped: output stride or tile table");
  if (M == 0) return 0;
  EpiArgs e{out, nullptr, 0, ldo, n_out, 0, 0, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, 0, 0, 0, 0, 0, act,
            tile_member, rows_index, (size_t)(N / 16) * (size_t)((K + 31) / 32) * 512, limit, slope, shift};
  const bf16_t* A = (const bf16_t*)x;
  const bf16_t* W = (const bf16_t*)w;
  // (the columns past n_out of an F32 product are the zero rows that pad a member to whole strips)
  const int cols = epilogue == EPI_SWIGLU ? N : n_out;
  if (epilogue == EPI_STORE) {
    if (bm == 64)
      hipLaunchKernelGGL((gemm_bf16_tiled<64, 64, 64, 2, 2, EPI_STORE, true>), dim3((cols + 63) / 64, M / 64, 1), dim3(256),
                         0, stream, A, W, e, M, cols, K);
    else if (wide)
      hipLaunchKernelGGL((gemm_bf16_tiled<128, 256, 64, 1, 8, EPI_STORE, true>), dim3((cols + 255) / 256, M / 128, 1),
                         dim3(512), 0, stream, A, W, e, M, cols, K);
    else
      hipLaunchKernelGGL((gemm_bf16_tiled<128, 128, 64, 1, 4, EPI_STORE, true>), dim3((cols + 127) / 128, M / 128, 1),
                         dim3(256), 0, stream, A, W, e, M, cols, K);
  } else if (bm == 64) {
    dim3 grid((cols + 63) / 64, M / 64, 1);
    if (epilogue == EPI_SWIGLU)
      hipLaunchKernelGGL((gemm_bf16_tiled<64, 64, 64, 2, 2, EPI_SWIGLU, true>), grid, dim3(256), 0, stream, A, W, e, M,
                         cols, K);
    else
      hipLaunchKernelGGL((gemm_bf16_tiled<64, 64, 64, 2, 2, EPI_F32, true>), grid, dim3(256), 0, stream, A, W, e, M,
                         cols, K);
  } else if (wide) {
    // (tiles of 128 rows and 256 columns, eight waves side by side)
    dim3 grid((cols + 255) / 256, M / 128, 1);
    if (epilogue == EPI_SWIGLU)
      hipLaunchKernelGGL((gemm_bf16_tiled<128, 256, 64, 1, 8, EPI_SWIGLU, true>), grid, dim3(512), 0, stream, A, W, e,
                         M, cols, K);
    else
      hipLaunchKernelGGL((gemm_bf16_tiled<128, 256, 64, 1, 8, EPI_F32, true>), grid, dim3(512), 0, stream, A, W, e, M,
                         cols, K);
  } else {
    dim3 grid((cols + 127) / 128, M / 128, 1);
    if (epilogue == EPI_SWIGLU)
      hipLaunchKernelGGL((gemm_bf16_tiled<128, 128, 64, 1, 4, EPI_SWIGLU, true>), grid, dim3(256), 0, stream, A, W, e,
                         M, cols, K);
    else
      hipLaunchKernelGGL((gemm_bf16_tiled<128, 128, 64, 1, 4, EPI_F32, true>), grid, dim3(256), 0, stream, A, W, e, M,
                         cols, K);
  }
  LLMLAB_LAUNCH_CHECK("linear_grouped");
  return 0;
}

// 65 to 128 rows in pieces: one tile of 128 rows reads W once where two of 64 read it twice, which
// the estimate does not know (128 rows of 3584 x 18944 in pieces: 45 us against 57, a decode
// step of 128 requests of that shape 7.11 ms against 7.30)
static bool takes_one_tile_of_128(int M, int N, int K) {
  return M > 64 && M <= 128 && g_force_tile == 0 && (double)N * K * 2.0 >= 64e6;
}

// The tile of a product that its caller cuts into so many pieces, whatever number the plan below would take
// (q/k/v products of 65 to 384 rows, two at least: 384 rows of 5120 x 3072 33.8 us in two with this tile, 40.5 with that of the whole product).
extern "C" int llmlab_pieces_tile(int M, int N, int K, int num_cus, int pieces) {
  if (num_cus <= 0) num_cus = 256;
  int kind = choose_tile(M, N, K, num_cus);
  if (takes_one_tile_of_128(M, N, K)) kind = TILE_128;
  else if (kind <= TILE_128 && few_blocks_range(M, N, K, num_cus) == 2)
    for (int other = TILE_64; other <= TILE_128; ++other)
      if (few_blocks_cost(other, M, N, K, num_cus, pieces) < few_blocks_cost(kind, M, N, K, num_cus, pieces)) kind = other;
  return addressable(kind, K);
}

// Whether (and into how many pieces along K) a product that adds into float32 rows should
// be left unsummed, and with which tile: out = {pieces (1: no), tile kind}, before direct_tile; in one piece the kind is that
// of a whole product (choose_tile; up to 128 rows of a wide matrix one_round_tile's widths go before it, which make
// no pieces).  A piece costs a write and a read of the result by whoever sums it up later.
extern "C" void llmlab_linear_plan(int M, int N, int K, int num_cus, int max_pieces, int min_tiles_per_piece,
                                   int* out) {
  if (num_cus <= 0) num_cus = 256;
  const int nk = (K + 63) / 64;
  // (a piece's write and read; the second is the price of large results, where that of the first kept whole what is
  // faster in pieces: with the norm 900 rows of 3584 x 3584 45 us in three pieces against 53 whole, 1400 of 4096 x 4096 66
  // in two against 85)
  const double piece = (double)M * N * (M < 512 || (double)M * N < 2e6 ? 2.2e-6 : 1.5e-6) + 0.3;
  int best_kind = choose_tile(M, N, K, num_cus), best_pieces = 1;
  // (the estimates of the tiles below 256 rows are low at long inner sizes, as in estimated_tile)
  auto cost = [&](int kind, int pieces) {
    return tile_cost(kind, M, N, K, num_cus, pieces) * (kind < TILE_256 && M >= 512 && K >= 3584 ? 1.25 : 1.0);
  };
  double best_cost = cost(best_kind, 1);
  const bool one_tile_of_128 = takes_one_tile_of_128(M, N, K);
  if (one_tile_of_128) {
    best_kind = TILE_128;
    best_cost = cost(TILE_128, 1);
  }
  for (int kind = TILE_64x128; kind < TILE_KINDS; ++kind) {
    if (kind == TILE_128x256) continue;
    if (one_tile_of_128 && kind != TILE_128) continue;
    if (kind >= TILE_256 && !(M >= g_pp_min_rows && K >= PP_MIN_INNER && K <= DIRECT_MAX_INNER && !g_without_wide)) continue;
    if (g_force_tile != 0 && kind != choose_tile(M, N, K, num_cus)) continue;
    for (int s = 2; s <= max_pieces; ++s) {
      if ((nk + s - 1) / s < min_tiles_per_piece) break;
      const double c = cost(kind, s) + s * piece;
      if (c < best_cost) {
        best_cost = c;
        best_kind = kind;
        best_pieces = s;
      }
    }
  }
  // Two or three well-filled tiles of 128 rows of a matrix 5,120 to 16,383 wide: four pieces of
  // the 128 x 128 tile, which the estimate prices too high there (with the norm that folds
  // them, 384 rows of 8192 x 29568: 248 us against 365 whole with 64 x 128; of 5120 x 27648:
  // 150 against 183 in two pieces; 256 rows of 8192 x 8192: 65 against 70; at 3,584 columns
  // it loses as often as it wins).  Inside prefill steps of 256 / 320 / 384 tokens of the 14B
  // shape 14.5 -> 14.2 / 16.5 -> 15.5 / 17.6 -> 16.7 ms, of the 32B shape 27.3 -> 27.0 / 34.0 ->
  // 31.2 / 35.9 -> 33.8; at 192 rows the 32B shape loses 5 % with it, hence from 256 on.
  if (M >= 256 && M <= 384 && 4 * M >= 3 * ((M + 127) / 128) * 128 && N >= 5120 && N < 16384 &&
      g_force_tile == 0 && max_pieces >= 4 && (nk + 3) / 4 >= min_tiles_per_piece) {
    best_kind = TILE_128;
    best_pieces = 4;
  }
  // One tile of rows in pieces: the small tile, if its blocks still find a compute unit
  // each (17 to 64 rows of matrices from 9 to 45 MB: 8.6 against 11.0, 12.4 against
  // 15.8, 15.1 against 18.8 us; with more blocks than units it is the slower one)
  if (M <= 64 && best_pieces > 1 && g_force_tile == 0 && (long)((N + 63) / 64) * best_pieces <= num_cus)
    best_kind = TILE_64;
  const int range = best_kind <= TILE_128 ? few_blocks_range(M, N, K, num_cus) : 0;
  if (range) {
    auto folded = [&](int pieces) { return pieces > 1 ? pieces * ((double)M * N * 1.1e-6 + 0.28) : 0.0; };
    double least = few_blocks_cost(best_kind, M, N, K, num_cus, best_pieces) + folded(best_pieces);
    for (int kind = TILE_64; kind <= (range == 2 ? TILE_128 : TILE_64x128); ++kind)
      for (int s = 1; s <= max_pieces && (s == 1 || (nk + s - 1) / s >= min_tiles_per_piece); ++s) {
        const double c = few_blocks_cost(kind, M, N, K, num_cus, s) + folded(s);
        if (c < least) {
          least = c;
          best_kind = kind;
          best_pieces = s;
        }
      }
  }
  if (best_pieces == 1) best_kind = choose_tile(M, N, K, num_cus);
  out[0] = best_pieces;
  out[1] = addressable(best_kind, K);
}

// The same for a float32 product (of more rows than the few-row kernel takes).
extern "C" void llmlab_linear_plan_f32(int M, int N, int K, int num_cus, int max_pieces, int min_steps_per_piece,
                                       int* out) {
  const F32Plan plan = f32_plan(M, N, K, num_cus > 0 ? num_cus : 256, max_pieces, min_steps_per_piece);
  out[0] = plan.pieces;
  out[1] = plan.tile;
}

// q/k/v projection of many rows with bias, rotation and cache write in the epilogue
// (bfloat16).  The tile is chosen as for any product; the head size must divide it.
extern "C" int llmlab_linear_qkv(const void* x, const void* w, const void* bias, int bias_dtype, void* q_out,
                                 int M, int N, int K, int ldo, const float* inv_freq, const int* positions,
                                 const int* row_req, const int* table, int table_stride, int page_size,
                                 void* kcache, void* vcache, int nq, int nkv, int d, int num_cus,
                                 hipStream_t stream) {
  LLMLAB_REQUIRE(M >= 0 && N > 0 && K > 0 && K % 8 == 0, "linear_qkv: bad sizes M=%d N=%d K=%d", M, N, K);
  LLMLAB_REQUIRE(d >= 16 && d % 16 == 0 && nq > 0 && nkv > 0 && N == (nq + 2 * nkv) * d && ldo >= nq * d,
                 "linear_qkv: %d + 2 x %d heads of %d do not make %d columns (row stride %d)", nq, nkv, d, N, ldo);
  LLMLAB_REQUIRE((kcache == nullptr) == (vcache == nullptr), "linear_qkv: both caches or none");
  LLMLAB_REQUIRE(positions != nullptr && (kcache == nullptr || (table && row_req && page_size > 0)),
                 "linear_qkv: positions and block table are needed");
  LLMLAB_REQUIRE(((uintptr_t)x % 16 == 0) && ((uintptr_t)w % 16 == 0) &&
                 ((uintptr_t)kcache % 16 == 0) && ((uintptr_t)vcache % 16 == 0),
                 "linear_qkv: operands must be 16-byte aligned");
  if (M == 0) return 0;
  if (num_cus <= 0) num_cus = 256;
  EpiArgs e{q_out, bias, bias_dtype == DT_BF16, ldo, N, 0, 0, inv_freq, positions, row_req, table,
            (bf16_t*)kcache, (bf16_t*)vcache, table_stride, page_size, nq, nkv, d};
  const int kind = heads_tile(M, N, K, d, num_cus);
  LLMLAB_REQUIRE(TILE_MODELS[kind].bn % d == 0, "linear_qkv: heads of %d do not divide the tile of %d columns", d,
                 TILE_MODELS[kind].bn);
  launch_tile<EPI_QKV>(kind, (const bf16_t*)x, (const bf16_t*)w, e, M, N, K, 1, num_cus, stream);
  LLMLAB_LAUNCH_CHECK("linear_qkv");
  return 0;
}

// The width of the tile (64, 128 or 256 columns) that the estimates name for a product of these sizes (for tests; direct_tile may
// put another in its place) ...
extern "C" int llmlab_linear_tile(int M, int N, int K, int num_cus) {
  if (num_cus <= 0) num_cus = 256;
  return TILE_MODELS[choose_tile(M, N, K, num_cus)].bn;
}

// ... and that llmlab_linear_qkv takes for heads of d, and keeps where direct_tile puts another in its place: for callers that must
// know whether a head fits it.
extern "C" int llmlab_linear_heads_tile(int M, int N, int K, int d, int num_cus) {
  return TILE_MODELS[heads_tile(M, N, K, d > 0 ? d : 1, num_cus > 0 ? num_cus : 256)].bn;
}

// The compute units of the chip (for a call that does not name them).
static int chip_units() {
  static const int units = [] {
    int device = 0, n = 0;
    const bool known = hipGetDevice(&device) == hipSuccess &&
                       hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess;
    return known && n > 0 ? n : 256;
  }();
  return units;
}

// parts[z] = x[:, K_z] . W[:, K_z]^T for `ksplit` ranges K_z of the inner size (whole K
// tiles of 64 each, in float32 whole steps of 32); bias in parts[0].  `tile` as llmlab_linear_plan gives it.
extern "C" int llmlab_linear_partials(const void* x, const void* w, int dtype, float* parts, const void* bias,
                                      int bias_dtype, int M, int N, int K, int ldo, int ksplit,
                                      size_t part_stride, int tile, hipStream_t stream) {
  LLMLAB_REQUIRE(M >= 0 && N > 0 && K > 0 && (dtype == DT_F32 || K % 8 == 0), "linear_partials: bad sizes M=%d N=%d K=%d",
                 M, N, K);
  LLMLAB_REQUIRE(ksplit >= 1 && ksplit <= 16 && ldo >= N && part_stride >= (size_t)M * ldo,
                 "linear_partials: %d pieces, row stride %d", ksplit, ldo);
  LLMLAB_REQUIRE(tile >= TILE_64 && tile < TILE_KINDS, "linear_partials: unknown tile %d", tile);
  if (dtype == DT_F32) {
    LLMLAB_REQUIRE(tile == TILE_64 || tile == TILE_128 || tile == TILE_128x256, "linear_partials(float32): tile %d", tile);
    if (M == 0) return 0;
    const int steps = (K + 31) / 32;
    EpiArgs e{parts, bias, bias_dtype == DT_BF16, ldo, N, (steps + ksplit - 1) / ksplit, part_stride};
    launch_f32_split<EPI_PART>(tile, (const float*)x, (const float*)w, e, M, N, K, ksplit, stream);
    LLMLAB_LAUNCH_CHECK("linear_partials(float32)");
    return 0;
  }
  LLMLAB_REQUIRE(((uintptr_t)x % 16 == 0) && ((uintptr_t)w % 16 == 0),
                 "linear_partials: operands must be 16-byte aligned");
  if (M == 0) return 0;
  const int nk = (K + 63) / 64;
  EpiArgs e{parts, bias, bias_dtype == DT_BF16, ldo, N, (nk + ksplit - 1) / ksplit, part_stride,
            nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, 0, 0, 0, 0, 0};
  launch_tile<EPI_PART>(tile, (const bf16_t*)x, (const bf16_t*)w, e, M, N, K, ksplit, chip_units(), stream);
  LLMLAB_LAUNCH_CHECK("linear_partials");
  return 0;
}

// x [M,K] (dtype), w [N,K] (float32: row-major; bfloat16: packed); epilogue selects what `out` is.  For SWIGLU N
// is the number of interleaved weight rows (2 * ceil16(n_out)).
extern "C" int llmlab_linear(const void* x, const void* w, int dtype, int epilogue, void* out,
                             const void* bias, int bias_dtype, int M, int N, int K, int ldo, int n_out,
                             int num_cus, float limit, float slope, float shift, hipStream_t stream) {
  LLMLAB_REQUIRE(M >= 0 && N > 0 && K > 0, "linear: bad sizes M=%d N=%d K=%d", M, N, K);
  // 6 at this interface: STORE with the squared-relu activation on the way; 7: the paired
  // product whose gate goes through gelu (tanh form); 8: the clamped pair with its three constants
  const int act = epilogue == 6 ? 1 : epilogue == 7 ? 2 : epilogue == 8 ? 3 : 0;
  if (act == 1) epilogue = EPI_STORE;
  if (act > 1) epilogue = EPI_SWIGLU;
  LLMLAB_REQUIRE(epilogue >= 0 && epilogue <= 3, "linear: unknown epilogue %d", epilogue);
  if (epilogue == EPI_SWIGLU) {
    LLMLAB_REQUIRE(N % 32 == 0 && n_out > 0 && 2 * ((n_out + 15) / 16 * 16) == N,
                   "linear(swiglu): %d weight rows do not interleave %d outputs", N, n_out);
    LLMLAB_REQUIRE(bias == nullptr, "linear(swiglu): no bias");
  } else {
    LLMLAB_REQUIRE(n_out == N, "linear: n_out %d != N %d", n_out, N);
  }
  LLMLAB_REQUIRE(ldo >= n_out, "linear: output row stride %d < %d columns", ldo, n_out);
  if (M == 0) return 0;
  EpiArgs e{out, bias, bias_dtype == DT_BF16, ldo, n_out, 0, 0,
            nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, 0, 0, 0, 0, 0, act, nullptr, nullptr, 0, limit, slope, shift};
  if (num_cus <= 0) num_cus = 256;
  if (dtype == DT_BF16) {
    LLMLAB_REQUIRE(K % 8 == 0, "linear(bfloat16): inner size %d must be a multiple of 8", K);
    LLMLAB_REQUIRE(((uintptr_t)x % 16 == 0) && ((uintptr_t)w % 16 == 0),
                   "linear(bfloat16): operands must be 16-byte aligned");
    const bf16_t* A = (const bf16_t*)x;
    const bf16_t* W = (const bf16_t*)w;
    const int kind = plain_tile(M, N, K, num_cus);
    switch (epilogue) {
      case EPI_STORE: launch_tile<EPI_STORE>(kind, A, W, e, M, N, K, 1, num_cus, stream); break;
      case EPI_RESID: launch_tile<EPI_RESID>(kind, A, W, e, M, N, K, 1, num_cus, stream); break;
      case EPI_F32: launch_tile<EPI_F32>(kind, A, W, e, M, N, K, 1, num_cus, stream); break;
      default: launch_tile<EPI_SWIGLU>(kind, A, W, e, M, N, K, 1, num_cus, stream); break;
    }
  } else {
    const float* A = (const float*)x;
    const float* W = (const float*)w;
    if (M <= F32_ROWS_MAX) {
      switch (epilogue) {
        case EPI_STORE: launch_f32_rows<EPI_STORE>(A, W, e, M, N, K, num_cus, stream); break;
        case EPI_RESID: launch_f32_rows<EPI_RESID>(A, W, e, M, N, K, num_cus, stream); break;
        case EPI_F32: launch_f32_rows<EPI_F32>(A, W, e, M, N, K, num_cus, stream); break;
        default: launch_f32_rows<EPI_SWIGLU>(A, W, e, M, N, K, num_cus, stream); break;
      }
      LLMLAB_LAUNCH_CHECK("linear(float32, few rows)");
      return 0;
    }
    switch (epilogue) {
      case EPI_STORE: launch_f32_tiled<EPI_STORE>(A, W, e, M, N, K, num_cus, stream); break;
      case EPI_RESID: launch_f32_tiled<EPI_RESID>(A, W, e, M, N, K, num_cus, stream); break;
      case EPI_F32: launch_f32_tiled<EPI_F32>(A, W, e, M, N, K, num_cus, stream); break;
      default: launch_f32_tiled<EPI_SWIGLU>(A, W, e, M, N, K, num_cus, stream); break;
    }
  }
  LLMLAB_LAUNCH_CHECK("linear");
  return 0;
}
