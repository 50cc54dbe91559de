// Merge of two partial attentions computed over disjoint key sets.
// Stands in for add_self_attentions (src/attn_utils.py:6-24 of the reference):
//   c = 1 / (1 + exp(lse2 - lse1)); attn = c*attn1 + (1-c)*attn2; lse = lse1 - log(c + eps).
// c is rounded to the attention's type before it is used, as the reference does (src/attn_utils.py:21);
// the rest is fp32, with the same eps = 2^-23 inside the log.  One 8-element piece (16 bytes) per lane.
#include "ha_common.h"

#include <algorithm>

namespace {

template <typename T>
__global__ __launch_bounds__(256) void lse_merge_kernel(const T* a1, const float* l1, const T* a2, const float* l2,
                                                        T* ao, float* lo, int64_t rows,
                                                        int pieces, int64_t s1, int64_t s2, int64_t so,
                                                        int64_t ls1, int64_t ls2, int64_t lso) {
  typedef typename ElemTraits<T>::vec8 vec8;
  const int64_t item = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t row = item / pieces;
  const int piece = (int)(item % pieces);
  if (row >= rows) return;
  const float x1 = l1[row * ls1], x2 = l2[row * ls2];
  const float c = (float)(T)(1.0f / (1.0f + __expf(x2 - x1)));
  const vec8 v1 = *reinterpret_cast<const vec8*>(a1 + row * s1 + piece * 8);
  const vec8 v2 = *reinterpret_cast<const vec8*>(a2 + row * s2 + piece * 8);
  vec8 r;
#pragma unroll
  for (int e = 0; e < 8; ++e) r[e] = (T)(c * (float)v1[e] + (1.0f - c) * (float)v2[e]);
  *reinterpret_cast<vec8*>(ao + row * so + piece * 8) = r;
  if (piece == 0) lo[row * lso] = x1 - __logf(c + 1.1920929e-07f);
}

}  // namespace

extern "C" int ha_lse_merge(const void* attn1, const float* lse1, const void* attn2, const float* lse2,
                            void* attn_out, float* lse_out, int64_t rows, int64_t d, int64_t attn1_stride,
                            int64_t attn2_stride, int64_t out_stride, int64_t lse1_stride, int64_t lse2_stride,
                            int64_t lse_out_stride, int dtype, void* stream) {
  HA_REQUIRE(attn1 && lse1 && attn2 && lse2 && attn_out && lse_out, HA_ERR_NULL, "ha_lse_merge: null pointer");
  HA_REQUIRE(dtype == HA_F16 || dtype == HA_BF16, HA_ERR_DTYPE, "ha_lse_merge: Only support fp16 and bf16");
  HA_REQUIRE(rows > 0 && d > 0 && d % 8 == 0, HA_ERR_SHAPE, "ha_lse_merge: rows > 0 and d % 8 == 0 required");
  HA_REQUIRE(attn1_stride % 8 == 0 && attn2_stride % 8 == 0 && out_stride % 8 == 0 &&
                 ((uintptr_t)attn1 % 16) == 0 && ((uintptr_t)attn2 % 16) == 0 && ((uintptr_t)attn_out % 16) == 0,
             HA_ERR_SHAPE, "ha_lse_merge: rows must be 16-byte aligned");
  const int pieces = (int)(d / 8);
  const int64_t items = rows * pieces;
  // In place, the lanes of a row read its log-sum-exps before one of them writes the merged one: that
  // holds inside a wave, so a row's d/8 lanes must not straddle two waves.
  const bool in_place = lse_out == lse1 || lse_out == lse2 || attn_out == attn1 || attn_out == attn2;
  HA_REQUIRE(!in_place || 64 % pieces == 0, HA_ERR_UNSUPPORTED,
             "ha_lse_merge: in place needs a head dimension of 8, 16, 32, 64, 128, 256 or 512");
  HA_REQUIRE((items + 255) / 256 < (1ll << 31), HA_ERR_SHAPE, "ha_lse_merge: too many rows");
  dim3 grid((unsigned)((items + 255) / 256));
  hipStream_t s = (hipStream_t)stream;
  if (dtype == HA_F16)
    hipLaunchKernelGGL((lse_merge_kernel<f16_t>), grid, dim3(256), 0, s, (const f16_t*)attn1, lse1,
                       (const f16_t*)attn2, lse2, (f16_t*)attn_out, lse_out, rows, pieces, attn1_stride,
                       attn2_stride, out_stride, lse1_stride, lse2_stride, lse_out_stride);
  else
    hipLaunchKernelGGL((lse_merge_kernel<bf16_t>), grid, dim3(256), 0, s, (const bf16_t*)attn1, lse1,
                       (const bf16_t*)attn2, lse2, (bf16_t*)attn_out, lse_out, rows, pieces, attn1_stride,
                       attn2_stride, out_stride, lse1_stride, lse2_stride, lse_out_stride);
  return ha_launch_status("ha_lse_merge");
}

// The same merge for rows that come in equal segments with their own strides (the second halves of
// the heads of a (batch, heads, n, d) tensor, say), in place if wanted, with the weight c of the first
// input written out as well: what the causal recursion needs per level, in one pass.  c is rounded to
// the attention's type before it is used, as the reference does (src/attn_utils.py:21).
namespace {

template <typename T>
__global__ __launch_bounds__(256) void lse_merge_segments_kernel(const T* a1, const float* l1, const T* a2,
                                                                 const float* l2, T* ao, float* lo,
                                                                 float* __restrict__ wo, int64_t rows,
                                                                 int64_t seg_len, int pieces, int64_t a1_ss, int64_t a1_rs,
                                                                 int64_t a2_ss, int64_t a2_rs, int64_t ao_ss, int64_t ao_rs,
                                                                 int64_t l1_ss, int64_t l2_ss, int64_t lo_ss, int64_t wo_ss) {
  typedef typename ElemTraits<T>::vec8 vec8;
  const int64_t item = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t row = item / pieces;
  const int piece = (int)(item % pieces);
  if (row >= rows) return;
  const int64_t seg = row / seg_len, i = row - seg * seg_len;
  const float x1 = l1[seg * l1_ss + i], x2 = l2[seg * l2_ss + i];
  const float c = (float)(T)(1.0f / (1.0f + __expf(x2 - x1)));
  const vec8 v1 = *reinterpret_cast<const vec8*>(a1 + seg * a1_ss + i * a1_rs + piece * 8);
  const vec8 v2 = *reinterpret_cast<const vec8*>(a2 + seg * a2_ss + i * a2_rs + piece * 8);
  vec8 r;
#pragma unroll
  for (int e = 0; e < 8; ++e) r[e] = (T)(c * (float)v1[e] + (1.0f - c) * (float)v2[e]);
  *reinterpret_cast<vec8*>(ao + seg * ao_ss + i * ao_rs + piece * 8) = r;
  if (piece == 0) {
    lo[seg * lo_ss + i] = x1 - __logf(c + 1.1920929e-07f);
    if (wo) wo[seg * wo_ss + i] = c;
  }
}

}  // namespace

extern "C" int ha_lse_merge_segments(const void* attn1, const float* lse1, const void* attn2, const float* lse2,
                                     void* attn_out, float* lse_out, float* weight_out, int64_t segs, int64_t seg_len,
                                     int64_t d, int64_t attn1_seg_stride, int64_t attn1_row_stride,
                                     int64_t attn2_seg_stride, int64_t attn2_row_stride, int64_t out_seg_stride,
                                     int64_t out_row_stride, int64_t lse1_seg_stride, int64_t lse2_seg_stride,
                                     int64_t lse_out_seg_stride, int64_t weight_seg_stride, int dtype, void* stream) {
  HA_REQUIRE(attn1 && lse1 && attn2 && lse2 && attn_out && lse_out, HA_ERR_NULL, "ha_lse_merge_segments: null pointer");
  HA_REQUIRE(dtype == HA_F16 || dtype == HA_BF16, HA_ERR_DTYPE, "ha_lse_merge_segments: Only support fp16 and bf16");
  HA_REQUIRE(segs > 0 && seg_len > 0 && d > 0 && d % 8 == 0, HA_ERR_SHAPE,
             "ha_lse_merge_segments: segs, seg_len > 0 and d % 8 == 0 required");
  const int64_t strides[] = {attn1_seg_stride, attn1_row_stride, attn2_seg_stride, attn2_row_stride, out_seg_stride, out_row_stride};
  for (int64_t s : strides) HA_REQUIRE(s % 8 == 0, HA_ERR_SHAPE, "ha_lse_merge_segments: rows must be 16-byte aligned");
  HA_REQUIRE(((uintptr_t)attn1 % 16) == 0 && ((uintptr_t)attn2 % 16) == 0 && ((uintptr_t)attn_out % 16) == 0, HA_ERR_SHAPE,
             "ha_lse_merge_segments: tensors must be 16-byte aligned");
  const int pieces = (int)(d / 8);
  const int64_t rows = segs * seg_len, items = rows * pieces;
  HA_REQUIRE((items + 255) / 256 < (1ll << 31), HA_ERR_SHAPE, "ha_lse_merge_segments: too many rows");
  // In place, the lanes of a row read its log-sum-exps before one of them writes the merged one: that
  // holds inside a wave, so a row's d/8 lanes must not straddle two waves.
  const bool in_place = lse_out == lse1 || lse_out == lse2 || attn_out == attn1 || attn_out == attn2;
  HA_REQUIRE(!in_place || 64 % pieces == 0, HA_ERR_UNSUPPORTED,
             "ha_lse_merge_segments: in place needs a head dimension of 8, 16, 32, 64, 128, 256 or 512");
  dim3 grid((unsigned)((items + 255) / 256));
  hipStream_t s = (hipStream_t)stream;
  if (dtype == HA_F16)
    hipLaunchKernelGGL((lse_merge_segments_kernel<f16_t>), grid, dim3(256), 0, s, (const f16_t*)attn1, lse1,
                       (const f16_t*)attn2, lse2, (f16_t*)attn_out, lse_out, weight_out, rows, seg_len, pieces,
                       attn1_seg_stride, attn1_row_stride, attn2_seg_stride, attn2_row_stride, out_seg_stride,
                       out_row_stride, lse1_seg_stride, lse2_seg_stride, lse_out_seg_stride, weight_seg_stride);
  else
    hipLaunchKernelGGL((lse_merge_segments_kernel<bf16_t>), grid, dim3(256), 0, s, (const bf16_t*)attn1, lse1,
                       (const bf16_t*)attn2, lse2, (bf16_t*)attn_out, lse_out, weight_out, rows, seg_len, pieces,
                       attn1_seg_stride, attn1_row_stride, attn2_seg_stride, attn2_row_stride, out_seg_stride,
                       out_row_stride, lse1_seg_stride, lse2_seg_stride, lse_out_seg_stride, weight_seg_stride);
  return ha_launch_status("ha_lse_merge_segments");
}

// All merges of the causal recursion in one pass over the rows.
// A row of a (batch, heads, n, d) tensor takes part in the un-masked call of level j (segments of n / 2^j
// rows) iff it lies in the second half of its segment.  Deepest level first, as the recursion returns
// (hyper_attention.py:86-89), its leaf result is merged with the results of those calls, each merge with the
// arithmetic of lse_merge_segments_kernel (weight rounded to the attention's type, merged rows rounded
// after every level).  All per-level arrays have the layout of the whole tensors; rows outside a level's
// second halves are neither read nor written.
//
// For a backward pass the row's weights are turned into shifted log-sum-exps on the way: the gradient of the
// output reaches the call of level j scaled by w_j = (1 - c_j) * prod of c_i over the shallower levels i the
// row takes part in, and the leaf by the product of all its c_i.  A call's gradients depend on its output
// gradient only through P = exp(s - lse) times that gradient, so scaling the gradient by w equals handing the
// call lse - log(w): those are written to shifted[j] and leaf_shifted (w = 0 gives +inf: P = 0).
namespace {

constexpr int MERGE_MAX_LEVELS = 24;

struct MergeLevels {
  const void* o_un[MERGE_MAX_LEVELS];
  const float* lse_un[MERGE_MAX_LEVELS];
  float* shifted[MERGE_MAX_LEVELS];
  int levels;
};

constexpr int MERGE_THREADS = 256;

struct MergeLevelsParams {
  const void* o_leaf;
  const float* lse_leaf;
  void* out;
  float *lse_out, *leaf_shifted;
  MergeLevels lv;
  int64_t n, rows;  // rows of a sequence, of all of them
  uint32_t leaf_len, chunks, chunk_rows, pieces;
  uint32_t row_of_item;  // ceil(2^22 / pieces), 0 where a chunk is one row: item * that >> 22 is the item's row in its chunk
  int packed;
};

// A workgroup merges up to 256 * UNROLL pieces of 16 bytes of consecutive rows of one leaf (more where a row alone has more): which
// levels they take part in and where those results lie is the same for all, in scalar registers.  A row's chain of weights is
// one thread's, while the pieces' loads are in flight; its pieces' threads read the weights from LDS.
// HBM-bound.  With a thread's row, its halves and its weights found by each of its pieces' threads (lse_merge_rows_kernel: 64-bit divisions, every
// weight 8 to 16 times) it was bound by instructions: 24 x 131072 rows of 128 bytes, six levels, 443 -> 366 us (5.5 TB/s), 32 x 16384
// of 256 bytes, three levels, 94 -> 83, 48 x 10240 of 128, two levels, 40 -> 36, 8 x 65536, nine levels, 171 -> 118.
// GROUP: levels whose pieces are loaded at once, all of them unless MORE.
template <typename T, int GROUP, int UNROLL, bool MORE>
__global__ __launch_bounds__(MERGE_THREADS) void lse_merge_levels_kernel(const MergeLevelsParams p) {
  ha_load_arguments<(int)sizeof(MergeLevelsParams)>();
  typedef typename ElemTraits<T>::vec8 vec8;
  extern __shared__ float weight[];  // [level][row of the chunk]
  const MergeLevels& lv = p.lv;
  const uint32_t in_leaf = blockIdx.x / p.chunks, chunk = blockIdx.x - in_leaf * p.chunks;
  // leaf number of the rows inside their sequence: its bit (levels - 1 - j) says which half of its level-j
  // segment a row is in (such a half is 2^(levels - 1 - j) leaves long)
  const uint32_t leaf_no = in_leaf & ((1u << lv.levels) - 1), row_in_leaf = chunk * p.chunk_rows;
  const int64_t seq = in_leaf >> lv.levels, row_in_seq = (int64_t)leaf_no * p.leaf_len + row_in_leaf, row0 = seq * p.n + row_in_seq;
  const uint32_t rows = min(p.chunk_rows, p.leaf_len - row_in_leaf), items = rows * p.pieces;
  auto takes_part = [&](int j) -> bool { return j < lv.levels && ((leaf_no >> (lv.levels - 1 - j)) & 1u); };
  // Row of the level-j arrays that holds the first row's result.  Packed arrays keep only the rows a level writes,
  // the second halves of its segments of n >> j rows one after the other: (batch * heads, n / 2) rows.
  auto level_row = [&](int j) -> int64_t {
    const int64_t half = p.n >> (j + 1), segment = leaf_no >> (lv.levels - j);
    return p.packed ? seq * (p.n >> 1) + row_in_seq - (segment + 1) * half : row0;
  };
  const int64_t row_bytes = (int64_t)p.pieces * 16;
  const bool own_row = threadIdx.x < rows;
  const float x_leaf = own_row ? p.lse_leaf[row0 + threadIdx.x] : 0.f;
  float x = x_leaf, x_of[GROUP];
  for (uint32_t base = 0; base < items; base += MERGE_THREADS * UNROLL) {
    vec8 r[UNROLL], v[GROUP][UNROLL];
    uint32_t item[UNROLL], row[UNROLL];
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      item[u] = base + u * MERGE_THREADS + threadIdx.x;
      row[u] = min(item[u], items - 1) * p.row_of_item >> 22;
    }
    auto load = [&](vec8 (&to)[UNROLL], const void* from, int64_t first_row) {
      const char* const rows0 = (const char*)from + first_row * row_bytes;
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) to[u] = *reinterpret_cast<const vec8*>(rows0 + min(item[u], items - 1) * 16);
    };
    for (int first = MORE ? (lv.levels - 1) / GROUP * GROUP : 0; first >= 0; first -= GROUP) {  // deepest levels first
      // the log-sum-exps before the pieces, so that they are back before those are
      if (base == 0 && own_row) {
#pragma unroll
        for (int j = GROUP - 1; j >= 0; --j) {
          x_of[j] = 0.f;
          if (takes_part(first + j)) x_of[j] = lv.lse_un[first + j][level_row(first + j) + threadIdx.x];
        }
      }
      if (!MORE || first + GROUP >= lv.levels) load(r, p.o_leaf, row0);
#pragma unroll
      for (int j = GROUP - 1; j >= 0; --j)
        if (takes_part(first + j)) load(v[j], lv.o_un[first + j], level_row(first + j));
      if (base == 0) {
        if (own_row) {
          // each level's weight needs the log-sum-exp the deeper levels left
#pragma unroll
          for (int j = GROUP - 1; j >= 0; --j) {
            if (takes_part(first + j)) {
              const float c = (float)(T)(1.0f / (1.0f + __expf(x_of[j] - x)));
              weight[(first + j) * p.chunk_rows + threadIdx.x] = c;
              x = x - __logf(c + 1.1920929e-07f);
            }
          }
        }
        __syncthreads();
      }
#pragma unroll
      for (int j = GROUP - 1; j >= 0; --j) {
        if (takes_part(first + j)) {
#pragma unroll
          for (int u = 0; u < UNROLL; ++u) {
            const float c = weight[(first + j) * p.chunk_rows + row[u]];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              float sum = __builtin_fmaf(c, (float)r[u][e], (1.0f - c) * (float)v[j][u][e]);
              asm volatile("" : "+v"(sum));  // rounded to fp32 before T, as in the other merges
              r[u][e] = (T)sum;
            }
          }
        }
      }
    }
#pragma unroll
    for (int u = 0; u < UNROLL; ++u)
      if (item[u] < items) *reinterpret_cast<vec8*>((char*)p.out + row0 * row_bytes + item[u] * 16) = r[u];
  }
  if (!own_row) return;
  p.lse_out[row0 + threadIdx.x] = x;
  if (!p.leaf_shifted) return;
  float log_w = 0.f;  // log of the product of the weights c of the shallower levels
  auto shift = [&](int j, float x_un) {
    const float c = weight[j * p.chunk_rows + threadIdx.x];
    lv.shifted[j][level_row(j) + threadIdx.x] = x_un - log1pf(-c) - log_w;
    log_w += logf(c);
  };
  if constexpr (MORE) {
    for (int j = 0; j < lv.levels; ++j)
      if (takes_part(j)) shift(j, lv.lse_un[j][level_row(j) + threadIdx.x]);
  } else {
#pragma unroll
    for (int j = 0; j < GROUP; ++j)
      if (takes_part(j)) shift(j, x_of[j]);
  }
  p.leaf_shifted[row0 + threadIdx.x] = x_leaf - log_w;
}

// One piece of a row per thread, whatever leaf it lies in: for leaves that whole workgroups do not fit (merge_by_leaf).
// MAXL: levels the instance is unrolled for (the recursion rarely goes deeper than 8)
template <typename T, int MAXL>
__global__ __launch_bounds__(MERGE_THREADS) void lse_merge_rows_kernel(const MergeLevelsParams p) {
  ha_load_arguments<(int)sizeof(MergeLevelsParams)>();
  typedef typename ElemTraits<T>::vec8 vec8;
  const MergeLevels& lv = p.lv;
  const int64_t item = (int64_t)blockIdx.x * MERGE_THREADS + threadIdx.x;
  const int64_t row = item / p.pieces;
  if (row >= p.rows) return;
  const int64_t seq = row / p.n;
  const uint32_t row_in_seq = (uint32_t)(row - seq * p.n), leaf_no = row_in_seq / p.leaf_len;
  float x = p.lse_leaf[row];
  const float x_leaf = x;
  vec8 r = *reinterpret_cast<const vec8*>((const char*)p.o_leaf + item * 16);
  float c_of[MAXL], x_of[MAXL];
  vec8 v_of[MAXL];
  auto takes_part = [&](int j) -> bool { return j < lv.levels && ((leaf_no >> (lv.levels - 1 - j)) & 1u); };
  auto level_row = [&](int j) -> int64_t {
    const int64_t half = p.n >> (j + 1), segment = leaf_no >> (lv.levels - j);
    return p.packed ? seq * (p.n >> 1) + row_in_seq - (segment + 1) * half : row;
  };
  // every load first, so that they are all in flight before the chain of weights (each level's weight needs
  // the log-sum-exp the deeper levels left) starts
#pragma unroll
  for (int j = MAXL - 1; j >= 0; --j) {
    c_of[j] = 1.f;
    x_of[j] = 0.f;
    if (takes_part(j)) {
      const int64_t at = level_row(j);
      x_of[j] = lv.lse_un[j][at];
      v_of[j] = *reinterpret_cast<const vec8*>((const char*)lv.o_un[j] + (item + (at - row) * p.pieces) * 16);
    }
  }
#pragma unroll
  for (int j = MAXL - 1; j >= 0; --j) {
    if (takes_part(j)) {
      const float c = (float)(T)(1.0f / (1.0f + __expf(x_of[j] - x)));
#pragma unroll
      for (int e = 0; e < 8; ++e) r[e] = (T)(c * (float)r[e] + (1.0f - c) * (float)v_of[j][e]);
      x = x - __logf(c + 1.1920929e-07f);
      c_of[j] = c;
    }
  }
  *reinterpret_cast<vec8*>((char*)p.out + item * 16) = r;
  if (item != row * p.pieces) return;
  p.lse_out[row] = x;
  if (!p.leaf_shifted) return;
  float log_w = 0.f;
#pragma unroll
  for (int j = 0; j < MAXL; ++j) {
    if (takes_part(j)) {
      lv.shifted[j][level_row(j)] = x_of[j] - log1pf(-c_of[j]) - log_w;
      log_w += logf(c_of[j]);
    }
  }
  p.leaf_shifted[row] = x_leaf - log_w;
}

// Whether a workgroup's rows lie in one leaf.  `full`: the part of the workgroups' threads that have a piece; a leaf that a chunk's rows do
// not divide, and a short one above all, leaves some without, and chunks that do not start at multiples of 32 rows share lines of log-sum-exps.
// Rows | by leaf, us (1300 launches of leaves of 1 to 4096 rows, 2^13 to 2^21 in all; where the rule takes the leaves they are 0.82 to 2 times as fast,
// 1.23 at the median; of the others a few are up to 1.7 times as fast by leaf, 0.84 at the median): one level, 2^21 rows of d = 64: leaves of 1 row 139 | 3402, of 16 124 | 223, of 65 124 | 167, of 822 182 | 191,
// of 64 (full) 145 | 128; three levels, 2^17 rows: leaves of 34 18 | 19, of 75 18 | 14; 3 * 2^20 rows, which no cache holds, of 41, d = 128, 561 | 586, of 392 287 | 276; six: 2^17
// rows, leaves of 43 (0.67) 27.4 | 25.1, 3 * 2^20 of 135 (0.7) 463 | 473, of 230 (0.9) 464 | 454.
static bool merge_by_leaf(int levels, double full, double bytes) {
  if (levels < 2) return full == 1;
  return full >= (bytes > 256e6 ? 0.9 : levels == 2 ? 0.8 : 0.7);
}

}  // namespace

extern "C" int ha_lse_merge_levels(const void* o_leaf, const float* lse_leaf, const void* const* o_un,
                                   const float* const* lse_un, float* const* lse_shifted, float* leaf_shifted,
                                   void* out, float* lse_out, int levels, int64_t batch_heads, int64_t n, int64_t d,
                                   int dtype, int packed, void* stream) {
  HA_REQUIRE(o_leaf && lse_leaf && out && lse_out && (levels == 0 || (o_un && lse_un)), HA_ERR_NULL,
             "ha_lse_merge_levels: null pointer");
  HA_REQUIRE(dtype == HA_F16 || dtype == HA_BF16, HA_ERR_DTYPE, "ha_lse_merge_levels: Only support fp16 and bf16");
  HA_REQUIRE(levels >= 0 && levels <= MERGE_MAX_LEVELS, HA_ERR_UNSUPPORTED, "ha_lse_merge_levels: at most %d levels",
             MERGE_MAX_LEVELS);
  HA_REQUIRE(batch_heads > 0 && n > 0 && d > 0 && d % 8 == 0, HA_ERR_SHAPE,
             "ha_lse_merge_levels: sizes must be positive and d % 8 == 0");
  HA_REQUIRE((n >> levels) << levels == n, HA_ERR_SHAPE, "ha_lse_merge_levels: n must be divisible by 2^levels");
  HA_REQUIRE((leaf_shifted != nullptr) == (lse_shifted != nullptr) || levels == 0, HA_ERR_NULL,
             "ha_lse_merge_levels: leaf_shifted and lse_shifted go together");
  HA_REQUIRE(((uintptr_t)o_leaf % 16) == 0 && ((uintptr_t)out % 16) == 0, HA_ERR_SHAPE,
             "ha_lse_merge_levels: tensors must be 16-byte aligned");
  HA_REQUIRE(out != o_leaf && lse_out != lse_leaf, HA_ERR_UNSUPPORTED, "ha_lse_merge_levels: not in place");
  MergeLevels lv;
  lv.levels = levels;
  for (int j = 0; j < MERGE_MAX_LEVELS; ++j) {
    lv.o_un[j] = nullptr; lv.lse_un[j] = nullptr; lv.shifted[j] = nullptr;
  }
  for (int j = 0; j < levels; ++j) {
    HA_REQUIRE(o_un[j] && lse_un[j] && (!leaf_shifted || lse_shifted[j]), HA_ERR_NULL,
               "ha_lse_merge_levels: null pointer for level %d", j);
    HA_REQUIRE(((uintptr_t)o_un[j] % 16) == 0, HA_ERR_SHAPE, "ha_lse_merge_levels: tensors must be 16-byte aligned");
    lv.o_un[j] = o_un[j];
    lv.lse_un[j] = lse_un[j];
    lv.shifted[j] = leaf_shifted ? lse_shifted[j] : nullptr;
  }
  MergeLevelsParams p;
  p.o_leaf = o_leaf; p.lse_leaf = lse_leaf; p.out = out; p.lse_out = lse_out; p.leaf_shifted = leaf_shifted;
  p.lv = lv;
  p.n = n;
  p.rows = batch_heads * n;
  p.packed = packed;
  const int64_t leaf_len = n >> levels, pieces = d / 8, items = p.rows * pieces;
  HA_REQUIRE((items + 255) / 256 < (1ll << 31) && n < (1ll << 32), HA_ERR_SHAPE, "ha_lse_merge_levels: too many rows");
  // chunks of a leaf: as few as there can be, of equal lengths but for the last
  const int unroll = levels > 4 && levels <= 8 ? 2 : 1;
  const int64_t most = std::min<int64_t>(std::max<int64_t>(1, MERGE_THREADS * unroll / pieces), MERGE_THREADS), chunks = (leaf_len + most - 1) / most;
  p.leaf_len = (uint32_t)leaf_len;
  p.chunks = (uint32_t)chunks;
  p.chunk_rows = (uint32_t)((leaf_len + chunks - 1) / chunks);
  p.pieces = (uint32_t)pieces;
  p.row_of_item = p.chunk_rows == 1 ? 0 : (uint32_t)(((1 << 22) + pieces - 1) / pieces);
  const int64_t leaf_groups = (batch_heads << levels) * chunks, trip = MERGE_THREADS * unroll;
  const double full = (double)items / ((double)leaf_groups * ((p.chunk_rows * pieces + trip - 1) / trip * trip));
  const bool by_leaf = leaf_groups < (1ll << 24) &&  // a launch has less than 2^32 threads
                       merge_by_leaf(levels, full, (double)items * 16 * (2 + 0.5 * levels));
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)(by_leaf ? leaf_groups : (items + MERGE_THREADS - 1) / MERGE_THREADS)), dim3(MERGE_THREADS),
                       by_leaf ? levels * p.chunk_rows * 4 : 0, (hipStream_t)stream, p);
  };
  // Two pieces per thread from five levels on (24 x 131072 rows of 128 bytes, six levels, one | two 377 | 366 us, 8 x 65536 of 256, five,
  // 113 | 110), one below (32 x 16384 of 256, three, 83 | 88, 48 x 10240 of 128, two, 35.9 | 37.2)
  auto launch_for = [&](auto element) {
    typedef decltype(element) T;
    if (!by_leaf && levels <= 8) launch(lse_merge_rows_kernel<T, 8>);
    else if (!by_leaf) launch(lse_merge_rows_kernel<T, MERGE_MAX_LEVELS>);
    else if (levels <= 4) launch(lse_merge_levels_kernel<T, 4, 1, false>);
    else if (levels <= 8) launch(lse_merge_levels_kernel<T, 8, 2, false>);
    else launch(lse_merge_levels_kernel<T, 8, 1, true>);
  };
  if (dtype == HA_F16) launch_for(f16_t());
  else launch_for(bf16_t());
  return ha_launch_status("ha_lse_merge_levels");
}
