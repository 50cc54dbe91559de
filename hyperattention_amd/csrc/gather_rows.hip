// Permuting row gather: out[b,h,s,:] = x[b,h,idx[b,h,s],:], rows past n_idx zero-filled.
// Stands in for indexing() (src/attn_utils.py:27-50 of the reference).  One 16-byte piece per
// lane; the lanes of a row are adjacent so every gathered row is read and written as whole
// cache lines.
#include "ha_common.h"

#include <algorithm>

namespace {

__global__ __launch_bounds__(256) void gather_rows_kernel(const unsigned char* __restrict__ x,
                                                          const void* __restrict__ idx, int idx64,
                                                          unsigned char* __restrict__ out, int heads,
                                                          int64_t n_idx, int64_t n_out, int pieces,
                                                          int64_t sb_bytes, int64_t sh_bytes, int64_t sn_bytes) {
  const int bh = blockIdx.y;
  const int b = bh / heads, h = bh % heads;
  const int64_t item = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t row = item / pieces;
  const int piece = (int)(item % pieces);
  if (row >= n_out) return;
  u32x4 val = {0u, 0u, 0u, 0u};
  if (row < n_idx) {
    const int src = ha_load_idx(idx, (int64_t)bh * n_idx + row, idx64);
    val = *reinterpret_cast<const u32x4*>(x + b * sb_bytes + h * sh_bytes + (int64_t)src * sn_bytes + piece * 16);
  }
  *reinterpret_cast<u32x4*>(out + (((int64_t)bh * n_out + row) * pieces + piece) * 16) = val;
}

// Rows of several tensors into rows of another width (ha_copy_rows): padding with zero columns and its reverse.  HBM-bound: a
// thread moves ROW_COPY_PIECES pieces of 16 bytes, loads before stores; one launch for all tensors of a call.  q, k, v, dO of 32
// heads of 4352 rows, 96 -> 128 columns: 83 us as four fills and copies, 48 in one launch.
constexpr int ROW_COPY_PIECES = 4;
struct RowCopies {
  const unsigned char* src[HA_ROW_COPIES];
  unsigned char* dst[HA_ROW_COPIES];
  int64_t src_sb[HA_ROW_COPIES], src_sh[HA_ROW_COPIES], src_sn[HA_ROW_COPIES];  // bytes
  int64_t dst_sb[HA_ROW_COPIES], dst_sh[HA_ROW_COPIES], dst_sn[HA_ROW_COPIES];
  int heads[HA_ROW_COPIES], seqs[HA_ROW_COPIES], rows[HA_ROW_COPIES];
  int src_pieces[HA_ROW_COPIES], dst_pieces[HA_ROW_COPIES];
};
__global__ __launch_bounds__(256) void copy_rows_kernel(const RowCopies c) {
  ha_load_arguments<(int)sizeof(RowCopies)>();
  const int job = blockIdx.z;
  const uint32_t pieces = c.dst_pieces[job], have = c.src_pieces[job];
  const uint32_t first = blockIdx.x * (256 * ROW_COPY_PIECES) + threadIdx.x, end = (uint32_t)c.rows[job] * pieces;
  for (int seq = blockIdx.y; seq < c.seqs[job]; seq += gridDim.y) {
    const int b = seq / c.heads[job], h = seq % c.heads[job];
    const unsigned char* const src = c.src[job] + b * c.src_sb[job] + h * c.src_sh[job];
    unsigned char* const dst = c.dst[job] + b * c.dst_sb[job] + h * c.dst_sh[job];
    u32x4 v[ROW_COPY_PIECES];
#pragma unroll
    for (int i = 0; i < ROW_COPY_PIECES; ++i) {
      const uint32_t item = min(first + 256 * i, end - 1), row = item / pieces, piece = item - row * pieces;
      v[i] = *reinterpret_cast<const u32x4*>(src + (int64_t)row * c.src_sn[job] + min(piece, have - 1) * 16);
      if (piece >= have) v[i] = u32x4{0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int i = 0; i < ROW_COPY_PIECES; ++i) {
      const uint32_t item = first + 256 * i;
      if (item >= end) continue;
      const uint32_t row = item / pieces, piece = item - row * pieces;
      *reinterpret_cast<u32x4*>(dst + (int64_t)row * c.dst_sn[job] + piece * 16) = v[i];
    }
  }
}

}  // namespace

extern "C" int ha_copy_rows(const ha_row_copy* copies, int count, void* stream) {
  HA_REQUIRE(copies, HA_ERR_NULL, "ha_copy_rows: null pointer");
  HA_REQUIRE(count >= 1 && count <= HA_ROW_COPIES, HA_ERR_SHAPE, "ha_copy_rows: 1 to %d tensors", HA_ROW_COPIES);
  RowCopies c = {};
  int64_t most_items = 0, most_seqs = 0;
  for (int i = 0; i < count; ++i) {
    const ha_row_copy& r = copies[i];
    HA_REQUIRE(r.src && r.dst, HA_ERR_NULL, "ha_copy_rows: null pointer");
    HA_REQUIRE(r.batch > 0 && r.heads > 0 && r.n > 0 && r.src_d > 0 && r.dst_d > 0, HA_ERR_SHAPE, "ha_copy_rows: sizes must be positive");
    HA_REQUIRE(r.src_d % 8 == 0 && r.dst_d % 8 == 0, HA_ERR_HEADDIM, "ha_copy_rows: row lengths must be multiples of 8");
    HA_REQUIRE(r.batch * r.heads < (1ll << 31) && r.n * (r.dst_d / 8) < (1ll << 31), HA_ERR_SHAPE, "ha_copy_rows: tensor too large");
    const int64_t strides[] = {r.src_stride_b, r.src_stride_h, r.src_stride_n, r.dst_stride_b, r.dst_stride_h, r.dst_stride_n};
    for (int64_t s : strides) HA_REQUIRE(s % 8 == 0, HA_ERR_SHAPE, "ha_copy_rows: rows must be 16-byte aligned");
    HA_REQUIRE(((uintptr_t)r.src % 16) == 0 && ((uintptr_t)r.dst % 16) == 0, HA_ERR_SHAPE, "ha_copy_rows: rows must be 16-byte aligned");
    c.src[i] = (const unsigned char*)r.src; c.dst[i] = (unsigned char*)r.dst;
    c.src_sb[i] = r.src_stride_b * 2; c.src_sh[i] = r.src_stride_h * 2; c.src_sn[i] = r.src_stride_n * 2;
    c.dst_sb[i] = r.dst_stride_b * 2; c.dst_sh[i] = r.dst_stride_h * 2; c.dst_sn[i] = r.dst_stride_n * 2;
    c.heads[i] = (int)r.heads; c.seqs[i] = (int)(r.batch * r.heads); c.rows[i] = (int)r.n;
    c.src_pieces[i] = (int)(r.src_d / 8); c.dst_pieces[i] = (int)(r.dst_d / 8);
    most_items = std::max<int64_t>(most_items, r.n * (r.dst_d / 8));
    most_seqs = std::max<int64_t>(most_seqs, r.batch * r.heads);
  }
  constexpr int PER_BLOCK = 256 * ROW_COPY_PIECES;
  dim3 grid((unsigned)((most_items + PER_BLOCK - 1) / PER_BLOCK), (unsigned)std::min<int64_t>(most_seqs, 65535), (unsigned)count);
  hipLaunchKernelGGL(copy_rows_kernel, grid, dim3(256), 0, (hipStream_t)stream, c);
  return ha_launch_status("ha_copy_rows");
}

extern "C" int ha_gather_rows(const void* x, const void* idx, int idx_type, void* out, int64_t batch,
                              int64_t heads, int64_t n_src, int64_t n_idx, int64_t n_out, int64_t d,
                              int64_t x_stride_b, int64_t x_stride_h, int64_t x_stride_n, int elem_bytes,
                              void* stream) {
  HA_REQUIRE(x && idx && out, HA_ERR_NULL, "ha_gather_rows: null pointer");
  HA_REQUIRE(idx_type == HA_IDX_I32 || idx_type == HA_IDX_I64, HA_ERR_DTYPE, "ha_gather_rows: bad idx_type");
  HA_REQUIRE(elem_bytes == 2 || elem_bytes == 4, HA_ERR_DTYPE, "ha_gather_rows: elem_bytes must be 2 or 4");
  HA_REQUIRE(batch > 0 && heads > 0 && n_src > 0 && n_idx >= 0 && n_out >= n_idx && n_out > 0 && d > 0,
             HA_ERR_SHAPE, "ha_gather_rows: bad sizes");
  HA_REQUIRE(batch * heads <= 65535, HA_ERR_SHAPE, "ha_gather_rows: batch*heads must be <= 65535");
  HA_REQUIRE((d * elem_bytes) % 16 == 0, HA_ERR_HEADDIM, "ha_gather_rows: row bytes must be a multiple of 16");
  HA_REQUIRE((x_stride_n * elem_bytes) % 16 == 0 && (x_stride_h * elem_bytes) % 16 == 0 &&
                 (x_stride_b * elem_bytes) % 16 == 0 && ((uintptr_t)x % 16) == 0 && ((uintptr_t)out % 16) == 0,
             HA_ERR_SHAPE, "ha_gather_rows: rows must be 16-byte aligned");
  const int pieces = (int)(d * elem_bytes / 16);
  const int64_t items = n_out * pieces;
  dim3 grid((unsigned)((items + 255) / 256), (unsigned)(batch * heads));
  hipLaunchKernelGGL(gather_rows_kernel, grid, dim3(256), 0, (hipStream_t)stream, (const unsigned char*)x, idx,
                     idx_type == HA_IDX_I64, (unsigned char*)out, (int)heads, n_idx, n_out, pieces,
                     x_stride_b * elem_bytes, x_stride_h * elem_bytes, x_stride_n * elem_bytes);
  return ha_launch_status("ha_gather_rows");
}
