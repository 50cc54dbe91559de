// Device-side parameter block of the attention kernels (validated and filled by the C entry points).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "bucket_sort.h"

// x / y for 0 <= x < 2^31 as (x * magic) >> shift, with shift = 31 + ceil(log2 y) and
// magic = floor(2^shift / y) + 1 < 2^32 (exact for every such x)
struct ha_divisor {
  uint32_t magic;
  int shift;
};

constexpr int HA_MAX_RAGGED_LEVELS = 30;

// Workgroups of an exact causal launch that hash and rank units of the same tensors' rows for the hashed levels that follow
// (unit_ranking.h).  They come in groups of eight, one per XCD, so that the others keep the XCD that their number gives them.
struct ha_rank_beside {
  const void* proj;       // (d, num_projs), num_projs <= 8
  uint32_t* sorted[2];    // of q's and k's units: as ha_rank_units
  uint32_t* hist[2];
  int32_t* out[2];
  int64_t n_read;         // rows of a sequence that exist; the others are zero rows
  int num_projs;
  int first_unit[2];
  int num_units;          // of a sequence
  int units0;             // of q
  int units;              // of q and k
  ha_unit_grid grid;
  int tiles;              // workgroups of the attention (filled by ha_attn_launch)
  int first_group, groups;  // groups of eight workgroups before the first ranking one, and of ranking ones (as well)
};

struct ha_attn_kernel_params {
  const void* q;
  const void* k;
  const void* v;
  void* out;
  float* lse;
  const void* q_idx;        // gather mode only
  const void* k_idx;
  const void* sampled_idx;  // may be null: rows 0..sample-1
  int64_t q_sb, q_sh, q_sn;
  int64_t k_sb, k_sh, k_sn;
  int64_t v_sb, v_sh, v_sn;
  int64_t o_sb, o_sh, o_sn;
  int64_t lse_sb, lse_sh;
  int64_t qi_sb, qi_sh, qi_sn;
  int64_t ki_sb, ki_sh, ki_sn;
  int64_t si_sb, si_sh;
  int64_t seg_stride, q_seg_off, k_seg_off;
  int batch, heads, segs, kv_group;
  int n_q, n_k;
  int block_tiles;    // ceil(block_size / 128)
  int sample_chunks;  // sample_size / 64
  int smooth, accumulate, idx64;
  int qk_pieces, v_pieces;  // 16-byte pieces in a row of q/k and of v/out (filled by ha_attn_launch)
  // residual estimator (gathered kernel, REWEIGHT instances only)
  const int32_t* sampled_pos;  // sorted-order position of every sampled key; null: nothing is masked
  float sample_bias_raw;       // added to the raw q.k of a sampled key: bias / softmax scale
  float scale_log2;   // softmax scale * log2(e)
  // Queries of the last segment of every head that exist (gathered kernel): an entry of its query order at or
  // past this number names a row that is not there (the zero row the causal recursion appends to an odd
  // length, hyper_attention.py:61-64); it is placed like any other row and its result is dropped.
  int n_q_last;
  int lse_rows;  // exact kernels: lse rows n_q .. lse_rows - 1 are written as zeros (0: none)
  // first row of segment g in the out / lse tensors: o_seg_off + g * o_seg_stride (= the query side's unless
  // the caller packs the rows a call writes)
  int64_t o_seg_off, o_seg_stride;
  int single;      // exact causal kernel: one tile per workgroup, longest first, instead of pairs (filled by ha_attn_launch)
  int split_keys;  // the keys of a query tile are split over the waves of a workgroup, 2: longest tiles first (filled by
                   // ha_attn_launch)
  int small_tiles;  // head dims up to 64: tiles of 128 queries (filled by ha_attn_launch)
  int large_tiles;  // head dims above 64: exact attention in tiles of 256 queries (filled by ha_attn_launch)
  int follow_max;  // the FOLLOW instances; gathered, and exact without mask at head dims above 64: in that many chunks of a row
                   // (filled by ha_attn_launch)
  // Ragged segments (exact kernels; rag_levels < 0: regular).  Inside a causal recursion with odd lengths the
  // segments of a level neither start at multiples of one stride nor hold the same number of rows: level i
  // cuts a segment of (padded) length 2*rag_half[i] into two, and the rows that exist are the first rag_n of
  // the whole sequence.  Segment number `seg` has rag_levels bits, most significant first: bit i says which
  // half of its level-i ancestor it lies in.
  int rag_levels, rag_n;
  int rag_half[HA_MAX_RAGGED_LEVELS];
  // the divisors of the workgroup -> (head, segment, tile) decomposition as multiply-and-shift
  // constants (filled by ha_attn_launch): the kernel never divides
  ha_divisor div_qtiles, div_segs, div_heads, div_kv_heads, div_kv_group, div_block_tiles;
};

// ranking: exact causal launches, or null
int ha_attn_launch(const ha_attn_kernel_params& p, int d, int dv, int dtype, bool gather, bool causal, bool reweight,
                   hipStream_t stream, const ha_rank_beside* ranking = nullptr);

// argument checks shared by the forward and backward entry points (defined in api.hip); `who` names
// the entry point in the error message
int ha_check_operands(const ha_attn_operands& t, const char* who);
int ha_check_block_attn_args(const ha_block_attn_args& a, const char* who);
