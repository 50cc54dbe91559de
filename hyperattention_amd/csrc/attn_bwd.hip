// MFMA attention backward kernels for gfx950: gradients of the sorted block-diagonal + sampled-column
// attention and of exact (flash) attention with respect to q, k and v.
//
// Reference semantics: _hyper_attn_backward with _bwd_preprocess_do_o_dot,
// _bwd_permuted_block_diagonal_kernel and _bwd_sampled_col_kernel (src/hyper_attn_triton.py:195-665,
// :745-893) and _flash_attn_backward (src/flash_attn_triton.py:270-792, :875-992): given dO, the
// forward's O and its log-sum-exp L (a gradient arriving for L itself is ignored, as in
// HyperAttnFunc.backward, src/hyper_attn_triton.py:922-945),
//   D_i  = sum_c dO_ic O_ic,            P_ij = exp(scale q_i.k_j - L_i),
//   dV_j = sum_i P_ij dO_i,             dS_ij = P_ij (dO_i.v_j - D_i) scale,
//   dQ_i = sum_j dS_ij k_j,             dK_j = sum_i dS_ij q_i,
// over exactly the (query, key) pairs the forward visits: a key that is both in a query's block and in
// the sample list counts twice.  P and dS are rounded to the input type before the products, as the
// reference does.
//
// One kernel body serves five passes.  A workgroup of 4 waves keeps 128 "stationary" rows (32 per wave, as B operands in
// registers; 64 rows where the steps are split over waves) and streams the rows of the other side through LDS, in tiles
// of 64 rows at d = 64 and of 32 at d = 128 (64 where the steps are split):
//   dQ passes    stationary = queries (Q, dO), streamed = keys (K, V):      dQ^T += K^T dS^T
//   dK/dV passes stationary = keys (K, V),     streamed = queries (Q, dO):  dK^T += Q^T dS, dV^T += dO^T P
// Both compute S' = Y1 X1^T and dP' = Y2 X2^T (streamed rows as MFMA rows, stationary rows as MFMA
// columns), so a lane holds 16 streamed rows of ONE stationary row and P', dS' are the B operands of
// the products that follow, whose A operands (Y^T) come from the transposing LDS reads.  The dQ passes
// see all keys of a query in one workgroup and store dQ.  The dK/dV pass of exact attention sees all
// queries of a key (of every query head of the key head's group, streamed one head after the other)
// and stores dK, dV.  With sorted blocks a key gets one contribution from its block (complete in one
// workgroup: stored like the exact pass's) and, if it is in the sample list, one from every query:
// those are computed per range of queries and summed in small fp32 rows, one per slot of
// the sample list (with atomics, or one share per range, see writes_shares), which a last kernel adds to the keys' rows of
// dK, dV.
// The forms of the exact passes: exact_form.  Plain blocks of 256 at head dim 64 take
// the one kernel of attn_bwd_block.hip in the place of the three gathered passes.
#include "ha_common.h"
#include "attn_tiles.h"
#include "attn_fwd.h"
#include "attn_bwd.h"
#include "attn_bwd_tiles.h"

#include <algorithm>
#include <type_traits>

namespace {

constexpr int WG_THREADS = 256;
constexpr int ST_ROWS = 128;       // stationary rows per workgroup
constexpr int MAX_SMOOTH_TILES = 1024;  // query tiles that can attend one 128-key tile (smoothed blocks)

// Scheduling groups: M times one MFMA followed by its share of V plain vector instructions and E transcendentals, and,
// from MFMA number 1 on, PER at a time of R LDS reads.  (Reads ahead of the first MFMA would be waited for by it: the
// wait counter holds 15, and more younger reads than that cannot be told from the operands.)
template <int M, int V, int E, int R, int PER, int I = 0>
__device__ __forceinline__ void interleave_groups() {
  if constexpr (I < M) {
    constexpr int v = V * (I + 1) / M - V * I / M, e = E * (I + 1) / M - E * I / M;
    constexpr int done = I > 0 ? (I - 1) * PER : 0, reads = I == 0 ? 0 : (R - done < PER ? R - done : PER);
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    if constexpr (reads > 0) __builtin_amdgcn_sched_group_barrier(0x100, reads, 0);
    if constexpr (v > 0) __builtin_amdgcn_sched_group_barrier(0x002, v, 0);
    if constexpr (e > 0) __builtin_amdgcn_sched_group_barrier(0x400, e, 0);
    interleave_groups<M, V, E, R, PER, I + 1>();
  }
}

// sum over the 16 lanes of a row of lanes
__device__ __forceinline__ float row16_sum(float v) {
  v += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x128, 0xf, 0xf, true));  // row_ror:8
  v += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x124, 0xf, 0xf, true));
  v += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x122, 0xf, 0xf, true));
  return v + __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x121, 0xf, 0xf, true));
}

template <typename T, int D, int PASS, bool CAUSAL, int HALVES>
__global__ __launch_bounds__(WG_THREADS, (D <= 64 || PASS == HA_BWD_DQ_BLOCK || (PASS == HA_BWD_DQ_EXACT && HALVES == 1) ? 2 : 1)) void ha_attn_bwd_kernel(const ha_attn_bwd_params p) {
  ha_load_arguments<(int)sizeof(ha_attn_bwd_params)>();
  typedef typename ElemTraits<T>::vec8 vec8;
  typedef typename ElemTraits<T>::vec4 vec4;
  constexpr bool KEY_ST = PASS == HA_BWD_DKV_EXACT || PASS == HA_BWD_DKV_BLOCK || PASS == HA_BWD_DKV_SAMPLED;
  constexpr int KSTEPS = D / 16;  // MFMA k-steps over the head dim
  constexpr int DB = D / 32;      // 32-row blocks of the transposed gradients
  constexpr int PR = D / 8;       // 16-byte pieces per row
  constexpr int RPL = 64 / PR;    // rows per tile load (one load = 64 lanes x 16 bytes)
  // Streamed rows per LDS tile and tiles in the ring: a step of 32 rows reads its own tile and the next step's, and
  // the tile after that is in flight; two steps per tile at d = 64, one at d = 128 (the same bytes).
  // HALVES == 2 (SPLIT): 64 stationary rows per workgroup; of the two steps of a tile waves 0, 1 take the first
  // and waves 2, 3 the second, and the two sums of a row meet in LDS at the end.
  constexpr int YC = D <= 64 || HALVES == 2 ? 64 : 32;
  constexpr int STEPS = YC / 32 / HALVES;  // steps that a wave takes from a tile
  constexpr int NBUF = STEPS == 2 ? 3 : 4;
  static_assert(HALVES == 1 || PASS == HA_BWD_DQ_EXACT || PASS == HA_BWD_DKV_EXACT, "built for the exact passes");
  constexpr int ST = ST_ROWS / HALVES;
  constexpr int CPT = 128 / YC;            // chunks per tile of 128 of the sorted order
  constexpr int LPW = YC * PR / 64 / 4;    // tile loads per wave per tile
  constexpr int TILE_BYTES = YC * D * 2;

  // The streamed tiles are separate LDS objects, named statically by the loop (unrolled over the ring of NBUF): the
  // compiler then knows that the tile being filled from memory is not one being read.  As one array with the
  // buffer's number as an index, every first read of a tile waited for the loads of the NEXT one, just issued.
  __shared__ __attribute__((aligned(1024))) unsigned char y1_0[TILE_BYTES], y1_1[TILE_BYTES], y1_2[TILE_BYTES];
  __shared__ __attribute__((aligned(1024))) unsigned char y2_0[TILE_BYTES], y2_1[TILE_BYTES], y2_2[TILE_BYTES];
  __shared__ __attribute__((aligned(1024))) unsigned char y1_3[NBUF > 3 ? TILE_BYTES : 16], y2_3[NBUF > 3 ? TILE_BYTES : 16];
  auto y1_tile = [&](int i) -> unsigned char* { return i == 0 ? y1_0 : i == 1 ? y1_1 : i == 2 ? y1_2 : y1_3; };
  auto y2_tile = [&](int i) -> unsigned char* { return i == 0 ? y2_0 : i == 1 ? y2_1 : i == 2 ? y2_2 : y2_3; };
  // dK/dV passes: -L / (scale log2 e) and -D of the streamed queries
  constexpr int SN = KEY_ST ? YC : 4;
  __shared__ __attribute__((aligned(16))) float lse_0[SN], lse_1[SN], lse_2[SN], lse_3[SN];
  __shared__ __attribute__((aligned(16))) float delta_0[SN], delta_1[SN], delta_2[SN], delta_3[SN];
  auto lse_tile = [&](int i) -> float* { return i == 0 ? lse_0 : i == 1 ? lse_1 : i == 2 ? lse_2 : lse_3; };
  auto delta_tile = [&](int i) -> float* { return i == 0 ? delta_0 : i == 1 ? delta_1 : i == 2 ? delta_2 : delta_3; };
  constexpr bool STAGE_X = KEY_ST || D <= 64, STAGE_TURNS = !STAGE_X && HALVES == 1;
  // staging of the second stationary operand (prologue); with four tiles of 64 rows in the ring there is room in them
  __shared__ __attribute__((aligned(1024))) unsigned char lds_x2[STAGE_X && HALVES == 1 ? ST_ROWS * D * 2 : 16];
  __shared__ int lds_tiles[PASS == HA_BWD_DKV_BLOCK ? MAX_SMOOTH_TILES : 1];
  __shared__ int lds_ntiles;

  const int tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63;
  const int wave_s = __builtin_amdgcn_readfirstlane(wave);
  const int hi = lane >> 5, col = lane & 31;
  const int half = HALVES == 2 ? wave_s >> 1 : 0;       // the step of a tile that the wave takes
  const int st_wave = HALVES == 2 ? wave_s & 1 : wave_s;  // its 32 stationary rows of the tile

  // ---- which head, which stationary tile ------------------------------------------------------
  const int st_total = PASS == HA_BWD_DKV_SAMPLED ? p.sample_size : (KEY_ST ? p.n_k : p.n_q);
  const int st_tiles = (st_total + ST - 1) / ST;
  const int splits = PASS == HA_BWD_DKV_SAMPLED ? (p.n_q + p.q_split - 1) / p.q_split : 1;
  // Exact causal attention: a workgroup takes the pair of stationary tiles (s, T-1-s), the one that streams more
  // rows first (the last query tile sees every key, the first key tile is seen by every query), so that every
  // workgroup of a launch streams the same number of rows.  The hardware hands out workgroups in order, and a
  // slot freed by a short one stays empty until the ones queued before it are placed.  Few tiles (single_tiles) come one by
  // one, the ones of all sequences that stream the most rows first, at d = 64, two workgroups per CU, the second 256 reversed.
  constexpr bool PAIRED = CAUSAL && HALVES == 1 && (PASS == HA_BWD_DQ_EXACT || PASS == HA_BWD_DKV_EXACT);
  // (dq at d = 128 gets no pairs: so many tiles go to the wide pass.  Compiled without the pair's second copy of the tile its
  // loop spills: 24 heads of 2048 rows 67 -> 75 us.)
  const bool single = PAIRED && p.single_tiles;
  const int wg_per_seq = PAIRED && !single ? (st_tiles + 1) / 2 : st_tiles;
  // Steps split over waves: no pairs; the tiles of all sequences that stream the most rows come first (tile-major)
  const bool tile_major = HALVES == 2 || single;
  const int n_vseq = tile_major ? gridDim.x / wg_per_seq : 1;
  int rest = tile_major ? (int)blockIdx.x : xcd_contiguous_id(blockIdx.x, gridDim.x);
  if (single && D <= 64) {
    const int second = min((int)gridDim.x, 512);
    if (rest >= 256 && rest < second) rest = 256 + second - 1 - rest;
  }
  const int slot = tile_major ? rest / n_vseq : rest % wg_per_seq;
  rest = tile_major ? rest - slot * n_vseq : rest / wg_per_seq;
  const int split = rest % splits;
  const int vseq = rest / splits;   // (batch, head, segment)
  const int seg = vseq % p.segs;
  const int bh = vseq / p.segs;
  // The dK/dV passes that see every query of a key (exact attention, the blocks) take one workgroup per
  // KEY head and stream the queries of all the query heads of its group, one head after the other, so
  // that the sums are complete in registers; the other passes take one workgroup per query head.
  constexpr bool GROUP_LOOP = PASS == HA_BWD_DKV_EXACT || PASS == HA_BWD_DKV_BLOCK;
  const int kv_heads = p.heads / p.kv_group;
  int b, h0, hk;
  if (GROUP_LOOP) {
    b = bh / kv_heads;
    hk = bh - b * kv_heads;
    h0 = hk * p.kv_group;
  } else {
    b = bh / p.heads;
    h0 = bh - b * p.heads;
    hk = h0 / p.kv_group;
  }
  const int n_group = GROUP_LOOP ? p.kv_group : 1;
  // first row of this segment in the query-side and in the key-side tensors
  const int64_t q_row0 = p.q_seg_off + (int64_t)seg * p.seg_stride;
  const int64_t k_row0 = p.k_seg_off + (int64_t)seg * p.seg_stride;
  const int64_t o_row0 = p.o_seg_off + (int64_t)seg * p.o_seg_stride;  // in the forward's out and lse

  // query-side tensors of query head h0 + gi
  auto q_head = [&](int gi) { return (const unsigned char*)((const T*)p.q + b * p.q_sb + (h0 + gi) * p.q_sh + q_row0 * p.q_sn); };
  auto do_head = [&](int gi) { return (const unsigned char*)((const T*)p.dout + b * p.do_sb + (h0 + gi) * p.do_sh + q_row0 * p.do_sn); };
  // per query: {L in log2 units, -D} with D_i = sum_c dO_ic O_ic (src/hyper_attn_triton.py:195-226),
  // written by the dq pass of the call
  auto stats_head = [&](int gi) { return p.stats + ((int64_t)(b * p.heads + h0 + gi) * p.segs + seg) * p.n_q; };
  const int idx_shift = p.idx64 ? 3 : 2;
  auto q_idx_head = [&](int gi) {
    return (const unsigned char*)p.q_idx + ((b * p.qi_sb + (h0 + gi) * p.qi_sh + (int64_t)seg * p.n_q * p.qi_sn) << idx_shift);
  };
  const unsigned char* const kb = (const unsigned char*)((const T*)p.k + b * p.k_sb + hk * p.k_sh + k_row0 * p.k_sn);
  const unsigned char* const vb = (const unsigned char*)((const T*)p.v + b * p.v_sb + hk * p.v_sh + k_row0 * p.v_sn);
  const uint32_t q_rb = (uint32_t)p.q_sn * 2, k_rb = (uint32_t)p.k_sn * 2, v_rb = (uint32_t)p.v_sn * 2,
                 do_rb = (uint32_t)p.do_sn * 2;
  const unsigned char* const k_idx = (const unsigned char*)p.k_idx + ((b * p.ki_sb + hk * p.ki_sh + (int64_t)seg * p.n_k * p.ki_sn) << idx_shift);
  const unsigned char* const s_idx =
      p.sampled_idx ? (const unsigned char*)p.sampled_idx + ((b * p.si_sb + hk * p.si_sh) << idx_shift) : nullptr;
  const uint32_t qi_rb = (uint32_t)p.qi_sn << idx_shift, ki_rb = (uint32_t)p.ki_sn << idx_shift;
  const uint32_t si_rb = 1u << idx_shift;

  // stationary (X) and streamed (Y) operands of this pass
  const unsigned char* const x1b = KEY_ST ? kb : q_head(0);
  const unsigned char* const x2b = KEY_ST ? vb : do_head(0);
  const uint32_t x1_rb = KEY_ST ? k_rb : q_rb, x2_rb = KEY_ST ? v_rb : do_rb;
  const uint32_t y1_rb = KEY_ST ? q_rb : k_rb, y2_rb = KEY_ST ? do_rb : v_rb;
  const int n_y = KEY_ST ? p.n_q : p.n_k;  // rows on the streamed side

  if constexpr (!PAIRED) {
    const int tile = HALVES == 2 && CAUSAL && PASS == HA_BWD_DQ_EXACT ? st_tiles - 1 - slot : slot;
#include "attn_bwd_tile.inc"
  } else {
    const int t_long = PASS == HA_BWD_DQ_EXACT ? st_tiles - 1 - slot : slot;
    const int t_short = st_tiles - 1 - t_long;
    {
      const int tile = t_long;
#include "attn_bwd_tile.inc"
    }
    if (!single && t_short != t_long) {  // an odd number of tiles: the middle one has no partner
      // the first tile's last reads of the staging areas and the streamed tiles are behind every wave
      __syncthreads();
      const int tile = t_short;
#include "attn_bwd_tile.inc"
    }
  }
}

__global__ __launch_bounds__(256) void ha_bwd_zero_kernel(f32x4* __restrict__ buf, int64_t n4) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n4) buf[i] = f32x4{0.f, 0.f, 0.f, 0.f};
}

struct AddSamplesParams {
  const float* sums[2];  // of dk (times k_factor) and dv: `shares` of them, rows by slot of the sample list or (FUSED) as ha_fused_share_at has them
  void* grad[2];         // dk, dv
  int64_t sb[2], sh[2], sn[2];
  const void* sampled_idx;
  int64_t si_sb, si_sh, seg_stride, k_seg_off;
  int idx64, kv_heads, sample_size, shares, segs;
  float k_factor;
};

// Sums of the sampled keys added to the rows of dk (blockIdx.y = 0) or dv.  A workgroup has 2048 elements of one (batch, kv head,
// segment), 8 per thread, so that rows are read and written whole; FUSED sums, which lie as the products leave them, are
// turned around in LDS.  A row that is listed several times is handled by its first slot alone, which adds the sums of all of
// them: no two lanes write the same row, whatever the list holds.
// HBM-bound.  With 4 elements per thread, FUSED rows written 8 bytes at a time and three 64-bit divisions a thread it took 56.7 us and takes 30.9
// for 768 segments of one share at d = 64 (6.5 TB/s), for 24 of 32 shares 21.0 | 20.9, 48 of 10 and 96 of 5 11.0 | 8.4, 16.6 | 14.2; d = 128,
// 8 segments of 16 shares 16.5 | 12.6.
template <typename T, int D, bool FUSED>
__global__ __launch_bounds__(256) void ha_bwd_add_samples_kernel(const AddSamplesParams p) {
  ha_load_arguments<(int)sizeof(AddSamplesParams)>();
  typedef typename ElemTraits<T>::vec8 vec8;
  constexpr int PR = D / 8, ROWS = 256 / PR;
  static_assert(!FUSED || ROWS == 32, "FUSED sums come in groups of 32 keys");
  const int tiles = p.sample_size / ROWS, bhs = blockIdx.x / tiles, slot0 = (blockIdx.x - bhs * tiles) * ROWS;
  const int bh = bhs / p.segs, seg = bhs - bh * p.segs, b = bh / p.kv_heads, h = bh - b * p.kv_heads, is_v = blockIdx.y;
  const int tid = threadIdx.x, r = tid / PR, piece = tid % PR, slot = slot0 + r;
  const int64_t share = (int64_t)p.sample_size * D;
  const float* const base = p.sums[is_v] + (int64_t)bhs * p.shares * share;
  T* const rows = (T*)p.grad[is_v] + b * p.sb[is_v] + h * p.sh[is_v] + (p.k_seg_off + (int64_t)seg * p.seg_stride) * p.sn[is_v] + piece * 8;
  const int64_t list = b * p.si_sb + h * p.si_sh;
  int row = slot;
  bool owner = true;  // no earlier slot has the row
  if (p.sampled_idx) {
    row = ha_load_idx(p.sampled_idx, list + slot, p.idx64);
    for (int s2 = 0; s2 < slot && owner; ++s2) owner = ha_load_idx(p.sampled_idx, list + s2, p.idx64) != row;
  }
  vec8* const dst = reinterpret_cast<vec8*>(rows + row * p.sn[is_v]);
  vec8 o = *dst;
  f32x4 sum[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
  auto add_shares = [&](const float* at0, const float* at1) {
#pragma unroll 8
    for (int k = 0; k < p.shares; ++k) {
      sum[0] += *reinterpret_cast<const f32x4*>(at0 + k * share);
      sum[1] += *reinterpret_cast<const f32x4*>(at1 + k * share);
    }
  };
  auto at = [&](int s2, int half) -> const float* {
    return base + (FUSED ? ha_fused_share_at(s2, 2 * piece + half) : s2 * D + piece * 8 + half * 4);
  };
  if constexpr (FUSED) {
    __shared__ f32x4 turn[512];  // [key][four elements]
    const float* const mine = base + (slot0 >> 5) * 2048 + tid * 4;
    add_shares(mine, mine + 1024);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int key = tid & 31, four = i * 8 + tid / 32;
      turn[key * 16 + (four ^ (key & 15))] = sum[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; ++i) sum[i] = turn[r * 16 + ((2 * piece + i) ^ (r & 15))];
  } else {
    add_shares(at(slot, 0), at(slot, 1));
  }
  if (!owner) return;
  if (p.sampled_idx)
    for (int s2 = slot + 1; s2 < p.sample_size; ++s2)
      if (ha_load_idx(p.sampled_idx, list + s2, p.idx64) == row) add_shares(at(s2, 0), at(s2, 1));
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] = (T)((float)o[e] + (FUSED && !is_v ? sum[e >> 2][e & 3] * p.k_factor : sum[e >> 2][e & 3]));
  *dst = o;
}

template <typename T, int D, int PASS, bool CAUSAL, int HALVES = 1>
int launch_pass(const ha_attn_bwd_params& p, int64_t grid, hipStream_t stream, const char* what) {
  if (grid <= 0) return HA_OK;
  if (grid >= (1ll << 31)) return ha_fail(HA_ERR_SHAPE, "%s: grid of %lld workgroups", what, (long long)grid);
  hipLaunchKernelGGL((ha_attn_bwd_kernel<T, D, PASS, CAUSAL, HALVES>), dim3((unsigned)grid), dim3(WG_THREADS), 0, stream, p);
  return ha_launch_status(what);
}

inline int64_t align256(int64_t v) { return (v + 255) & ~(int64_t)255; }

// Every query attends every sampled key: the queries are cut into ranges, one workgroup each per tile of sampled
// keys.  Taken is the number of ranges with the least time by the rounds of workgroups the chip needs and the
// rows of a round; setting up a workgroup and the adds it ends in cost about as much as 384 rows.
struct QueryRanges {
  int64_t rows, count;
};
QueryRanges query_ranges(int64_t n_q, int64_t tiles, int64_t slots) {
  QueryRanges r = {n_q, 1};
  int64_t best = INT64_MAX;
  for (int64_t n = 1; n <= std::min<int64_t>(64, (n_q + 511) / 512); ++n) {
    const int64_t rows = ((n_q + n - 1) / n + 63) / 64 * 64, count = (n_q + rows - 1) / rows;
    const int64_t cost = (tiles * count + slots - 1) / slots * (rows + 384);
    if (cost < best) {
      best = cost;
      r = {rows, count};
    }
  }
  return r;
}

// Whether the sampled keys' sums are made by workgroups of 256 keys that write their share of them (rows of a range of one
// query head's queries) to the workspace, to be added up at the end, instead of adding them there with atomics, which took
// 54 us of a pass for the 64 MB of 256 workgroups; to write and read them takes about 20.  This pass, clearing and final adds together, in us at d = 128, atomics -> shares (256 samples): 32 query heads
// on 8 of 4096 rows 99 -> 61, of 8192 146 -> 97, 32 of 8192 149 -> 96, 33 of 2048 64 -> 45; small launches: 4 of 2048 rows 34.3
// -> 35.0, 2 of 8192 41 -> 36, 64 of 512 41 -> 41, 8 of 4096 49 -> 38.  Ranges as many as with atomics.
bool writes_shares(const ha_attn_operands& t, int64_t sample_size, QueryRanges& r) {
  if (t.d != 128 || sample_size == 0 || sample_size % 256 != 0) return false;
  r = query_ranges(t.n_q, t.batch * t.heads * t.segs * (sample_size / 256), 256);
  return true;
}

struct Workspace {
  f32x2* stats;  // per query {L * log2(e), -D}
  float* dk32;  // sums of the sampled keys, (batch, kv_heads, segs, shares, sample_size, d) fp32
  float* dv32;
  int64_t acc_floats;  // per accumulator
  int64_t bytes;
};

Workspace carve(const ha_attn_operands& t, int64_t sample_size, int64_t shares, void* base) {
  Workspace w;
  const int64_t delta_bytes = align256(t.batch * t.heads * t.segs * t.n_q * 8);
  w.acc_floats = t.batch * (t.heads / t.kv_group) * t.segs * shares * sample_size * t.d;
  const int64_t acc_bytes = align256(w.acc_floats * 4);
  w.stats = (f32x2*)base;
  w.dk32 = (float*)((char*)base + delta_bytes);
  w.dv32 = (float*)((char*)base + delta_bytes + acc_bytes);
  w.bytes = delta_bytes + 2 * acc_bytes;
  return w;
}

int check_grads(const ha_attn_operands& t, int64_t sample_size, const ha_attn_grads& g, const char* who) {
  HA_REQUIRE(g.dout && g.dq && g.dk && g.dv, HA_ERR_NULL, "%s: null gradient pointer", who);
  HA_REQUIRE((t.d == 64 || t.d == 128) && t.dv == t.d, HA_ERR_UNSUPPORTED,
             "%s: the backward is built for head dims 64 and 128 with a value dim equal to them", who);
  HA_REQUIRE(g.out_d >= 0 && g.out_d <= t.d && g.out_d % 8 == 0, HA_ERR_SHAPE, "%s: out_d must be a multiple of 8 up to the head dim", who);
  const int64_t strides[] = {g.do_stride_b, g.do_stride_h, g.do_stride_n, g.dq_stride_b, g.dq_stride_h, g.dq_stride_n,
                             g.dk_stride_b, g.dk_stride_h, g.dk_stride_n, g.dv_stride_b, g.dv_stride_h, g.dv_stride_n};
  for (int64_t s : strides) HA_REQUIRE(s % 8 == 0, HA_ERR_SHAPE, "%s: gradient rows must be 16-byte aligned", who);
  HA_REQUIRE(((uintptr_t)g.dout % 16) == 0 && ((uintptr_t)g.dq % 16) == 0 && ((uintptr_t)g.dk % 16) == 0 &&
                 ((uintptr_t)g.dv % 16) == 0,
             HA_ERR_SHAPE, "%s: gradient tensors must be 16-byte aligned", who);
  const int64_t row_strides[] = {g.do_stride_n, g.dq_stride_n, g.dk_stride_n, g.dv_stride_n};
  const int64_t row_counts[] = {t.n_q, t.n_q, t.n_k, t.n_k};
  for (int i = 0; i < 4; ++i) {
    HA_REQUIRE(row_strides[i] > 0 && row_strides[i] * 2 < (1ll << 24), HA_ERR_UNSUPPORTED,
               "%s: gradient row strides must be positive and below 16 MiB", who);
    HA_REQUIRE((row_counts[i] - 1) * row_strides[i] * 2 + t.d * 2 <= (1ll << 32), HA_ERR_UNSUPPORTED,
               "%s: one head of a gradient tensor may span 4 GiB at most", who);
  }
  const Workspace w = carve(t, sample_size, 1, nullptr);  // what every form can work in
  HA_REQUIRE(g.workspace && g.workspace_bytes >= w.bytes && ((uintptr_t)g.workspace % 256) == 0, HA_ERR_WORKSPACE,
             "%s: workspace of %lld bytes (256-byte aligned) required", who, (long long)w.bytes);
  return HA_OK;
}

void fill_bwd_params(const ha_attn_operands& t, const ha_attn_grads& g, const Workspace& w, ha_attn_bwd_params& p) {
  p.q = t.q; p.k = t.k; p.v = t.v; p.dout = g.dout;
  p.out = t.out; p.lse = t.lse;
  p.o_sb = t.o_stride_b; p.o_sh = t.o_stride_h; p.o_sn = t.o_stride_n;
  p.lse_sb = t.lse_stride_b; p.lse_sh = t.lse_stride_h;
  p.stats = w.stats;
  p.dq = g.dq; p.dk = g.dk; p.dv = g.dv; p.dk32 = w.dk32; p.dv32 = w.dv32;
  p.q_sb = t.q_stride_b; p.q_sh = t.q_stride_h; p.q_sn = t.q_stride_n;
  p.k_sb = t.k_stride_b; p.k_sh = t.k_stride_h; p.k_sn = t.k_stride_n;
  p.v_sb = t.v_stride_b; p.v_sh = t.v_stride_h; p.v_sn = t.v_stride_n;
  p.do_sb = g.do_stride_b; p.do_sh = g.do_stride_h; p.do_sn = g.do_stride_n;
  p.dq_sb = g.dq_stride_b; p.dq_sh = g.dq_stride_h; p.dq_sn = g.dq_stride_n;
  p.dk_sb = g.dk_stride_b; p.dk_sh = g.dk_stride_h; p.dk_sn = g.dk_stride_n;
  p.dv_sb = g.dv_stride_b; p.dv_sh = g.dv_stride_h; p.dv_sn = g.dv_stride_n;
  p.q_idx = p.k_idx = p.sampled_idx = nullptr;
  p.qi_sb = p.qi_sh = p.qi_sn = 0;
  p.ki_sb = p.ki_sh = p.ki_sn = 0;
  p.si_sb = p.si_sh = 0;
  p.batch = (int)t.batch; p.heads = (int)t.heads; p.kv_group = (int)t.kv_group;
  p.segs = (int)t.segs; p.seg_stride = t.seg_stride_rows; p.q_seg_off = t.q_seg_offset; p.k_seg_off = t.k_seg_offset;
  p.o_seg_stride = t.o_seg_stride_rows > 0 ? t.o_seg_stride_rows : t.seg_stride_rows;
  p.o_seg_off = t.o_seg_stride_rows > 0 ? t.o_seg_offset : t.q_seg_offset;
  p.n_q = (int)t.n_q; p.n_k = (int)t.n_k;
  p.block_tiles = 1; p.sample_size = 0; p.smooth = 0; p.idx64 = 0;
  p.out_last = (int)((g.out_d ? g.out_d : t.d) / 8) - 1;
  p.accumulate = g.accumulate != 0;
  p.single_tiles = 0;
  p.q_split = (int)t.n_q;
  p.scale = t.scale;
  p.scale_log2 = t.scale * LOG2E;
  p.neg_inv_scale = -1.f / t.scale;
}

// the sampled keys' sums onto their rows of dk, dv
template <typename T, int D, bool FUSED = false>
int launch_add_samples(const ha_block_attn_args& a, const ha_attn_grads& g, const Workspace& w, int64_t shares, hipStream_t stream) {
  const ha_attn_operands& t = a.t;
  const int64_t kv_heads = t.heads / t.kv_group;
  AddSamplesParams p;
  p.sums[0] = w.dk32; p.sums[1] = w.dv32;
  p.grad[0] = g.dk; p.grad[1] = g.dv;
  p.sb[0] = g.dk_stride_b; p.sh[0] = g.dk_stride_h; p.sn[0] = g.dk_stride_n;
  p.sb[1] = g.dv_stride_b; p.sh[1] = g.dv_stride_h; p.sn[1] = g.dv_stride_n;
  p.sampled_idx = a.sampled_idx;
  p.si_sb = a.sampled_stride_b; p.si_sh = a.sampled_stride_h;
  p.seg_stride = t.seg_stride_rows; p.k_seg_off = t.k_seg_offset;
  p.idx64 = a.idx_type == HA_IDX_I64;
  p.kv_heads = (int)kv_heads; p.sample_size = (int)a.sample_size; p.shares = (int)shares; p.segs = (int)t.segs;
  p.k_factor = t.scale;
  const int64_t workgroups = t.batch * kv_heads * t.segs * a.sample_size * (D / 8) / 256;  // sample_size is a multiple of 128
  if (workgroups >= (1ll << 31)) return ha_fail(HA_ERR_SHAPE, "attention backward: %lld workgroups", (long long)workgroups);
  hipLaunchKernelGGL((ha_bwd_add_samples_kernel<T, D, FUSED>), dim3((unsigned)workgroups, 2), dim3(256), 0, stream, p);
  return ha_launch_status("attention backward: sampled keys");
}

template <typename T, int D>
int run_block_bwd(const ha_block_attn_args& a, const ha_attn_grads& g, hipStream_t stream) {
  const ha_attn_operands& t = a.t;
  QueryRanges ranges;
  const bool shared_out = writes_shares(t, a.sample_size, ranges), one_kernel = ha_block_bwd_fused_takes(a);
  const int64_t wanted = shared_out ? t.kv_group * ranges.count : one_kernel ? ha_block_bwd_fused_shares(t.batch * t.heads * t.segs, t.n_q) : 1;
  // (a workspace for the sums alone takes the passes that add them with atomics)
  const bool room = carve(t, a.sample_size, wanted, nullptr).bytes <= g.workspace_bytes;
  const int64_t shares = room ? wanted : 1;
  const bool wide_samples = shared_out && room;
  const Workspace w = carve(t, a.sample_size, shares, g.workspace);
  int st;
  ha_attn_bwd_params p;
  fill_bwd_params(t, g, w, p);
  p.q_idx = a.q_idx; p.k_idx = a.k_idx; p.sampled_idx = a.sampled_idx;
  p.qi_sb = a.q_idx_stride_b; p.qi_sh = a.q_idx_stride_h; p.qi_sn = a.q_idx_stride_n;
  p.ki_sb = a.k_idx_stride_b; p.ki_sh = a.k_idx_stride_h; p.ki_sn = a.k_idx_stride_n;
  p.si_sb = a.sampled_stride_b; p.si_sh = a.sampled_stride_h;
  p.block_tiles = (int)((a.block_size + 127) / 128);
  p.sample_size = (int)a.sample_size;
  p.smooth = a.smooth_block != 0;
  p.idx64 = a.idx_type == HA_IDX_I64;
  const int64_t bh = t.batch * t.heads * t.segs, bhk = t.batch * (t.heads / t.kv_group) * t.segs;
  if (one_kernel && room) {
    st = ha_launch_block_bwd_fused(p, std::is_same<T, f16_t>::value, stream);
    if (st != HA_OK || a.sample_size == 0) return st;
    if constexpr (D == 64) return launch_add_samples<T, D, true>(a, g, w, shares, stream);
  }
  if (a.sample_size > 0 && !wide_samples) {
    // the two arrays of sums lie one behind the other in the workspace (each a multiple of 256 bytes): one fill
    const int64_t n4 = (int64_t)(((char*)w.dv32 - (char*)w.dk32) + align256(w.acc_floats * 4)) / 16;
    hipLaunchKernelGGL(ha_bwd_zero_kernel, dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0, stream, (f32x4*)w.dk32, n4);
    st = ha_launch_status("attention backward: clear");
    if (st != HA_OK) return st;
  }
  st = launch_pass<T, D, HA_BWD_DQ_BLOCK, false>(p, bh * (t.n_q / ST_ROWS), stream, "ha_block_attn_bwd: dq");
  if (st != HA_OK) return st;
  // 256 keys per workgroup where their tiles are all of one block, smooth windows apart, and more than half the chip
  // has work.  dk, dv of the blocks in us, d 128, 128 -> 256 keys, workgroups of 256 in brackets: 8 heads of 4096 rows
  // in blocks of 256 (128) 20.7 -> 24.8, 9 heads (144) 35.9 -> 25.5, 17 (272) 56.7 -> 49.3, 32 query heads on 8 of 4096
  // (128) 53 -> 61, of 4224 (136) 76 -> 61, of 16384 (512) 225 -> 159; blocks of 512, 32 on 8 of 8320 (264) 221 -> 162.
  const int64_t wide_wgs = bhk * ((t.n_k + 255) / 256);
  if (D == 128 && !p.smooth && p.block_tiles % 2 == 0 && wide_wgs > 128)
    st = ha_launch_bwd_wide(p, HA_BWD_DKV_BLOCK, false, std::is_same<T, f16_t>::value, wide_wgs, stream,
                            "ha_block_attn_bwd: dk, dv of the blocks");
  else
    st = launch_pass<T, D, HA_BWD_DKV_BLOCK, false>(p, bhk * (t.n_k / ST_ROWS), stream, "ha_block_attn_bwd: dk, dv of the blocks");
  if (st != HA_OK) return st;
  if (a.sample_size > 0) {
    if (wide_samples) {
      p.q_split = (int)ranges.rows;
      st = ha_launch_bwd_wide(p, HA_BWD_DKV_SAMPLED, false, std::is_same<T, f16_t>::value, bh * (a.sample_size / 256) * ranges.count, stream,
                              "ha_block_attn_bwd: dk, dv of the sampled keys");
    } else {
      const int64_t tiles = bh * (a.sample_size / ST_ROWS);
      const QueryRanges r = query_ranges(t.n_q, tiles, D <= 64 ? 512 : 256);
      p.q_split = (int)r.rows;
      st = launch_pass<T, D, HA_BWD_DKV_SAMPLED, false>(p, tiles * r.count, stream, "ha_block_attn_bwd: dk, dv of the sampled keys");
    }
    if (st != HA_OK) return st;
    return launch_add_samples<T, D>(a, g, w, shares, stream);
  }
  return HA_OK;
}

// The form of a pass of exact attention with the least estimated time.
//   WHOLE: 128 stationary rows per workgroup, causal tiles in pairs.
//   SINGLE: causal tiles one by one, longest first.
//   SPLIT: 64, the steps of the streamed tiles split over waves (HALVES = 2), half as many steps per wave.
//   WIDE: 256 (d = 128; dk, dv: attn_bwd_wide.hip, dq: attn_bwd_wide_dq.hip).
// What bounds a launch of few workgroups is the longest chain of steps of one of them with CUs idle: a wave alone on its
// SIMD issues steps as fast as two together, so smaller workgroups fill the idle CUs; on a full chip they do the same
// work slower (twice the set-up and tile loads per row; dq at d = 128 also one workgroup per CU instead of two).
//
// Pairs of causal tiles are equal workgroups, which leave CUs idle in a last round that is not full.  Single ones fill it,
// but read a sequence's rows at times far apart: up to 4.5 pairs per CU they are never slower.  Pairs | split | single, dq,
// then dk, dv, in us at d = 64, pairs per CU in brackets: 24 heads of 2048 rows (0.75) 40 | 33 | 36, 58 | 41 | 53; 48 (1.5) 60
// | 55 | 51, 80 | 71 | 67; 80 (2.5) 88 | 87 | 74, 125 | 113 | 105; 128 (4) 119 | 139 | 114, 161 | 179 | 154; 300 (9.4) 292 |
// 426 | 299, 405 | 482 | 411; 700 (22) 670 | 1077 | 773, 920 | 1206 | 998; 24 of 4096 (1.5) 105 | 97 | 89, 141 | 129 | 117; 32
// query heads on 8 of 2048 (1, dk, dv 0.25) 39 | 40 | 38, 178 | 101 | 162.  d = 128: 24 of 2048 83 | 83 | 67, 108 | 99 | 95.
// Their estimates in us at d = 64: the longest chain and a part of the load beside it, or a CU's share of the steps and
// starts; within 10 % of the times at 27 shapes.
//
// The others are estimated in steps of 32 streamed rows: rounds of workgroups over the CUs times their chain, or, for causal
// tiles one by one (longest first), the longest chain or a CU's share of all.  The weights are fitted to the times of WHOLE
// and SPLIT of both passes at 57 shapes per head dim (4 to 128 heads, grouped and not, 512 to 4096 rows).
// Times in us, whole -> split, dq | dk, dv, bf16 causal: d 64, 4 heads of 1000 rows 24 -> 13 | 29 -> 16; d 128, 12 heads of
// 2048 75 -> 41 | 93 -> 49, 32 on 8 of 2048 78 (split 98: stays) | 320 -> 161.  Full: d 64, 48 heads of 4096 rows without
// mask 295 (split 335) | 387 (451).
// A wide step of dk, dv is 1.05 whole steps long on an idle chip and 1.3 on a full one, for twice the pairs.  The better of
// the others -> wide, dk, dv in us at 35 shapes, among them (causal) 24 heads of 4096 rows 307 -> 223, 32 387 -> 271, of 8192
// 1347 -> 972, 256 of 256 41 -> 32; (not causal) 24 of 2048 147 -> 108, 32 of 4096 684 -> 477; 32 on 8, 300 on 8192 rows 124
// -> 84.  Where the chip is not full the others stay: causal 32 on 8 heads of 4096 413 (wide 696), 12 of 2048 56 (103).
// dq: causal, wide from two and a half tiles of 128 rows per CU on, the better of the others -> wide in us: 24 heads of 2048
// rows (1.5) 67 -> 71, 32 of 2048 (2) 71 -> 75, 300 of 256 (2.3) 35 -> 37, 20 of 4096 (2.5) 140 -> 144, 80 of 1024 (2.5) 55 ->
// 46, 24 of 4096 (3) 161 -> 154, 128 of 1024 (4) 72 -> 68, 32 of 4096 (4) 209 -> 185, 2048 of 128 (8) 174 -> 115, 8 segments of
// 2048 with 32 heads (16) 500 -> 466.  Without mask, where wide workgroups occupy more than half of the CUs (in brackets)
// and have more than 128 keys: 16 of 2000 (128) 62 -> 64, 17 (136) 82 -> 66, 33 of 2048 (264) 149 -> 151, 32 of 4096 (512)
// 376 -> 342, of 4096 on 256 keys (512) 51 -> 52, on 128 42 -> 44, 2048 of 128 (2048) 108 -> 121.
enum ExactForm { WHOLE, SINGLE, SPLIT, WIDE };
ExactForm exact_form(int d, bool dkv, int64_t seqs, int64_t rows, int64_t streamed_rows, int64_t group, bool causal) {
  const double cus = 256., set_up = 2., margin = 0.97;
  const double tiles = (double)((rows + 127) / 128), split_tiles = (double)((rows + 63) / 64), split_wgs = seqs * split_tiles;
  if (d == 128 && !dkv && (causal ? seqs * tiles >= 2.5 * cus : seqs * ((rows + 255) / 256) > cus / 2 && streamed_rows > 128)) return WIDE;
  const bool few_pairs = causal && seqs * std::ceil(tiles / 2) <= 4.5 * cus;
  if (d == 64 && causal) {
    if (!few_pairs) return WHOLE;
    const double wgs = seqs * tiles, share = 2. * group * wgs * (tiles + 1) / cus, chain = 4. * group * tiles;
    const double split_share = group * split_wgs * (split_tiles + 1) / 2 / cus, split_chain = group * split_tiles;
    const double single = dkv ? std::max(0.61 * chain + 0.06 * share + 8, 0.53 * share + 1.6 * wgs / cus + 5)
                              : std::max(0.43 * chain + 0.06 * share + 5, 0.39 * share + 1.6 * wgs / cus + 5);
    const double split = dkv ? std::max(0.75 * split_chain + 7, 0.58 * split_share + 1.5 * split_wgs / cus + 5)
                             : std::max(0.56 * split_chain + 6, 0.43 * split_share + 1.7 * split_wgs / cus + 5);
    return split < single ? SPLIT : SINGLE;
  }
  // time of a step where a CU has several workgroups to take, against one alone
  const double full_whole = d == 64 || dkv ? 0.95 : 0.8, full_split = d == 64 ? 1.25 : dkv ? 1. : 1.4;
  const double rounds = std::ceil(seqs * (causal ? std::ceil(tiles / 2) : tiles) / cus);
  double whole, split;
  if (causal) {
    whole = (rounds > 1 ? full_whole : 1.) * rounds * 4 * (tiles + 1) * group + 2 * set_up * rounds;
    split = std::max(split_tiles * group + set_up,
                     full_split * split_wgs / cus * group * (split_tiles + 1) / 2 + set_up * std::max(1., split_wgs / cus));
  } else {
    const double streamed = (double)((streamed_rows + 127) / 128), split_rounds = std::ceil(split_wgs / cus);
    whole = (rounds > 1 ? full_whole : 1.) * rounds * 4 * streamed * group + set_up * rounds;
    split = (split_rounds > 1 ? full_split : 1.) * split_rounds * 2 * streamed * group + set_up * split_rounds;
  }
  const ExactForm narrow = split < margin * whole ? SPLIT : few_pairs ? SINGLE : WHOLE;
  if (d != 128 || !dkv) return narrow;
  const double wide_tiles = (double)((rows + 255) / 256), wide_wgs = seqs * wide_tiles, chain = (double)((streamed_rows + 31) / 32) * group;
  const double step = 1.05 + 0.25 * std::min(1., wide_wgs / cus), wide_rounds = std::ceil(wide_wgs / cus), wide_set_up = 3.;
  const double wide = causal ? std::max(1.05 * chain + wide_set_up, 1.3 * wide_wgs / cus * std::max(chain / 2, chain - 4 * (wide_tiles - 1) * group) +
                                                                        wide_set_up * std::max(1., wide_wgs / cus))
                             : wide_rounds * (step * chain + wide_set_up);
  return wide < margin * std::min(whole, split) ? WIDE : narrow;
}

// one pass of exact attention over `seqs` sequences with `rows` stationary rows each
template <typename T, int D, int PASS>
int launch_exact(const ha_attn_bwd_params& p, int64_t seqs, int64_t rows, int64_t streamed_rows, int64_t group, bool causal,
                 hipStream_t stream, const char* what) {
  const ExactForm form = exact_form(D, PASS == HA_BWD_DKV_EXACT, seqs, rows, streamed_rows, group, causal);
  if (form == WIDE) {
    constexpr int is_f16 = std::is_same<T, f16_t>::value;
    const int64_t grid = seqs * ((rows + 255) / 256);
    return PASS == HA_BWD_DQ_EXACT ? ha_launch_bwd_wide_dq(p, causal, is_f16, grid, stream, what) : ha_launch_bwd_wide(p, PASS, causal, is_f16, grid, stream, what);
  }
  if (form == SPLIT) {
    const int64_t grid = seqs * ((rows + 63) / 64);
    return causal ? launch_pass<T, D, PASS, true, 2>(p, grid, stream, what) : launch_pass<T, D, PASS, false, 2>(p, grid, stream, what);
  }
  const int64_t tiles = (rows + ST_ROWS - 1) / ST_ROWS;
  if (causal && form == SINGLE) {
    ha_attn_bwd_params single = p;
    single.single_tiles = 1;
    return launch_pass<T, D, PASS, true>(single, seqs * tiles, stream, what);
  }
  if (causal) return launch_pass<T, D, PASS, true>(p, seqs * ((tiles + 1) / 2), stream, what);
  return launch_pass<T, D, PASS, false>(p, seqs * tiles, stream, what);
}

template <typename T, int D>
int run_flash_bwd(const ha_attn_operands& t, bool causal, const ha_attn_grads& g, hipStream_t stream) {
  const Workspace w = carve(t, 0, 1, g.workspace);
  ha_attn_bwd_params p;
  fill_bwd_params(t, g, w, p);
  const int64_t bh = t.batch * t.heads * t.segs, bhk = t.batch * (t.heads / t.kv_group) * t.segs;
  const int st = launch_exact<T, D, HA_BWD_DQ_EXACT>(p, bh, t.n_q, t.n_k, 1, causal, stream, "ha_flash_attn_bwd: dq");
  if (st != HA_OK) return st;
  return launch_exact<T, D, HA_BWD_DKV_EXACT>(p, bhk, t.n_k, t.n_q, t.kv_group, causal, stream, "ha_flash_attn_bwd: dk, dv");
}

}  // namespace

extern "C" int64_t ha_attn_bwd_workspace_bytes(const ha_attn_operands* t, int64_t sample_size) {
  if (!t || t->batch <= 0 || t->heads <= 0 || t->n_q <= 0 || t->n_k <= 0 || t->d <= 0 || t->kv_group <= 0 ||
      t->heads % t->kv_group != 0 || sample_size < 0 || t->segs < 1)
    return ha_fail(HA_ERR_SHAPE, "ha_attn_bwd_workspace_bytes: sizes must be positive, kv_group dividing heads, segs >= 1");
  QueryRanges r;
  int64_t shares = 1;
  if (writes_shares(*t, sample_size, r)) shares = t->kv_group * r.count;
  else if (ha_block_bwd_fused_shape(*t, sample_size)) shares = ha_block_bwd_fused_shares(t->batch * t->heads * t->segs, t->n_q);
  return carve(*t, sample_size, shares, nullptr).bytes;
}

extern "C" int64_t ha_block_attn_bwd_workspace_bytes(const ha_block_attn_args* args) {
  if (!args) return ha_fail(HA_ERR_NULL, "ha_block_attn_bwd_workspace_bytes: null argument block");
  const ha_block_attn_args& a = *args;
  const int64_t most = ha_attn_bwd_workspace_bytes(&a.t, a.sample_size);
  QueryRanges r;
  if (most < 0 || writes_shares(a.t, a.sample_size, r) || ha_block_bwd_fused_takes(a)) return most;
  return carve(a.t, a.sample_size, 1, nullptr).bytes;
}

extern "C" int ha_block_attn_bwd(const ha_block_attn_args* args, const ha_attn_grads* grads, void* stream) {
  HA_REQUIRE(args && grads, HA_ERR_NULL, "ha_block_attn_bwd: null argument");
  const ha_block_attn_args& a = *args;
  int st = ha_check_block_attn_args(a, "ha_block_attn_bwd");
  if (st != HA_OK) return st;
  st = check_grads(a.t, a.sample_size, *grads, "ha_block_attn_bwd");
  if (st != HA_OK) return st;
  HA_REQUIRE(!a.accumulate, HA_ERR_UNSUPPORTED, "ha_block_attn_bwd: no backward of the fused merge (accumulate)");
  HA_REQUIRE(a.sample_bias == 0.f && !a.mask_sampled_in_block, HA_ERR_UNSUPPORTED,
             "ha_block_attn_bwd: no backward of the residual estimator (sample_bias, mask_sampled_in_block)");
  HA_REQUIRE(!a.smooth_block || a.block_size <= 128 * (MAX_SMOOTH_TILES - 1), HA_ERR_UNSUPPORTED,
             "ha_block_attn_bwd: smoothed blocks longer than %d rows are not built", 128 * (MAX_SMOOTH_TILES - 1));
  hipStream_t s = (hipStream_t)stream;
  if (a.t.dtype == HA_F16) return a.t.d == 64 ? run_block_bwd<f16_t, 64>(a, *grads, s) : run_block_bwd<f16_t, 128>(a, *grads, s);
  return a.t.d == 64 ? run_block_bwd<bf16_t, 64>(a, *grads, s) : run_block_bwd<bf16_t, 128>(a, *grads, s);
}

extern "C" int ha_flash_attn_bwd(const ha_attn_operands* t, int causal, const ha_attn_grads* grads, void* stream) {
  HA_REQUIRE(t && grads, HA_ERR_NULL, "ha_flash_attn_bwd: null argument");
  int st = ha_check_operands(*t, "ha_flash_attn_bwd");
  if (st != HA_OK) return st;
  st = check_grads(*t, 0, *grads, "ha_flash_attn_bwd");
  if (st != HA_OK) return st;
  hipStream_t s = (hipStream_t)stream;
  if (t->dtype == HA_F16)
    return t->d == 64 ? run_flash_bwd<f16_t, 64>(*t, causal != 0, *grads, s) : run_flash_bwd<f16_t, 128>(*t, causal != 0, *grads, s);
  return t->d == 64 ? run_flash_bwd<bf16_t, 64>(*t, causal != 0, *grads, s) : run_flash_bwd<bf16_t, 128>(*t, causal != 0, *grads, s);
}
