// MFMA attention forward kernels for gfx950: the sorted block-diagonal + sampled-column kernel and
// the exact (flash) kernel share one body.
//
// Reference semantics: _fwd_hyper_kernel (src/hyper_attn_triton.py:26-192) and _fwd_kernel with
// bias "none" (src/flash_attn_triton.py:57-267); the resume-from-a-previous-partial-result mode
// folds add_self_attentions (src/attn_utils.py:6-50) into the kernel.
//
// Work decomposition.  A workgroup of 4 waves owns consecutive (sorted) query positions of one (virtual) head:
// 256 at head dim 64, 64 queries (two 32-wide MFMA column blocks) per wave, 128 at head dim 128, 32 queries per
// wave (WaveShape below), and a CU holds two workgroups (exact attention at head dim 128 also 8 waves, 256 queries, one
// workgroup: large_tiles); at head dim 64 launches of few workgroups and windows that neighbouring
// reference tiles do not share take 128 queries too (NB = 1), three workgroups per CU.  Query rows and key
// rows go from HBM straight into LDS (global_load_lds, 16 bytes per lane, whole rows per
// instruction, no staging registers), row-major with their 16-byte pieces XOR-swizzled by the row
// number (the swizzle is applied on the source side: a lane fetches the piece that belongs in its
// LDS slot).  Q and K operands are read with ds_read_b128, the V^T operand with the transposing
// ds_read_b64_tr_b16.
//
// MFMA formulation (v_mfma_f32_32x32x16_{f16,bf16}; A: lane -> row lane%32, k = 8*(lane/32)..+7;
// B: lane -> column lane%32, same k; C: lane -> column lane%32, rows 8*(i/4) + 4*(lane/32) + i%4):
//   S^T = K  Q^T   (M = keys,  N = queries, K = head dim)   -> a lane holds 16 keys of ONE query
//   O^T = V^T P^T  (M = dv,    N = queries, K = keys)       -> P^T comes straight from the S^T registers
// so the soft-max statistics are per-lane scalars.  ds_read_b64_tr_b16 gives lane i of a 16-lane
// group element i%4 of the 8-byte words addressed by lanes 4j + i/4 (j = 0..3), so a group that
// points its lanes at (key j, dv word w) receives V[key 0..3][dv base + i]: the V^T operand in
// exactly the key order of the C registers.
//
// Software pipeline.  The loop body is a chain of straight-line blocks, one per half-step of 16 keys, and
// each block mixes three independent things: the exponentials of half-step u, the P.V MFMAs of
// half-step u-1 and half of the S^T MFMAs of the next 32-key step, issued one MFMA and its share of the
// vector work at a time (clustering the MFMAs of a block, with or without a raised wave priority, measured
// 4 to 6 % slower); two waves per SIMD fill each other's gaps.  Keys are streamed in tiles of 64
// rows; the K tiles are shifted by 32 keys against the V tiles (K tile c holds keys 64c-32..64c+31),
// so the K rows read during an iteration all sit in one tile, which is read in that iteration only
// and can be refilled in the next, and the V^T operands of a half-step are fetched one block ahead.
//
// Soft-max without a running maximum.  The exponentials use the current reference exponent m of
// the row as is (base 2, scale*log2(e) folded into one FMA; v_exp_f32 is 2^x); P is rounded to the
// input type before P.V as the reference does (src/hyper_attn_triton.py:135) and the row sums are
// taken over the rounded values.  Only when the sum of a lane's 8 values of a half-step reaches 2^14
// (or is not a number: nothing seen yet) is the row maximum computed, m raised, the accumulators
// rescaled and the half-step redone; below that bound every value is finite in fp16 and the result
// does not depend on m beyond rounding.  m only ever grows, and starts from the true maximum of the
// first keys or from the log-sum-exp of the partial result that is being resumed.  What rounding it depends on: the
// key whose score is m has a weight of exactly 1, and the split kernel (attn_fwd_split.inc) has four such keys per row.  Where
// single causal tiles of this kernel take its place, m follows the row maximum in a sequence's first tile (FOLLOW),
// whose rows of few keys are most of the error.  Error against float64 over that of the split kernel, without | with, 16-bit
// types, N(0,1) and clustered data: d = 64, 100 heads of 600 rows to 32 of 4096 1.015 to 1.024 | 0.992 to 0.997, d = 128, 48 of
// 685 to 16 of 4096 1.010 to 1.024 | 0.994 to 1.000.  It costs nothing where the first tiles run beside longer ones (48 of
// 2048 rows 44 us, d = 128 44 of 1024 32) and up to 5 us where they are a round of their own (d = 64 130 of 1024 35.5 -> 38.1,
// 100 of 700 21.0 -> 23.3, d = 128 96 of 520 26.4 -> 31.0; the split kernel 59, 27 and 37; 150 of 300 16.3 -> 18.9, split 17.0).
#include "ha_common.h"
#include "attn_tiles.h"
#include "attn_fwd.h"
#include "unit_ranking.h"

#include <stdlib.h>

#include <algorithm>
#include <cmath>

namespace {

constexpr int KC = 64;           // keys per LDS tile
constexpr float HALF_SUM_LIMIT = 16384.f;  // 2^14: a lane's half-step sum below this has no fp16 overflow
// Reference exponent (log2 units) of a row that has seen no key yet.  Finite on purpose: a masked score
// (-inf) then gives P = 2^(-inf) = 0 without any special case, where -inf - (-inf) would be a NaN that
// sends every half-step of a masked chunk through the rescaling path; a real score gives 2^(+huge) = inf,
// which takes that path once and sets the row's true exponent.
constexpr float M_FLOOR = -1e30f;

// A workgroup's waves and their queries.  A wave's registers hold the output accumulators
// of its queries (queries x head dim floats over 64 lanes), their query fragments and two S^T buffers: 64
// queries per wave fit 256 registers at head dim 64, at head dim 128 only 32 do.  256 registers is what lets
// two waves share a SIMD, and a wave on its own leaves the matrix pipe idle through every stretch of vector
// work and every wait (one wave per SIMD with 64 queries and 512 registers ran the d = 128 loop at 1170
// cycles per 16 keys where its MFMAs alone take 512).  The two waves of a SIMD belong to two workgroups: neither waits at the
// other's barriers, and one's set-up and output stage run beside the other's loop.  With 8 waves of 32 queries at
// d = 128 (256 queries, one workgroup per CU) a wave stood at the barrier of a 64-key iteration for a quarter of it: 2 x 32
// heads of 65536 rows, smooth blocks of 512 2.80 -> 2.58 ms, 16 x 20479 causal, d = 96 508 -> 457 us (whole call, 2.5 rounds of 256
// workgroups), leaves of 2048 rows, 32 x 32768 671 -> 650, 24 heads of 2048 causal 55 -> 38.  Exact attention still takes 8 waves where
// that fills a last round better (large_tiles).
template <int D>
struct WaveShape {
  static constexpr int NB = D <= 64 ? 2 : 1;        // 32-query MFMA column blocks per wave
  static constexpr int QW = 32 * NB;                // queries per wave
  static constexpr int WAVES = 4;                   // waves per workgroup
  static constexpr int QUERIES = QW * WAVES;        // sorted query positions per workgroup
  static constexpr int THREADS = 64 * WAVES;
};

// x / y for 0 <= x < 2^31 by the divisor's multiply-and-shift constants
__device__ __forceinline__ int fast_div(int x, ha_divisor y) { return (int)(((uint64_t)(uint32_t)x * y.magic) >> y.shift); }

// What workgroup `id` of a launch with ranking workgroups does: a unit's number, or -1; in `id` and `count` its number among
// the others and how many they are, no less than which means that it is none of them.
__device__ __forceinline__ int ranking_unit(const ha_rank_beside& a, int& id, int& count) {
  const int unit = id - a.first_group * NUM_XCD, ranking = a.groups * NUM_XCD;
  count = a.tiles;
  if (unit < 0) return -1;
  id = unit < ranking ? count : id - ranking;
  return unit < a.units ? unit : -1;
}

// LDS byte offsets of one lane's operand reads, relative to a tile base (fixed for the whole kernel).
template <int DC>
struct LaneOffsets {
  int k[DC / 16];  // Q / K operand piece of k-step ks for tile row lane%32 (add 32 rows for the upper half)
  int v[DC / 32];  // V^T operand word for dv block db, keys 0..3 (+4 for the upper lane half) of a 16-key half-step
};

// P of the 8 values of half-step H a lane holds per query block (elements 8H..8H+7 of its S^T
// registers), rounded to T, and their sums.  m is the reference exponent (log2 units).
// sums of the 8 values per query block of a half-step's P.  They go through the matrix pipe: v_dot2
// does not overlap with the big MFMAs at all.
template <typename T, int NB>
__device__ __forceinline__ void half_step_sums(const typename ElemTraits<T>::vec8 (&pn)[NB], float (&sum)[NB]) {
  typedef typename ElemTraits<T>::vec4 vec4;
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    const vec4 lo = __builtin_shufflevector(pn[nb], pn[nb], 0, 1, 2, 3);
    const vec4 hi = __builtin_shufflevector(pn[nb], pn[nb], 4, 5, 6, 7);
    f32x4 acc_sum = {0.f, 0.f, 0.f, 0.f};
    acc_sum = Mfma<T>::quad_sum(lo, acc_sum);
    acc_sum = Mfma<T>::quad_sum(hi, acc_sum);
    sum[nb] = acc_sum[0];
  }
}
template <typename T, int NB, int H>
__device__ __forceinline__ void half_step_p(const f32x16 (&s_use)[NB], const float (&m)[NB], float scale_log2,
                                            typename ElemTraits<T>::vec8 (&pn)[NB], float (&sum)[NB]) {
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
      const f32x2 two = {__builtin_amdgcn_exp2f(__builtin_fmaf(s_use[nb][H * 8 + e], scale_log2, -m[nb])),
                         __builtin_amdgcn_exp2f(__builtin_fmaf(s_use[nb][H * 8 + e + 1], scale_log2, -m[nb]))};
      const typename ElemTraits<T>::vec2 p2 = __builtin_convertvector(two, typename ElemTraits<T>::vec2);
      pn[nb][e] = p2[0];
      pn[nb][e + 1] = p2[1];
    }
  half_step_sums<T, NB>(pn, sum);
}

// The rare path of a half-step: raise the reference exponents to the row maxima of the half-step,
// rescale the row sums and redo the half-step's P.  alpha is what everything accumulated under the old
// exponents has to be multiplied by.
template <typename T, int NB, int H>
__device__ __forceinline__ void half_step_rescale(const f32x16 (&s_use)[NB], float scale_log2,
                                                  float (&alpha)[NB], float (&m_run)[NB], float (&l_run)[NB],
                                                  typename ElemTraits<T>::vec8 (&pn)[NB], float (&sum)[NB], bool follow) {
  float m_use[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    // only this half-step's values: the other half of the step raises the exponents itself if it has
    // to, and the two rare paths of a step then share no work the compiler would compute up front
    float v = s_use[nb][H * 8];
#pragma unroll
    for (int e = 1; e < 8; ++e) v = fmaxf(v, s_use[nb][H * 8 + e]);
    if (H == 0 && follow) {  // the whole step's: its second half goes on under the same exponents
#pragma unroll
      for (int e = 8; e < 16; ++e) v = fmaxf(v, s_use[nb][e]);
    }
    v = ha_max_xor32(v) * scale_log2;
    const float m_new = fmaxf(m_run[nb], v);
    // 2^(old - new) <= 1; nothing is accumulated yet under the floor exponent of a fresh row
    alpha[nb] = __builtin_amdgcn_exp2f(m_run[nb] - m_new);
    m_run[nb] = m_new;
    l_run[nb] *= alpha[nb];
    // rows that have seen no key yet (all masked) keep the floor; their P is 2^(-inf) = 0
    m_use[nb] = m_new;
  }
  half_step_p<T, NB, H>(s_use, m_use, scale_log2, pn, sum);
}

// Issue order of a block: each of its NB*DC/16 large MFMAs is followed by a share of the P arithmetic (8 NB multiply-adds,
// 4 NB conversions, 8 NB exponentials in all), so the soft-max fills the issue slots behind every MFMA instead of running as
// one burst after the last of them.  Measured 3 % faster than the scheduler's own order at d = 64, 8 % at d = 128.
// With one 32-query block per wave (d = 128) a block reads twice as much from LDS per MFMA, and the issue of 12 reads in a row
// is half as long as its MFMAs: they are spread behind the first six, the K operands (needed by the second half of the MFMAs)
// first.  32 x 32768 grouped: leaves 641 -> 617 us, a level 200 -> 198, smooth 2 x 32 x 65536 2.495 -> 2.455 ms.  At d = 64
// (six reads) the same order measured 0 to 1 % slower; there they stay at the head of the block.
template <int NB, int DC, int G = 0>
__device__ __forceinline__ void half_step_order() {
  constexpr int MFMAS = NB * DC / 16, DB = DC / 32;
  constexpr int V_LEFT = 2 * DB - (G < 4 ? 2 * (G - 1) : G + 2);  // transposing V^T reads not issued yet (G > 0)
  constexpr int READS = NB > 1 ? 0 : G == 0 ? DC / 32 : V_LEFT > (G < 4 ? 2 : 1) ? (G < 4 ? 2 : 1) : V_LEFT;
  __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                                // one MFMA
  if constexpr (READS > 0) __builtin_amdgcn_sched_group_barrier(0x100, READS, 0);   // LDS reads
  __builtin_amdgcn_sched_group_barrier(0x002, (12 * NB + MFMAS - 1) / MFMAS, 0);    // its share of plain VALU
  __builtin_amdgcn_sched_group_barrier(0x400, (8 * NB + MFMAS - 1) / MFMAS, 0);     // and of the transcendentals
  if constexpr (G + 1 < MFMAS) half_step_order<NB, DC, G + 1>();
}

// One block of the pipeline: half-step H (16 keys) of the 32-key step whose S^T is s_use.
//   MFMAs : P.V of the previous half-step (operands vf, pb, both in registers) and this half's share
//           (k-steps H*KSTEPS/2 ..) of the next step's S^T, K rows k_row_off.. of k_tile
//   VALU  : P of this half-step from s_use -> pb (for the next block) and the row sums
//   follow: the reference exponents follow the rows' maxima, raised at every step of 32 keys
//   LDS   : V^T of this half-step's keys (v_key_off.. of v_tile) -> vf (for the next block)
template <typename T, int D, int H, int DC, int NB>
__device__ __forceinline__ void half_step(const f32x16 (&s_use)[NB], f32x16 (&s_fill)[NB],
                                          const unsigned char* k_tile, int k_row_off,
                                          const unsigned char* v_tile, int v_key_off, const LaneOffsets<DC>& lo,
                                          const typename ElemTraits<T>::vec8 (&qf)[NB][DC / 16],
                                          f32x16 (&acc)[DC / 32][NB], float (&m_run)[NB],
                                          float (&l_run)[NB],
                                          typename ElemTraits<T>::vec8 (&pb)[NB],
                                          typename ElemTraits<T>::vec8 (&vf)[DC / 32], float scale_log2,
                                          bool follow = false) {
  typedef typename ElemTraits<T>::vec8 vec8;
  constexpr int KH = DC / 32;  // k-steps of this half
  constexpr int DB = DC / 32;

  vec8 kf[KH];
#pragma unroll
  for (int k2 = 0; k2 < KH; ++k2) kf[k2] = lds_read_k<T>(k_tile, lo.k[H * KH + k2] + k_row_off);
  vec8 vf_next[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) vf_next[db] = lds_read_vt<T>(v_tile, lo.v[db] + v_key_off, D * 2);
  // d = 64: the LDS reads stay at the head of the block: their latency hides behind the P.V MFMAs and the
  // exponentials instead of being waited for where the compiler would sink them to
  if constexpr (NB > 1) __builtin_amdgcn_sched_barrier(0);

#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[db][nb] = Mfma<T>::run(vf[db], pb[nb], acc[db][nb]);
  if (H == 0) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int i = 0; i < 16; ++i) s_fill[nb][i] = 0.f;
  }
#pragma unroll
  for (int k2 = 0; k2 < KH; ++k2)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) s_fill[nb] = Mfma<T>::run(kf[k2], qf[nb][H * KH + k2], s_fill[nb]);

  vec8 pn[NB];
  float sum[NB];
  half_step_p<T, NB, H>(s_use, m_run, scale_log2, pn, sum);
  half_step_order<NB, DC>();
  // One compare for all query blocks: their sums are >= 0 or NaN, so the total is below the limit
  // only if every one is.  Not "total >= limit": a NaN (row that has seen nothing yet) must take the rare
  // path too.
  float total = sum[0];
#pragma unroll
  for (int nb = 1; nb < NB; ++nb) total += sum[nb];
  const bool redo = (H == 0 && follow) || !(total < HALF_SUM_LIMIT);
  if (__builtin_expect(__builtin_amdgcn_ballot_w64(redo) != 0, false)) {
    float alpha[NB];
    half_step_rescale<T, NB, H>(s_use, scale_log2, alpha, m_run, l_run, pn, sum, follow);
    // the accumulators hold everything up to the previous half-step (its P.V was issued above; the
    // P.V of this half-step is added by the next block, under the new exponents)
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[db][nb][i] *= alpha[nb];
  }
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    l_run[nb] += sum[nb];
    pb[nb] = pn[nb];
  }
#pragma unroll
  for (int db = 0; db < DB; ++db) vf[db] = vf_next[db];
}

}  // namespace

// FORM (gathered kernel only): the common configurations, default samples (rows 0 .. sample_size-1), have instances in which the
// general one's source of sampled rows and, for PLAIN blocks, the wrap of smooth windows are compiled out of every iteration.  Two 128-query
// tiles of a workgroup (d = 64) share their keys: PLAIN with both inside one key block (where the second tile is past the end, its
// waves work on row 0 and store nothing); the other forms have one.  SMOOTH against the general instance: 2 x 32 heads of 65536
// rows, d = 128, blocks of 512, the whole call 2897 -> 2820 us; d = 64, 32 of 36352 437 -> 428.
enum GatherForm { GENERAL = 0, PLAIN = 1, SMOOTH = 2 };

// Head dims below the built width D (NARROW kernels): a row holds fewer 16-byte pieces than its LDS slot.
// A lane whose piece lies past the end of the row fetches these zeros instead, so the tiles hold the rows
// zero-padded to D: zero columns change neither q.k nor the other columns of the output.
// Of the padded columns only the first DC (a multiple of 32) are computed with.
__device__ __attribute__((aligned(16))) const unsigned char ha_zero_piece[16] = {0};

template <bool NARROW>
__device__ __forceinline__ const unsigned char* piece_address(const unsigned char* base, int row, uint32_t stride_bytes,
                                                              uint32_t piece, int pieces_in_row) {
  const unsigned char* a = row_address(base, row, stride_bytes, piece << 4);
  if (NARROW && (int)piece >= pieces_in_row) a = ha_zero_piece;
  return a;
}

// Rows of segment `seg`: how many queries and keys it has and where they start in the query-side, key-side and
// out / lse tensors.
struct SegmentRows {
  int n_q, n_k;
  int64_t q_row, k_row, o_row;
};
template <bool GATHER>
__device__ __forceinline__ SegmentRows segment_rows(const ha_attn_kernel_params& p, int seg) {
  SegmentRows r;
  r.n_q = p.n_q;
  r.n_k = p.n_k;
  r.q_row = p.q_seg_off + (int64_t)seg * p.seg_stride;
  r.k_row = p.k_seg_off + (int64_t)seg * p.seg_stride;
  r.o_row = p.o_seg_off + (int64_t)seg * p.o_seg_stride;
  if (!GATHER && p.rag_levels >= 0) {
    // walk down from the whole sequence: where the segment starts and how many of its rows exist
    int start = 0, real = p.rag_n;
    for (int i = 0; i < p.rag_levels; ++i) {
      const int c = p.rag_half[i];
      if ((seg >> (p.rag_levels - 1 - i)) & 1) {
        start += c;
        real = max(real - c, 0);
      } else {
        real = min(real, c);
      }
    }
    r.o_row = r.q_row = r.k_row = start;
    r.n_q = r.n_k = real;
  }
  return r;
}

// FOLLOW (p.follow_max): the reference exponents follow the row maxima at every step of 32 keys, in exact causal single tiles in a
// sequence's first tile, gathered (plain or not, tiles of 128 queries) and at head dims above 64 without mask in a row's first p.follow_max chunks.  An
// instance of its own: as an argument's value it cost every pair of tiles 0.5 %.
template <typename T, int D, bool GATHER, bool CAUSAL, int FORM = GENERAL, bool NARROW = false, bool REWEIGHT = false,
          int DC = D, bool FOLLOW = false, int NB = WaveShape<D>::NB, int WAVES = WaveShape<D>::WAVES>
__global__ __launch_bounds__(64 * WAVES, D == 64 && NB == 1 ? 3 : 2) void ha_attn_fwd_kernel(const ha_attn_kernel_params p) {
#include "attn_fwd_body.inc"
}
// exact causal, with workgroups that hash and rank (place_ranking)
template <typename T, int D, bool GATHER, bool CAUSAL, int FORM = GENERAL, bool NARROW = false, bool REWEIGHT = false,
          int DC = D, bool FOLLOW = false, int NB = WaveShape<D>::NB, int WAVES = WaveShape<D>::WAVES>
__global__ __launch_bounds__(64 * WAVES, D == 64 && NB == 1 ? 3 : 2) void ha_attn_fwd_kernel(const ha_attn_kernel_params p,
                                                                                          const ha_rank_beside ranking) {
#define HA_WITH_RANKING
#include "attn_fwd_body.inc"
#undef HA_WITH_RANKING
}

#include "attn_fwd_split.inc"

namespace {

template <typename T, int D, bool GATHER, bool CAUSAL, int FORM = GENERAL, bool NARROW = false, bool REWEIGHT = false,
          int DC = D, bool FOLLOW = false, int NB = WaveShape<D>::NB, int WAVES = WaveShape<D>::WAVES>
int launch_one(const ha_attn_kernel_params& p, int grid, hipStream_t stream, const char* what) {
  void (*const kernel)(ha_attn_kernel_params) = ha_attn_fwd_kernel<T, D, GATHER, CAUSAL, FORM, NARROW, REWEIGHT, DC, FOLLOW, NB, WAVES>;
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(64 * WAVES), 0, stream, p);
  return ha_launch_status(what);
}

// exact causal, in instances of their own with ranking workgroups: the branch and the longer argument block cost every
// other launch 0.2 to 0.3 us
template <typename T, int D, bool NARROW, int DC, bool FOLLOW = false, int NB = WaveShape<D>::NB, int WAVES = WaveShape<D>::WAVES>
int launch_causal(const ha_attn_kernel_params& p, const ha_rank_beside* r, int grid, hipStream_t stream) {
  const char* const what = "ha_flash_attn_fwd";
  if (!r) return launch_one<T, D, false, true, GENERAL, NARROW, false, DC, FOLLOW, NB, WAVES>(p, grid, stream, what);
  void (*const kernel)(ha_attn_kernel_params, ha_rank_beside) =
      ha_attn_fwd_kernel<T, D, false, true, GENERAL, NARROW, false, DC, FOLLOW, NB, WAVES>;
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(64 * WAVES), 0, stream, p, *r);
  return ha_launch_status(what);
}

template <typename T, int D, bool GATHER, bool CAUSAL, bool NARROW, int DC>
int launch_split(const ha_attn_kernel_params& p, const ha_rank_beside* r, int grid, hipStream_t stream, const char* what) {
  if constexpr (CAUSAL) {
    if (r) {
      hipLaunchKernelGGL((ha_attn_fwd_split_kernel<T, D, GATHER, CAUSAL, NARROW, DC, ha_rank_beside>), dim3(grid),
                         dim3(SplitShape<D>::THREADS), 0, stream, p, *r);
      return ha_launch_status(what);
    }
  }
  hipLaunchKernelGGL((ha_attn_fwd_split_kernel<T, D, GATHER, CAUSAL, NARROW, DC>), dim3(grid), dim3(SplitShape<D>::THREADS), 0,
                     stream, p);
  return ha_launch_status(what);
}

// gathered launches in workgroups of 128 queries
template <typename T, int D, bool NARROW, int DC, bool FOLLOW = false>
int launch_gathered(const ha_attn_kernel_params& p, int grid, GatherForm form, hipStream_t stream) {
  const char* const what = "ha_block_attn_fwd";
  if (form == PLAIN) return launch_one<T, D, true, false, PLAIN, NARROW, false, DC, FOLLOW, 1>(p, grid, stream, what);
  if (form == SMOOTH) return launch_one<T, D, true, false, SMOOTH, NARROW, false, DC, FOLLOW, 1>(p, grid, stream, what);
  return launch_one<T, D, true, false, GENERAL, NARROW, false, DC, FOLLOW, 1>(p, grid, stream, what);
}

// Head dims below the built width.  At D = 128 the ones up to 96 (80 and 96 are models' head dims) compute with three
// quarters of the row: a quarter of the MFMAs and LDS operand reads and 30 to 40 registers less.  16 heads of 20479
// causal rows of d = 96: 546 -> 507 us (gathered level 87 -> 76, leaves 173 -> 151); 8 heads of 16384 rows without mask:
// 896 -> 791 us.
template <typename T, int D, int DC>
int launch_narrow(const ha_attn_kernel_params& p, const ha_rank_beside* r, int grid, bool gather, bool causal, GatherForm form, hipStream_t stream) {
  if (p.split_keys) {
    if (gather) return launch_split<T, D, true, false, true, DC>(p, r, grid, stream, "ha_block_attn_fwd");
    if (causal) return launch_split<T, D, false, true, true, DC>(p, r, grid, stream, "ha_flash_attn_fwd");
    return launch_split<T, D, false, false, true, DC>(p, r, grid, stream, "ha_flash_attn_fwd");
  }
  // the plain instance: d = 96, 16 heads of 32768 rows 205 -> 182 us, d = 40 98 -> 88
  if (gather && D == 64 && !p.small_tiles) return launch_one<T, D, true, false, PLAIN, true, false, DC>(p, grid, stream, "ha_block_attn_fwd");
  if constexpr (D == 128) {
    if (gather && p.follow_max) return launch_gathered<T, D, true, DC, true>(p, grid, form, stream);
  }
  if (gather) return launch_gathered<T, D, true, DC>(p, grid, form, stream);
  if constexpr (D == 128) {
    if (causal && p.large_tiles) return launch_causal<T, D, true, DC, true, 1, 8>(p, r, grid, stream);
  }
  if (causal && p.follow_max) return launch_causal<T, D, true, DC, true>(p, r, grid, stream);
  if (causal) return launch_causal<T, D, true, DC>(p, r, grid, stream);
  if constexpr (D == 128) {
    if (p.large_tiles) return launch_one<T, D, false, false, GENERAL, true, false, DC, false, 1, 8>(p, grid, stream, "ha_flash_attn_fwd");
    if (p.follow_max) return launch_one<T, D, false, false, GENERAL, true, false, DC, true>(p, grid, stream, "ha_flash_attn_fwd");
  }
  return launch_one<T, D, false, false, GENERAL, true, false, DC>(p, grid, stream, "ha_flash_attn_fwd");
}

template <typename T, int D>
int launch_variant(const ha_attn_kernel_params& p, const ha_rank_beside* r, int grid, bool gather, bool causal, bool reweight, hipStream_t stream) {
  if (gather && reweight)  // the entry point has checked that the head dims are the built ones
    return launch_one<T, D, true, false, GENERAL, false, true, D, false, 1>(p, grid, stream, "ha_block_attn_fwd");
  const GatherForm form = p.sampled_idx ? GENERAL : p.smooth ? SMOOTH : PLAIN;
  if (p.qk_pieces != D / 8 || p.v_pieces != D / 8) {
    if constexpr (D == 128) {
      if (p.qk_pieces <= 12 && p.v_pieces <= 12) return launch_narrow<T, D, 96>(p, r, grid, gather, causal, form, stream);
    }
    return launch_narrow<T, D, D>(p, r, grid, gather, causal, form, stream);
  }
  if (p.split_keys) {
    if (gather) return launch_split<T, D, true, false, false, D>(p, r, grid, stream, "ha_block_attn_fwd");
    if (causal) return launch_split<T, D, false, true, false, D>(p, r, grid, stream, "ha_flash_attn_fwd");
    return launch_split<T, D, false, false, false, D>(p, r, grid, stream, "ha_flash_attn_fwd");
  }
  if constexpr (D == 64) {
    if (gather && p.follow_max) return launch_gathered<T, D, false, D, true>(p, grid, form, stream);
    if (gather && !p.small_tiles) return launch_one<T, D, true, false, PLAIN>(p, grid, stream, "ha_block_attn_fwd");
    if (!gather && p.small_tiles) {
      if (causal) return launch_causal<T, D, false, D, true, 1>(p, r, grid, stream);
      return launch_one<T, D, false, false, GENERAL, false, false, D, false, 1>(p, grid, stream, "ha_flash_attn_fwd");
    }
  }
  if constexpr (D == 128) {
    if (gather && p.follow_max) return launch_gathered<T, D, false, D, true>(p, grid, form, stream);
    if (causal && p.large_tiles) return launch_causal<T, D, false, D, true, 1, 8>(p, r, grid, stream);
  }
  if (gather) return launch_gathered<T, D, false, D>(p, grid, form, stream);
  if (causal && p.follow_max) return launch_causal<T, D, false, D, true>(p, r, grid, stream);
  if (causal) return launch_causal<T, D, false, D>(p, r, grid, stream);
  if constexpr (D == 128) {
    if (p.large_tiles) return launch_one<T, D, false, false, GENERAL, false, false, D, false, 1, 8>(p, grid, stream, "ha_flash_attn_fwd");
    if (p.follow_max) return launch_one<T, D, false, false, GENERAL, false, false, D, true>(p, grid, stream, "ha_flash_attn_fwd");
  }
  return launch_one<T, D, false, false>(p, grid, stream, "ha_flash_attn_fwd");
}

}  // namespace

static ha_divisor make_divisor(int64_t y) {
  if (y < 1) y = 1;
  int s = 0;
  while ((int64_t(1) << s) < y) ++s;
  ha_divisor d;
  d.shift = 31 + s;
  d.magic = (uint32_t)((uint64_t(1) << d.shift) / (uint64_t)y + 1);
  return d;
}

// Whether a launch is better off with the keys of its query tiles split over waves (attn_fwd_split.inc): estimated
// times in us of the two kernels, from how many steps a workgroup takes and how many workgroups a CU has to take.  A step
// of the kernels that do not split is 64 keys, one of a split workgroup 64 queries x 128 keys.  What the estimates have to catch:
// - workgroups of 256 queries (d = 64): up to one per CU the launch takes as long as one of them; the first ones past 256 cost most
//   of a second round (48 causal heads of 3000 rows, 288 pairs: 97 us, 24 heads 66).  A CU works on two at a time, so beyond
//   that it is the CU's share that counts.
// - split workgroups: the longest one, or a CU's share of all; causal ones run longest first, so a CU's share ends with
//   short ones and some of the set-up hides behind other workgroups; at d = 128 equal ones go in whole rounds.
// d = 64: constants fitted to the kernels' times inside calls of the module, 645 launches (2 to 256
// heads, grouped and not, 300 to 4133 rows exact, 2048 to 16384 rows hashed).  Times whole | split in us, causal: 24 heads of 1000
// rows 31 | 13, of 2048 39 | 28, of 4096 72 | 72; 48 of 2048 41 | 45, of 4096 116 | 143; without mask 16 of 4096 rows
// 75 | 86.
// d = 128, causal: fitted to 93 launches each of 128 and of 96 columns (4 to 128 heads of 512 to 4096 rows), at which the choice
// is 0.2 % slower than the best one on average (worst: 40 heads of 512 rows, 96 columns 10 %, 24 of 700, 128 columns 8 %).  Single tiles of 128
// queries | split: 12 heads of 1000 rows 20.7 | 17.2, 24 of 1000 20.6 | 22.3, 48 25.1 | 37; 8 of 512 13.3 | 12.3, 96 columns 13.2 | 10.3;
// 16 of 2048 35.3 | 34.3, 24 38.4 | 50; 8 of 4096 65 | 51, 12 70 | 85.
// d = 128, without mask or gathered: the estimate of `whole` is that of 256-query tiles, which gathered launches no longer have and
// exact ones take in few places (large_tiles); tiles of 128 outrun it.  It stays the line because the split form is the closer one to
// float64 (four exact weights per row: 2 to 4 % for 256 to 1024 keys a row, 0.2 to 2 % above), and the launches that it gives to it lose little: 8 heads of 2048 rows, blocks and samples of 128 10.7 | 12.2,
// 256 14.5 | 14.5, 512 22.8 | 19.8; without mask 12 of 1000 19.8 | 17.1, 4 of 4096 57 | 44.  What it gives the split kernel beyond
// one round ha_attn_launch takes back.
//
// d = 64, tiles of 256 | 128 queries (`large`, `small`; 470 launches of 6 to 512 heads, 512 to 8192 rows, mean error 3 %; a choice that lost 2.5 % or more is not among them).  A
// workgroup of 128 queries takes half as long, a CU holds three, and ragged rows waste less; its waves read the keys
// for half as many queries, 10 % more time on a full chip.  Exact causal, us: 48 heads of 2048 rows 40.0 | 35.9, 32 of 3000 53.8 |
// 48.6, 64 of 1000 23.2 | 18.6, 24 of 4096 70.3 | 64.5, but 48 of 4096 113 | 115.5, 160 of 4096 341 | 376; without mask 48 of
// 2048 62 | 58, 64 of 2048 69 | 76 (what the split kernel takes from tiles of 256 without mask stays with it: the closer one to float64); whole calls with blocks and samples of 256: 16 heads of 2560 rows 24.6 | 23.7, 24 of
// 4096 37.0 | 36.0, 24 of 6144 54.5 | 51.2, 24 of 8192 58.3 | 59.4.
struct LaunchTimes {
  double whole, single, split;  // a tile per workgroup (exact causal: pairs of tiles), single causal tiles, the split kernel
  double large, small;          // d = 64: tiles of 256 and of 128 queries (exact causal: single ones)
  double split_rounds;          // the split kernel's with whole rounds of workgroups per CU
};
static LaunchTimes launch_times(const ha_attn_kernel_params& p, int width, bool gather, bool causal) {
  struct Fit {
    double step, pair, start, crowd, second, share, rest;    // 256-query tiles
    double split_step, split_start, set_up, share_up, hidden;  // split kernel; share_up: the set-up in a CU's share
  };
  const bool paired = causal && !gather;
  const bool columns_96 = p.qk_pieces <= 12 && p.v_pieces <= 12;
  const Fit f = width == 64 ? Fit{0.97, 4.4, 6.2, 0.08, 1.85, 0.94, 0.45, 0.56, 5.6, 4.3, 4.3, 0.34}
                : paired    ? (columns_96 ? Fit{0, 0, 0, 0, 0, 0, 0, 1.02, 4.0, 2.4, 4.9, 0.} : Fit{0, 0, 0, 0, 0, 0, 0, 1.07, 4.2, 3.5, 6.4, 0.})
                            : Fit{1.25, 2.0, 7.0, 0.37, 1.47, 1.58, 0.29, 1.23, 1.3, 5.4, 5.4, 0.22};
  const double cus = 256., vheads = (double)p.batch * p.heads * p.segs;
  const double tiles = (p.n_q + 255) / 256, split_tiles = (p.n_q + 63) / 64;
  const double keys = gather ? 128. * p.block_tiles + 64. * p.sample_chunks : p.n_k;

  LaunchTimes t;
  if (paired && width == 128) {
    // two workgroups of 128 queries per CU: the longest chain, slowed by its neighbour, or a CU's share of all
    const double tiles_128 = (p.n_q + 127) / 128, wgs = vheads * tiles_128 / cus;
    const double longest = 2. * tiles_128, beside = std::min(1., wgs / 2), share = wgs * (tiles_128 + 1);
    t.single = columns_96 ? 7.8 + std::max(0.638 * longest * (1 + 0.376 * beside), 0.748 * share + 2.57 * wgs)
                          : 7.65 + std::max(0.688 * longest * (1 + 0.478 * beside), 0.929 * share + 1.71 * wgs + 2.3);
    t.whole = t.single;  // pairs are for launches that are too large for the split kernel (single_tiles)
  } else {
    const double per_cu = vheads * (paired ? std::ceil(tiles / 2) : tiles) / cus;
    const double one = paired ? 4. * (tiles + 1) * f.step + f.pair : std::ceil(keys / 64.) * f.step;  // a workgroup
    double rounds;
    if (per_cu <= 1) rounds = 1 + f.crowd * per_cu;
    else if (width == 64) rounds = std::max(f.second, f.share * per_cu + f.rest);
    else rounds = f.second * std::ceil(per_cu);
    t.whole = t.single = f.start + (gather ? 3.5 : 0.) + one * rounds;  // gathered: a chain of row numbers, then rows
    if (paired) {
      // one tile per workgroup, longest first: the longest chain, slowed by its neighbours, or a CU's share of all
      const double longest = 4. * tiles, share = vheads * 2. * tiles * (tiles + 1) / cus, wgs = vheads * tiles / cus;
      t.single = f.start + std::max(f.step * (longest + 0.1 * share), 0.97 * share + 2. * wgs);
    }
  }

  t.large = t.small = 0;
  if (width == 64) {
    // start, a chunk of 64 keys, its slowdown by the neighbours; causal: a CU's share of chunks and of workgroups,
    // and what more than three of them cost (`less`: a CU holds three small ones); else a
    // round's chunks and what it costs beside them, in whole rounds while they are few
    struct TileFit {
      double start, chunk, crowd, share, less, per_wg;
    };
    auto time = [&](double rows, const TileFit& c) {
      const double count = std::ceil(p.n_q / rows), wgs = vheads * count / cus;
      if (paired) {
        const double longest = rows / 64 * count, share = wgs * (count + 1) * rows / 128;
        return c.start + std::max(c.chunk * (longest + c.crowd * share), c.share * share + c.per_wg * wgs + (wgs > 3 ? c.less : 0));
      }
      const double rounds = wgs <= 1 ? 1 + c.crowd * wgs : c.share * (wgs <= 6 ? std::ceil(wgs) : wgs + 0.3) - c.less;
      return c.start + (std::ceil(keys / 64.) * c.chunk + c.per_wg) * rounds;
    };
    t.large = time(256, paired ? TileFit{8.2, 0.783, 0.261, 0.912, 0., 2.2} : TileFit{5.85, 0.815, 0.156, 1.222, 0.33, 1.41});
    t.small = time(128, paired ? TileFit{7.2, 0.51, 0.29, 0.524, 1.5, 1.2} : TileFit{5.05, 0.542, 0.139, 1.005, 0.235, 1.1});
  }

  const double chain = std::ceil(keys / 128.), split_per_cu = vheads * split_tiles / cus;
  double all;
  if (paired) all = split_per_cu * (chain / 2 + 0.5 + f.share_up) - f.hidden * chain;
  else all = (width == 64 ? split_per_cu : std::ceil(split_per_cu)) * (chain + f.share_up);
  t.split = f.split_start + f.split_step * std::max(chain + f.set_up, all);
  t.split_rounds = f.split_start + f.split_step * std::ceil(split_per_cu) * (chain + f.set_up);
  return t;
}

// Whether exact causal attention takes one query tile per workgroup, longest first, instead of a pair of tiles.  Pairs
// leave CUs idle in a last round that is not full; single tiles fill it, but read a sequence's keys at times
// far apart, which costs where there are many rounds, and full rounds of pairs are as fast or faster.
// Times in us, pairs | single.  d = 64, 256-query pairs per CU in brackets: 48 heads of 2048 rows
// (0.75) 49.9 | 43.0, 80 (1.25) 74.1 | 58.1, 96 of 1024 (0.75) 32.8 | 26.8, 128 of 2048 (2) 82.9 | 81.2, 200 (3.1) 151 |
// 130, 256 (4) 170 | 175, 700 (11) 448 | 490, 2048 (32) 1292 | 1462.
// d = 128 (and 96): what a last round of pairs leaves idle against what reading the keys of many sequences at once costs, which
// grows with their number times the columns (fewer tiles in flight share a key's read).  Fitted to 450 launches (128 and 96 columns, 8 to 512
// heads, 512 to 11000 rows), 0.3 % slower than the better form on average (worst: 128 heads of 892 rows 9 %).  Rounds of 512 pairs of 128-query
// tiles in brackets: 24 of 2365 (0.47) 50.3 | 47.5, 80 of 2560 (1.56) 163 | 142, 88 of 2120 (1.55) 129 | 117, 112 of 2560 (2.19) 215 |
// 198, 200 of 892 (1.56) 71.4 | 63.0, 160 of 2572 (3.44) 321 | 309, 48 of 3000 (1.12) 148 | 123, but 256 of 1000 (2) 92 | 104, 288 of 768 (1.69) 72.9 |
// 84.5, 256 of 512 (1) 37.4 | 45.0, 112 of 4096 (3.5) 477 | 498, 144 of 4512 (5.06) 781 | 837, 256 of 3584 (7) 854 | 1076; 96 columns: 160 of 2560 (3.12)
// 257 | 236, 224 of 1403 (2.62) 140 | 121, 400 of 596 (2.34) 71.5 | 71.6.
// Rows of up to 128 are single tiles in any number, of up to 192 in less than 384: there the split kernel would be the faster one but for
// these tiles, and tiles without FOLLOW have 1.007 to 1.024 times its error, with it less (300 to 2048 sequences, normal and clustered).
// Split | pairs | single, us: 512 of 65 28.3 | 12.1 | 13.0, of 128 35.6 | 17.0 | 17.2, 320 of 150 26.0 | 20.4 | 21.3; 96 columns: 512 of 128 28.1 |
// 13.7 | 13.9.  From 384 on two rounds of pairs are closer to full (480 of 172, 80 columns 22 | 20.5 | 23.5, 1016 of 172 50.5 | 45.4 | 47.8).
// One round of sequences of 129 to 256 rows, which fill the chip with tiles that all follow, pays the most for it: up to 2 us against tiles of
// 256 without, 256 of 200 16.7 | 18.7, of 130 12.3 | 13.4 (large_tiles), 200 of 200 14.4 | 15.1, 96 columns 248 of 220 14.3 | 15.4.
static bool single_tiles(const ha_attn_kernel_params& p, int width) {
  const int64_t pair_rows = width == 64 ? 2 * WaveShape<64>::QUERIES : 2 * WaveShape<128>::QUERIES;
  const double vheads = (double)p.batch * p.heads * p.segs, pairs = vheads * ((p.n_q + pair_rows - 1) / pair_rows) / 256.;
  if (width == 64) return pairs <= 3.5;
  if (p.n_q <= 128 || (p.n_q <= 192 && vheads < 384)) return true;
  const double rounds = pairs / 2, columns = 8. * std::max(p.qk_pieces, p.v_pieces);
  return rounds <= 3.8 && vheads * columns <= 18000 + 30000 * (std::ceil(rounds) / rounds - 1);
}

// Whether exact attention at head dims above 64 takes workgroups of 8 waves, 256 queries, one per CU, instead of two of 128
// queries per CU.  Per CU both have 256 queries in flight, the larger ones read the keys once for all of them; the smaller ones fill a last
// round of up to half of the CUs' places in less time, waste less of a ragged end, and at many rounds run without waiting for each other.
// Without mask, 256 | 128 queries per workgroup in us, rounds of the chip in brackets (470 launches in all, the rule 0.4 % slower than the
// better form on average): 24 heads of 1298 rows (0.56 | 0.52) 35.8 | 38.0, 24 of 1500 42.1 | 44.4, 35 of 827 (0.55 | 0.48) 24.6 | 19.7, 45 of
// 2340 (1.76 | 1.67) 136 | 141, 25 of 7193 (2.83 | 2.78) 588 | 619, 73 of 2056 (2.57 | 2.42) 176 | 167, 90 of 3393 (4.92 | 4.75) 509 | 524,
// 122 of 1328 (2.86 | 2.62) 129 | 129, 368 of 412 (2.88 | 2.88) 56 | 54; 96 columns: 9 of 3915 (0.56 | 0.54) 72 | 87, 12 of 3458 72.8 | 79.6, 40 of 4332 (2.66)
// 301 | 321, 242 of 666 (2.84) 58 | 61, 620 of 387 (4.84) 74 | 72, 402 of 130 (1.57; three quarters of the queries exist) 18.8 | 19.9.
// Causal, single tiles, longest first: a launch works on the same tile of all sequences at a time, and the tiles of a sequence meet
// in one XCD's L2 only where the number of sequences is a multiple of the 8 XCDs (of 4: in two, of 2: in four).  With others the
// smaller workgroups, which read the keys twice as often, wait for them.  256 | 128 queries, us (370 launches; where the rule chooses 256, they
// are at most 1 % slower, on average 8 % faster): 127 heads of 1953 rows 150 | 177, 35 of 3574 121 | 139, 33 of 6382 339 | 396, 81 of 3581 271 |
// 319, 181 of 935 71 | 78, 66 of 2013 88 | 97, 50 of 5022 316 | 338, 156 of 2514 285 | 311, but 88 of 2071 (a multiple of 8) 128 | 112, 132 of 1621 124 | 123, 46 of 2861 119 | 113,
// 28 of 1185 30.9 | 24.5 (0.5 rounds), 141 of 795 (7 tiles of 128 in 4 of 256) 55.6 | 49.7; with 96 columns rarely (70 of 1873 74 | 71).  And up to one
// per CU where a quarter of a sequence's 256 queries does not exist: 248 of 150 13.7 | 15.4, 125 of 426 19.3 | 21.2, 96 columns 256 of 180 12.8 | 14.4.
static bool large_tiles(const ha_attn_kernel_params& p, bool causal) {
  const double vheads = (double)p.batch * p.heads * p.segs;
  const double rounds_256 = vheads * ((p.n_q + 255) / 256) / 256, rounds_128 = vheads * ((p.n_q + 127) / 128) / 512;
  const double rounds = std::ceil(rounds_128);
  const bool columns_96 = p.qk_pieces <= 12 && p.v_pieces <= 12;
  if (causal) {
    const int last = (p.n_q - 1) % 256 + 1;  // queries of the last tile
    if (rounds_256 > 0.8 && rounds_256 <= 1 && p.n_q <= 448 && last > 128 && last <= 192) return true;
    const int64_t seqs = (int64_t)p.batch * p.heads * p.segs;
    const double least = seqs % 2 ? 1.5 : seqs % 4 ? (seqs >= 64 ? 1.5 : 3.5) : 5;
    return !columns_96 && seqs % 8 != 0 && p.n_q >= 640 && rounds_128 >= least && rounds_256 <= 1.1 * rounds_128;
  }
  if (rounds_128 <= rounds - 0.5 || std::ceil(rounds_256) != rounds) return false;
  if (columns_96 && rounds <= 3 && p.n_q <= 192) return true;
  return rounds == 1 || (rounds <= 6 && p.n_q >= (columns_96 ? 200 : 500) * rounds);
}

// Where a grid of `tiles` workgroups of exact causal attention, `per_cu` of which a CU holds, has its ranking workgroups.  Behind the
// others where all of the grid is resident at once, and in launches of many rounds: there the order of the tiles over the CUs stays what
// it is without them (the launch grows by about what hashing takes alone all the same: unit_ranking.h).  Else in front: a ranking workgroup takes about as
// long as a short tile, and behind one or two rounds of tiles it would be what the launch ends with.  Whole calls, hash and rank
// launches | in front | behind, us (36 drawn calls and 4 others, 1.035 times faster in the geometric mean in front, 1.022 behind, none slower
// by this rule): 12 heads of 7167 rows (672 tiles on 768 places) 78.0 | 70.7 | 65.5, 8 of 9728 85.9 | 80.0 | 74.6; 24 of 4096 (768 on 768)
// 63.3 | 56.8 | 59.8, 12 of 14335, d = 96 (2.6 rounds) 272 | 260 | 282, 32 of 11520, d = 128 (3) 558 | 553 | 579; pairs of tiles, d = 64: 16 of
// 29696 (2) 380 | 371 | 360, 24 of 29184 (3) 848 | 830 | 817; d = 128, 16 of 77824 (10) 2010 | 1998 | 1969.
// Spread between the tiles of launches of many rounds, a group after every few groups of tiles, they cost the tiles more than hashing beside them
// hides, behind | spread: 4 heads of 131072 474 | 498 us, 8 of 65536 422 | 443, d = 96, 16 of 20479 364 | 371, 32 of 131072 3900 | 3910.
static int64_t place_ranking(ha_rank_beside& a, int64_t tiles, int per_cu, bool pairs_64) {
  const int64_t groups = (tiles + NUM_XCD - 1) / NUM_XCD, places = 256 * per_cu;
  a.groups = (a.units + NUM_XCD - 1) / NUM_XCD;
  const bool behind = (groups + a.groups) * NUM_XCD <= places || pairs_64 || tiles >= 4 * places;
  a.first_group = behind ? (int)groups : 0;
  a.tiles = (int)tiles;
  return (groups + a.groups) * NUM_XCD;
}

int ha_attn_launch(const ha_attn_kernel_params& params, int d, int dv, int dtype, bool gather, bool causal,
                   bool reweight, hipStream_t stream, const ha_rank_beside* ranking) {
  ha_attn_kernel_params p = params;
  // the kernels are built for rows of 64 and 128 elements; other head dims (multiples of 8) run in the
  // next width with the missing pieces of every row read as zeros
  const int width = d <= 64 && dv <= 64 ? 64 : 128;
  p.qk_pieces = d / 8;
  p.v_pieces = dv / 8;
  const bool single = causal && !gather && single_tiles(p, width);
  const bool plain = !p.smooth && !p.sampled_idx && p.block_tiles % 2 == 0;
  const bool full_rows = p.qk_pieces == width / 8 && p.v_pieces == width / 8;
  const LaunchTimes t = launch_times(p, width, gather, causal);
  const char* split_env = getenv("HA_SPLIT");  // measurement aid: 1 forces the split kernel, 0 the other
  p.split_keys = !reweight && (split_env ? atoi(split_env) != 0 : t.split < (single ? t.single : t.whole));
  // Head dims up to 64, tiles of 128 queries: gathered launches that are not plain always, since two tiles of 128 share neither
  // their window nor a block of 128 (a workgroup of 256 queries went through what either has, 1.05 to 1.2 times the time from 4
  // heads of 4096 rows to 128 of 32768, smooth blocks of 512 0.99 to 1.07); others of full rows by the estimates.
  // Gathered ones take the place of the split kernel where that has more workgroups than CUs.  It is the closer one to float64, so the
  // exponents follow the row maxima in half of the chunks: 0.97 to 0.99 of its error with blocks and samples of 128 and 256
  // (without 1.01 and more), 12 heads of 2560 rows, blocks of 128 20.9 -> 19.7 us, 256 23.3 -> 22.4, 12 of 3072 25.8 -> 22.7
  // and 29.1 -> 26.2.  With 1024 keys a row the half costs what the tiles gain.
  p.small_tiles = p.large_tiles = p.follow_max = 0;
  const bool choice = width == 64 && full_rows && !reweight;
  const int chunks = 2 * p.block_tiles + p.sample_chunks;  // gathered: of a row's keys
  if (choice && gather && p.split_keys && !split_env && chunks <= 8 && t.small + 1.5 < t.split_rounds) {
    p.split_keys = 0;
    p.small_tiles = 1;
    p.follow_max = (chunks + 1) / 2;
  } else if (width == 64 && gather && (!plain || reweight)) {
    p.small_tiles = !p.split_keys;
  } else if (choice && causal && !gather) {
    p.small_tiles = single && !split_env && 1.01 * t.small < std::min(t.large, t.split);
    if (p.small_tiles) p.split_keys = 0;
  } else if (choice && !p.split_keys) {
    p.small_tiles = 1.02 * t.small < t.large;
  } else if (width == 128 && !p.split_keys && !gather && (single || !causal)) {
    p.large_tiles = large_tiles(p, causal);
  } else if (width == 128 && p.split_keys && !split_env && (gather || !causal)) {
    // Head dims above 64, exact without mask and gathered: split workgroups go in whole rounds, and from the second on tiles of 128
    // queries are faster, but for tiles that just miss one per CU against two rounds (24 heads of 1300 rows 40.7 us, split
    // 38.7).  The split form is the closer one to float64, so the exponents follow the row maxima: without mask in an eighth of
    // the chunks, at least four (half of fewer than eight), 0.98 to 0.998 of its error from 520 to 4096 keys on normal and on
    // clustered rows (1.001 to 1.015 without) for 4 to 12 % of the tiles' time; gathered in five eighths (1024 keys a row: 0.975 to 0.998, in half 0.98 to
    // 1.002, without 1.04).  Split -> tiles, us, without mask: 16 heads of 2048 rows 53 -> 43, 8 of 3000 65 -> 54, 24 of 2676 122 -> 91, 96
    // columns 48 -> 40, 59 -> 49, 110 -> 78; blocks and samples of 512: 12 heads of 2688 rows 50 -> 42, 24 87 -> 62, 96 columns 44 -> 37, 78 -> 54.
    const int64_t vheads = (int64_t)p.batch * p.heads * p.segs;
    const int64_t rounds = (vheads * ((p.n_q + 63) / 64) + 255) / 256, tiles = vheads * ((p.n_q + 127) / 128);
    if (rounds > 2 || (rounds == 2 && tiles <= 256)) {
      const int exact_chunks = (p.n_k + 63) / 64;
      p.split_keys = 0;
      p.follow_max = gather ? (5 * chunks + 7) / 8 : std::max(std::min(4, (exact_chunks + 1) / 2), 1 + exact_chunks / 8);
    }
  }
  const int tile_rows = p.large_tiles || (width == 64 && !p.small_tiles) ? 256 : 128;
  int64_t qtiles = (p.n_q + tile_rows - 1) / tile_rows;
  if (causal && !gather && !single) qtiles = (qtiles + 1) / 2;  // one workgroup per pair of tiles
  if (p.split_keys) qtiles = (p.n_q + 63) / 64;
  // causal launches of more split workgroups than CUs run longest first: tile number before sequence number
  if (p.split_keys && causal && !gather && qtiles * p.batch * p.heads * p.segs > 256) p.split_keys = 2;
  p.single = single && !p.split_keys;
  if (p.single) p.follow_max = width == 128 || t.split < t.whole;
  p.div_qtiles = make_divisor(p.split_keys == 2 || p.single ? (int64_t)p.batch * p.heads * p.segs : qtiles);
  p.div_segs = make_divisor(p.segs);
  p.div_heads = make_divisor(p.heads);
  p.div_kv_heads = make_divisor(p.heads / p.kv_group);
  p.div_kv_group = make_divisor(p.kv_group);
  p.div_block_tiles = make_divisor(p.block_tiles);
  int64_t grid = qtiles * p.batch * p.heads * p.segs;
  ha_rank_beside beside;
  if (ranking) {
    beside = *ranking;
    ranking = &beside;
    const int per_cu = p.split_keys ? (width == 64 ? 2 : 1) : p.large_tiles ? 1 : p.small_tiles ? 3 : 2;
    grid = place_ranking(beside, grid, per_cu, width == 64 && !p.single && !p.split_keys);
  }
  if (grid <= 0 || grid >= (1ll << 31)) return ha_fail(HA_ERR_SHAPE, "attention: grid of %lld workgroups", (long long)grid);
  if (dtype == HA_F16) {
    if (width == 64) return launch_variant<f16_t, 64>(p, ranking, (int)grid, gather, causal, reweight, stream);
    return launch_variant<f16_t, 128>(p, ranking, (int)grid, gather, causal, reweight, stream);
  }
  if (width == 64) return launch_variant<bf16_t, 64>(p, ranking, (int)grid, gather, causal, reweight, stream);
  return launch_variant<bf16_t, 128>(p, ranking, (int)grid, gather, causal, reweight, stream);
}
