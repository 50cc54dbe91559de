// Backward of the sorted blocks and the sampled keys in ONE kernel: plain blocks of 256 at head dim 64, as many key/value
// heads as query heads (the three passes of attn_bwd.hip serve everything else; see ha_block_bwd_fused_takes).
//
// The passes gather a level's rows three times (4.0 GB at 24 heads of 65536 rows with gradients added to; dq 447 us, dk/dv of
// the blocks 403, of the sampled keys 229) and compute the scores twice (7 products per pair).  Here a workgroup gathers the
// q, k, v, dO, O rows of a block of 256 queries and 256 keys once, computes every score once (5 products) and leaves dq, dk,
// dv of the block and its share of the sampled keys' sums: 3.4 GB, 735 to 766 us in the same launch (without adding, 24 heads
// of 16384, the whole call: 269 -> 215 us).  What bounds it now: not the board's power limit (2.18 to 2.39 GHz, matrix pipe busy 0.33 of
// the time, 0.37 where nothing is added to); of a block's 65k cycles (57k where nothing is added to) 43k are the steps, bound by the LDS (1750 of a step's 2700 cycles), the others the ends
// of its phases, where every wave does the same memory and vector work with one workgroup per CU and nothing beside it.
//
// A workgroup: 8 waves, a run of consecutive blocks of one (head, segment).  A block has a phase for its own keys and one
// per 256 sampled keys.  In a phase a wave keeps 32 keys (k, v rows as MFMA B operands, sums of dK^T, dV^T in registers) and
// goes through the block's queries in 8 steps of 32, their q and dO rows in LDS for the whole block (64 KB: 256 queries are
// what fits).  dS of a step, 32 queries x 256 keys, goes through LDS once; of dq^T = sum K^T dS^T a wave sums 16 elements of
// the head dim of 16 queries of every step over all keys.  All sums of a block are complete in registers: 64 (dk, dv) and 32
// (dq) of them.  The sampled keys' sums, 64 KB per tensor and phase, stay in the registers over two blocks in a row and
// else wait in memory of the workgroup's own, in the order of its registers, until ha_bwd_add_samples_kernel adds up the workgroups' shares.
// (Added to one array with atomics, each time, they took 10 to 16 thousand cycles of every second block, and a launch to
// clear it: 24 heads of 16384 rows 225 -> 215 us the call, of 4096 74 -> 64, 8 of 8192 67 -> 50, 24 of 65536 745 -> 735, with 512 samples 1148 -> 1099.)
// The next block's rows come in while this one is worked on: q and dO rows into a step's place once the step is done for the
// last time, k rows into an LDS stage, v rows through registers, O rows (for D) four queries of a step per wave.
#include "ha_common.h"
#include "attn_tiles.h"
#include "attn_bwd_tiles.h"
#include "attn_bwd.h"

#include <algorithm>
#include <type_traits>

namespace {

constexpr int FUSED_WAVES = 8, FUSED_THREADS = 64 * FUSED_WAVES;
constexpr int FUSED_ROWS = 256;  // queries, and keys of a phase, per workgroup
constexpr int FD = 64;           // head dim
constexpr int FUSED_MAX_SAMPLES = 1024;  // their row numbers are kept in LDS
constexpr int STEPS = FUSED_ROWS / 32;

template <typename T>
struct Mfma16;
template <>
struct Mfma16<f16_t> {
  static __device__ __forceinline__ f32x4 run(f16x8 a, f16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }
};
template <>
struct Mfma16<bf16_t> {
  static __device__ __forceinline__ f32x4 run(bf16x8 a, bf16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
};

template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}

// LDS, by address: q rows (4 KB) and dO rows (4 KB) of the eight steps; dS of three steps, [key][query of the step]; the k
// rows of a phase; -L / scale and -D of a block's queries and the next one's; query and key rows of a block and the next
// one; rows of the sampled keys.  As numbers, so that all but a few of the loop's addresses are a register and an offset
// in the instruction.
constexpr uint32_t TILES = 0, DS = TILES + STEPS * 8192, KEYS = DS + 3 * 16384, LSE = KEYS + 32768, DELTA = LSE + 2 * FUSED_ROWS * 4,
                   ROWS = DELTA + 2 * FUSED_ROWS * 4, SAMPLE_ROWS = ROWS + 4 * FUSED_ROWS * 4, LDS_BYTES = SAMPLE_ROWS + FUSED_MAX_SAMPLES * 4;
static_assert(LDS_BYTES <= 163840, "one workgroup per CU");

// SHORT_O: O's rows are shorter than dO's (p.out_last), an instance of its own: as a clamp in every call 0.4 % of the kernel
template <typename T, bool ACC, bool SHORT_O>
__global__ __launch_bounds__(FUSED_THREADS, 2) void ha_block_bwd_fused_kernel(const ha_attn_bwd_params p) {
  ha_load_arguments<(int)sizeof(ha_attn_bwd_params)>();
  typedef typename ElemTraits<T>::vec8 vec8;
  typedef typename ElemTraits<T>::vec4 vec4;
  constexpr int KSTEPS = FD / 16;
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds_block[];  // LDS_BYTES, from address 0 on
  (void)lds_block;
  const uint32_t tid = threadIdx.x, hi = (tid >> 5) & 1, col = tid & 31;
  uint32_t lane = tid & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  // ---- which run of blocks ----
  const int n = p.n_q, blocks = (n + FUSED_ROWS - 1) / FUSED_ROWS;
  const int runs = (blocks + p.run_blocks - 1) / p.run_blocks;
  const int id = xcd_contiguous_id(blockIdx.x, gridDim.x);
  const int vseq = id / runs, run = id - vseq * runs;
  const int seg = vseq % p.segs, bh = vseq / p.segs, b = bh / p.heads, h = bh - b * p.heads;
  const int first_block = run * p.run_blocks, end_block = min(first_block + p.run_blocks, blocks);
  const int n_phases = 1 + p.sample_size / FUSED_ROWS;

  const int64_t q_row0 = p.q_seg_off + (int64_t)seg * p.seg_stride, k_row0 = p.k_seg_off + (int64_t)seg * p.seg_stride;
  const int64_t o_row0 = p.o_seg_off + (int64_t)seg * p.o_seg_stride;
  const unsigned char* const qb = (const unsigned char*)((const T*)p.q + b * p.q_sb + h * p.q_sh + q_row0 * p.q_sn);
  const unsigned char* const dob = (const unsigned char*)((const T*)p.dout + b * p.do_sb + h * p.do_sh + q_row0 * p.do_sn);
  const unsigned char* const kb = (const unsigned char*)((const T*)p.k + b * p.k_sb + h * p.k_sh + k_row0 * p.k_sn);
  const unsigned char* const vb = (const unsigned char*)((const T*)p.v + b * p.v_sb + h * p.v_sh + k_row0 * p.v_sn);
  const unsigned char* const ob = (const unsigned char*)((const T*)p.out + b * p.o_sb + h * p.o_sh + o_row0 * p.o_sn);
  const float* const lseb = p.lse + b * p.lse_sb + h * p.lse_sh + o_row0;
  unsigned char* const dqb = (unsigned char*)((T*)p.dq + b * p.dq_sb + h * p.dq_sh + q_row0 * p.dq_sn);
  unsigned char* const dkb = (unsigned char*)((T*)p.dk + b * p.dk_sb + h * p.dk_sh + k_row0 * p.dk_sn);
  unsigned char* const dvb = (unsigned char*)((T*)p.dv + b * p.dv_sb + h * p.dv_sh + k_row0 * p.dv_sn);
  const uint32_t q_rb = (uint32_t)p.q_sn * 2, k_rb = (uint32_t)p.k_sn * 2, v_rb = (uint32_t)p.v_sn * 2,
                 do_rb = (uint32_t)p.do_sn * 2, o_rb = (uint32_t)p.o_sn * 2, dq_rb = (uint32_t)p.dq_sn * 2,
                 dk_rb = (uint32_t)p.dk_sn * 2, dv_rb = (uint32_t)p.dv_sn * 2;
  // the workgroup's own sums of the sampled keys in memory: [256 keys][wave][quarter of a sum's registers][lane], 16 bytes each
  const int64_t sums0 = (((((int64_t)b * p.heads + h) * p.segs + seg) * runs + run) * p.sample_size + wave * 32) * FD;

  // ---- row numbers: of a block and the next one, of the sampled keys ----
  const int idx_shift = p.idx64 ? 3 : 2;
  // threads 0..255 fetch query rows, 256..511 key rows
  const unsigned char* const idx_b =
      wave < 4 ? (const unsigned char*)p.q_idx + ((b * p.qi_sb + h * p.qi_sh + (int64_t)seg * n * p.qi_sn) << idx_shift)
               : (const unsigned char*)p.k_idx + ((b * p.ki_sb + h * p.ki_sh + (int64_t)seg * n * p.ki_sn) << idx_shift);
  const uint32_t idx_rb = (uint32_t)(wave < 4 ? p.qi_sn : p.ki_sn) << idx_shift;
  auto opaque_lane = [&]() -> uint32_t {  // offsets made from it are not kept in registers across the loop
    asm volatile("" : "+v"(lane));
    return lane;
  };
  auto fetch_row = [&](int bl) -> int {
    const int pos = min(bl * FUSED_ROWS + (int)((wave & 3) * 64 + opaque_lane()), n - 1);
    return *reinterpret_cast<const int*>(row_address(idx_b, pos, idx_rb, 0));
  };
  auto rows_of = [&](int bl) -> uint32_t { return ROWS + (bl & 1) * (2 * FUSED_ROWS * 4); };  // query rows, then key rows
  auto keep_row = [&](int bl, int row) { lds_put<int>(rows_of(bl) + (wave * 64 + opaque_lane()) * 4, row); };
  auto query_row = [&](int bl, uint32_t r) -> uint32_t { return lds_get<int>(rows_of(bl) + r * 4); };
  auto key_row = [&](int bl, int ph, uint32_t r) -> uint32_t {
    return lds_get<int>((ph == 0 ? rows_of(bl) + FUSED_ROWS * 4 : SAMPLE_ROWS + (ph - 1) * (FUSED_ROWS * 4)) + r * 4);
  };

  // ---- loads ----
  // q or dO rows of step u: waves 0..3 eight q rows each, waves 4..7 eight dO rows
  const unsigned char* const fill_b = wave < 4 ? qb : dob;
  const uint32_t fill_rb = wave < 4 ? q_rb : do_rb;
  const uint32_t fill_row_at = ((wave & 3) * 8 + lane / 8) * 4, stats_row_at = (wave * 4 + lane / 16) * 4;  // in a step's rows
  const uint32_t fill_piece = ((lane & 7) ^ bwd_swizzle<FD>((wave & 3) * 8 + lane / 8)) << 4;
  auto fill_tile = [&](int u, uint32_t row) { load_to_lds(fill_b, __umul24(row, fill_rb) + fill_piece, TILES + u * 8192 + wave * 1024); };
  // the wave's 32 k rows of a phase
  auto stage_keys = [&](int bl, int ph) {
    const uint32_t ln = opaque_lane();
    uint32_t rows[4];
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) rows[j] = key_row(bl, ph, wave * 32 + j * 8 + ln / 8);
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j)
      load_to_lds(kb, __umul24(rows[j], k_rb) + (((ln & 7) ^ bwd_swizzle<FD>(j * 8 + ln / 8)) << 4), KEYS + wave * 4096 + j * 1024);
  };
  // -L / scale and -D of a block's queries, four queries of 32 per wave: loaded, and a step later put in place.
  // A query past the end has L = inf: its weights are zero.
  struct Stats {
    vec4 o, g;
    float l;
  };
  auto load_stats = [&](uint32_t row) -> Stats {
    const uint32_t piece = (opaque_lane() & 15) * 8;
    Stats st;
    // the last 8 bytes of a short row stand in for those that are missing, which meet zeros of dO
    st.o = *reinterpret_cast<const vec4*>(row_address(ob, row, o_rb, SHORT_O ? min(piece, (uint32_t)p.out_last * 16 + 8) : piece));
    st.g = *reinterpret_cast<const vec4*>(row_address(dob, row, do_rb, piece));
    st.l = lseb[row];
    return st;
  };
  auto keep_stats = [&](int bl, int u, const Stats& st) {
    const uint32_t ln = opaque_lane(), r = u * 32 + wave * 4 + ln / 16;
    float d = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) d = __builtin_fmaf((float)st.o[e], (float)st.g[e], d);
    d += dpp<0xB1>(d);   // lane ^ 1
    d += dpp<0x4E>(d);   // lane ^ 2
    d += dpp<0x141>(d);  // the other four lanes of eight
    d += dpp<0x140>(d);  // the other eight lanes of sixteen
    if ((ln & 15) == 0) {
      const uint32_t at = LSE + (bl & 1) * (FUSED_ROWS * 4) + r * 4;
      lds_put<float>(at, (bl * FUSED_ROWS + (int)r < n ? st.l : __builtin_inff()) * p.neg_inv_scale);
      lds_put<float>(at + (DELTA - LSE), -d);
    }
  };

  // ---- LDS addresses of the operand reads: of step 0 ----
  uint32_t row_at = TILES + bwd_tile_offset<FD>(col, hi), tr_at;
  {  // 32x32 operands: as in attn_bwd_tile.inc
    const uint32_t g = lane >> 4, sl = lane & 15, key = (g >> 1) * 4 + (sl >> 2), w = sl & 3;
    tr_at = TILES + bwd_tile_offset<FD>(key, (g & 1) * 2 + (w >> 1)) + (w & 1) * 8;  // rows 8 further on: 1024 further, another swizzle
  }
  // dS of a step is [256 keys][32 queries]: a lane's 16 queries (8g + 4 hi + e) side by side, the 16-byte pieces of a row
  // XOR-ed with two bits of the key number
  uint32_t ds_write = DS + (wave * 32 + col) * 64 + (((2 * hi) ^ ((col >> 2) & 3)) << 4);
  const uint32_t qw = wave & 1, dw = wave >> 1;  // the 16 queries of a step, the 16 elements of the head dim whose dq the wave sums
  uint32_t ds_at;
  {
    const uint32_t g = lane >> 4, sl = lane & 15, key = 8 * g + (sl >> 2), w = sl & 3, piece = 2 * qw + (w >> 1);
    ds_at = DS + key * 64 + ((piece ^ ((key >> 2) & 3)) << 4) + (w & 1) * 8;  // keys 4 further on: 256 further, another swizzle
  }

  // ---- first block ----
  keep_row(first_block, fetch_row(first_block));
  for (int i = tid; i < p.sample_size; i += FUSED_THREADS)
    lds_put<int>(SAMPLE_ROWS + i * 4, p.sampled_idx ? ha_load_idx(p.sampled_idx, b * p.si_sb + h * p.si_sh + i, p.idx64) : i);
  __syncthreads();
  // v rows of the wave's keys: loaded whole rows at a time, then turned through 4 KB of LDS into the products' operands
  vec8 x2f[KSTEPS];
  auto load_v = [&](int bl, int ph) {
    const uint32_t ln = opaque_lane();
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j)
      x2f[j] = *reinterpret_cast<const vec8*>(row_address(vb, key_row(bl, ph, wave * 32 + j * 8 + ln / 8), v_rb, (ln & 7) * 16));
  };
  const uint32_t turn = DS + (wave < 4 ? 0 : 2 * 16384) + (wave & 3) * 4096;  // dq of a phase's last step is read from between
  auto turn_v = [&]() {
    const uint32_t ln = opaque_lane();
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) lds_put<vec8>(turn + (j * 8 + ln / 8) * 128 + (((ln & 7) ^ bwd_swizzle<FD>(j * 8 + ln / 8)) << 4), x2f[j]);
    wave_lds_order();
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) x2f[ks] = lds_get<vec8>(turn + (row_at ^ (ks << 5)));
    wave_lds_order();
  };
  stage_keys(first_block, 0);
#pragma unroll
  for (int u = 0; u < STEPS; ++u) fill_tile(u, lds_get<int>(rows_of(first_block) + fill_row_at + u * 128));
  load_v(first_block, 0);
  Stats first_stats[STEPS];
#pragma unroll
  for (int u = 0; u < STEPS; ++u) first_stats[u] = load_stats(lds_get<int>(rows_of(first_block) + stats_row_at + u * 128));
#pragma unroll
  for (int u = 0; u < STEPS; ++u) keep_stats(first_block, u, first_stats[u]);
  int row_ahead = fetch_row(first_block + 1);  // of the block after the next one, from the first block on
  turn_v();
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)

  f32x16 acc1[2], acc2[2];  // dK^T, dV^T of the wave's keys
  for (int bl = first_block; bl < end_block; ++bl) {
    const int n_waves = min(n - bl * FUSED_ROWS, FUSED_ROWS) / 32;  // with rows that exist; 4 or 8: n is a multiple of 128
    const bool more_blocks = bl + 1 < end_block;
    keep_row(bl + 1, row_ahead);
    row_ahead = fetch_row(bl + 2);
    f32x4 dq[STEPS];
#pragma unroll
    for (int u = 0; u < STEPS; ++u) dq[u] = f32x4{0.f, 0.f, 0.f, 0.f};
    // every other block goes through its phases backwards: two blocks in a row then share the sums of their sampled keys
    const bool backwards = (bl - first_block) & 1;
    for (int i_ph = 0; i_ph < n_phases; ++i_ph) {
      const int ph = backwards ? n_phases - 1 - i_ph : i_ph;
      const bool last_phase = i_ph + 1 == n_phases, more = !last_phase || more_blocks;
      const int next_bl = last_phase ? bl + 1 : bl, next_ph = last_phase ? ph : backwards ? ph - 1 : ph + 1;
      // ---- the phase's keys ----
      lds_barrier();
      vec8 x1f[KSTEPS], kt[STEPS];  // k rows of the wave's keys; 16 elements of every key's row, for dq
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ++ks) x1f[ks] = lds_get<vec8>(KEYS - TILES + wave * 4096 + (row_at ^ (ks << 5)));
      {
        const uint32_t ln = opaque_lane(), g = ln >> 4, sl = ln & 15, key = 8 * g + (sl >> 2), w = sl & 3;
        const uint32_t lo = KEYS + bwd_tile_offset<FD>(key, 2 * dw + (w >> 1)) + (w & 1) * 8, hi4 = KEYS + bwd_tile_offset<FD>(key + 4, 2 * dw + (w >> 1)) + (w & 1) * 8;
#pragma unroll
        for (int ks = 0; ks < STEPS; ++ks) kt[ks] = lds_get_tr<T>(lo + ks * 4096, hi4 + ks * 4096);
        if (ph == 0 && n_waves < FUSED_WAVES) {  // keys that do not exist take no part in dq
#pragma unroll
          for (int ks = STEPS / 2; ks < STEPS; ++ks) kt[ks] = vec8{};
        }
      }
      // Sums of a phase: of the block's own keys from zero; of sampled keys as the block before left them in registers
      // (a backward block's first phase), else as the last block left them in memory
      if (ph == 0 || bl == first_block) {
#pragma unroll
        for (int d2 = 0; d2 < 2; ++d2)
#pragma unroll
          for (int i = 0; i < 16; ++i) acc1[d2][i] = acc2[d2][i] = 0.f;
      } else if (i_ph > 0) {
        const int64_t at = sums0 + (int64_t)(ph - 1) * FUSED_ROWS * FD + opaque_lane() * 4;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const f32x4 a1 = *reinterpret_cast<const f32x4*>(p.dk32 + at + i * 256), a2 = *reinterpret_cast<const f32x4*>(p.dv32 + at + i * 256);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            acc1[i >> 2][(i & 3) * 4 + e] = a1[e];
            acc2[i >> 2][(i & 3) * 4 + e] = a2[e];
          }
        }
      }

      // ---- 32 queries a step ----
      f32x16 s, dp;
      vec8 rq[KSTEPS], rg[KSTEPS];   // q and dO rows of a step
      uint32_t stats_at = LSE + (bl & 1) * (FUSED_ROWS * 4) + hi * 16;
      const uint32_t next_rows = rows_of(bl + 1);
      auto read_statistics = [&](int u, int g) {
        const f32x4 l = lds_get<f32x4>(stats_at + u * 128 + g * 32), nd = lds_get<f32x4>(stats_at + (DELTA - LSE) + u * 128 + g * 32);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          s[g * 4 + e] = l[e];
          dp[g * 4 + e] = nd[e];
        }
      };
      Stats st = {};
      vec8 old1[4], old2[4], old3[4];  // what the call adds to: rows of dk, dv (blocks), of dq (last phase)
#pragma unroll
      for (int j = 0; j < 4; ++j) old1[j] = old2[j] = old3[j] = vec8{};
      auto load_old = [&](vec8 (&old)[4], const unsigned char* base, uint32_t rb, uint32_t list) {
        const uint32_t ln = opaque_lane();
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) {
          const uint32_t row = query_row(bl, list + wave * 32 + j * 8 + ln / 8);
          old[j] = *reinterpret_cast<const vec8*>(row_address(base, row, rb, (ln & 7) * 16));
        }
      };
      vec8 pn[2], dsn[2], tq[2][2], tg[2][2];
      // the operands' addresses: not known here, so that a step's offset stays in the instructions and what an address and
      // an offset add up to is not kept in registers of its own
      auto opaque_addresses = [&]() {
        asm volatile("" : "+v"(row_at), "+v"(tr_at), "+v"(ds_write), "+v"(ds_at), "+v"(stats_at));
      };
      // P and dS of step u, dS into LDS; what the products of the step need is read
      auto weights = [&](int u) {
        opaque_addresses();
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            const float pv = __builtin_amdgcn_exp2f(s[kk * 8 + i] * p.scale_log2);
            pn[kk][i] = (T)pv;
            dsn[kk][i] = (T)(pv * dp[kk * 8 + i]);
          }
#pragma unroll
          for (int d2 = 0; d2 < 2; ++d2) {
            const uint32_t at = u * 8192 + kk * 16 * FD * 2;
            const uint32_t lo = tr_at ^ (d2 << 6), hi8 = (tr_at ^ (d2 << 6) ^ 16) + 1024;
            tq[kk][d2] = lds_get_tr<T>(lo + at, hi8 + at);
            tg[kk][d2] = lds_get_tr<T>(lo + at + 4096, hi8 + at + 4096);
          }
          lds_put<vec8>((ds_write ^ (kk << 4)) + u % 3 * 16384, dsn[kk]);
          asm volatile("" : "+v"(pn[kk]), "+v"(dsn[kk]));  // rounded here, not behind a branch
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x400, 1, 0);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      };
      vec8 rs[STEPS];
      auto read_ds = [&](int u, int ks) {  // of 32 keys
        rs[ks] = lds_get_tr<T>(ds_at + u % 3 * 16384 + ks * 2048, (ds_at ^ 16) + 256 + u % 3 * 16384 + ks * 2048);
      };
      auto add_dq = [&](int u, int ks) { dq[u] = Mfma16<T>::run(kt[ks], rs[ks], dq[u]); };
      auto add_dkv = [&](int kk, int which) {  // four products
        if (which & 1) acc2[which >> 1] = Mfma<T>::run(tg[kk][which >> 1], pn[kk], acc2[which >> 1]);
        else acc1[which >> 1] = Mfma<T>::run(tq[kk][which >> 1], dsn[kk], acc1[which >> 1]);
      };
      auto read_rows = [&](int u, int ks) {
        rq[ks] = lds_get<vec8>((row_at ^ (ks << 5)) + u * 8192);
        rg[ks] = lds_get<vec8>((row_at ^ (ks << 5)) + u * 8192 + 4096);
      };
      auto add_scores = [&]() {
#pragma unroll
        for (int ks = 0; ks < KSTEPS; ++ks) {
          s = Mfma<T>::run(rq[ks], x1f[ks], s);
          dp = Mfma<T>::run(rg[ks], x2f[ks], dp);
        }
      };
      auto in_order = [&]() { __builtin_amdgcn_sched_barrier(0); };
      // the products: dk, dv of step u, dq of step u-1, the scores of step u+1, in the order written: behind each a few LDS
      // reads (more at once would leave the matrix pipe idle while they are issued), of operands that are used four or more
      // products later
      auto products = [&](int u) {
        __builtin_amdgcn_s_setprio(1);  // of the two waves on a SIMD the one with matrix work first
        const bool more_steps = u + 1 < STEPS;
        auto read = [&](int ds_ks, int stat_g, int rows_ks) {
          if (ds_ks >= 0 && u > 0) read_ds(u - 1, ds_ks);
          if (more_steps && stat_g >= 0) read_statistics(u + 1, stat_g);
          if (more_steps && rows_ks >= 0) read_rows(u + 1, rows_ks);
          in_order();
        };
        auto dq_of = [&](int ks) {
          if (u > 0) add_dq(u - 1, ks);
        };
        in_order();
        add_dkv(0, 0);
        read(0, -1, -1);
        read(1, -1, -1);
        add_dkv(0, 1);
        read(2, -1, -1);
        add_dkv(0, 2);
        read(3, -1, -1);
        add_dkv(0, 3);
        read(-1, 0, -1);
        add_dkv(1, 0);
        read(4, 1, -1);
        add_dkv(1, 1);
        read(5, 2, -1);
        dq_of(0);
        dq_of(1);
        read(-1, 3, -1);
        dq_of(2);
        dq_of(3);
        read(-1, -1, 0);
        add_dkv(1, 2);
        read(6, -1, -1);
        read(7, -1, -1);
        dq_of(4);
        read(-1, -1, 1);
        dq_of(5);
        add_dkv(1, 3);
        read(-1, -1, 2);
        if (u + 1 == STEPS) {
          if (ACC && ph == 0) load_old(old2, dvb, dv_rb, FUSED_ROWS);
          in_order();
        }
        dq_of(6);
        dq_of(7);
        read(-1, -1, 3);
        uint32_t frow = 0, srow;  // rows of the next block
        if (u > 0) frow = lds_get<int>(next_rows + fill_row_at + (u - 1) * 128);
        srow = lds_get<int>(next_rows + stats_row_at + u * 128);
        in_order();
        if (more_steps) add_scores();
        __builtin_amdgcn_s_setprio(0);
        in_order();
        if (__builtin_expect(i_ph == 0, true)) {  // the next block's statistics
          if (u > 0) keep_stats(bl + 1, u - 1, st);
          // the last tiles of this block, loaded since the end of the one before, have landed as well
          if (u == 1) __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
          st = load_stats(srow);
        }
        if (u == 1 && more) stage_keys(next_bl, next_ph);  // every wave is done with the keys of this phase
        if (u > 0 && __builtin_expect(last_phase && more_blocks, true)) fill_tile(u - 1, frow);  // every wave is done with step u-1
        in_order();
        if (u + 2 == STEPS) {
          // the last scores are done: their operands' registers take the v rows of the next phase and dk rows that this one
          // adds to, the scores' dv and dq rows (adding, 24 x 65536 812 -> 804 us; dv rows here too 808)
          load_v(more ? next_bl : bl, next_ph);
          if (ACC && ph == 0) load_old(old1, dkb, dk_rb, FUSED_ROWS);
          in_order();
        }
        if (ACC && u + 1 == STEPS && last_phase) {
          load_old(old3, dqb, dq_rb, 0);
          in_order();
        }
      };
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        read_rows(0, i);
        read_statistics(0, i);
      }
      add_scores();
      // One barrier a step; of the two waves on a SIMD one has it behind the weights and one behind the products, so that
      // the one's vector work meets the other's matrix work.
      weights(0);
#pragma unroll
      for (int u = 0; u < STEPS; ++u) {
        products(u);
        if (wave >= 4 || u + 1 == STEPS) lds_barrier();
        if (u + 1 < STEPS) {
          weights(u + 1);
          if (wave < 4) lds_barrier();
        }
      }
      const uint32_t frow = lds_get<int>(next_rows + fill_row_at + (STEPS - 1) * 128);
#pragma unroll
      for (int ks = 0; ks < STEPS; ++ks) read_ds(STEPS - 1, ks);
#pragma unroll
      for (int ks = 0; ks < STEPS; ++ks) add_dq(STEPS - 1, ks);
      if (i_ph == 0) keep_stats(bl + 1, STEPS - 1, st);
      // the next phase's v rows have landed, and with them all loads into LDS; not to be waited for behind the stores
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ++ks) asm volatile("" : "+v"(x2f[ks]));
      asm volatile("" : "+v"(row_ahead));
      if (ACC && ph == 0) {
#pragma unroll
        for (int j = 0; j < 4; ++j) asm volatile("" : "+v"(old1[j]), "+v"(old2[j]));
      }
      if (last_phase && more_blocks) fill_tile(STEPS - 1, frow);
      turn_v();
      // ---- the keys' gradients: turned around in the wave's 4 KB of the dS tiles ----
      const uint32_t ln = opaque_lane();
      if (ph == 0) {
        uint32_t rows[4];
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) rows[j] = key_row(bl, 0, wave * 32 + j * 8 + ln / 8);
        if (wave < (uint32_t)n_waves) {
          auto store = [&](const f32x16 (&acc)[2], float factor, unsigned char* base, uint32_t rb, const vec8 (&old)[4]) {
#pragma unroll
            for (int d2 = 0; d2 < 2; ++d2)
#pragma unroll
              for (int g = 0; g < 4; ++g) {
                vec4 o;
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = (T)(acc[d2][g * 4 + e] * factor);
                lds_put<vec4>(turn + (ln & 31) * 128 + (((4 * d2 + g) ^ (ln & 7)) << 4) + (ln >> 5) * 8, o);
              }
            wave_lds_order();
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) {
              const uint32_t r = j * 8 + ln / 8;
              vec8 o = lds_get<vec8>(turn + r * 128 + (((ln & 7) ^ (r & 7)) << 4));
              if constexpr (ACC) {
#pragma unroll
                for (int e = 0; e < 8; ++e) o[e] = (T)((float)o[e] + (float)old[j][e]);
              }
              *reinterpret_cast<vec8*>(base + (uint32_t)(__umul24(rows[j], rb) + (ln & 7) * 16)) = o;
            }
          };
          store(acc1, p.scale, dkb, dk_rb, old1);
          wave_lds_order();
          store(acc2, 1.f, dvb, dv_rb, old2);
        }
      } else if (!last_phase || !more_blocks) {  // else the next block goes on with the same sampled keys
        const int64_t at = sums0 + (int64_t)(ph - 1) * FUSED_ROWS * FD + ln * 4;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const f32x16 &a1 = acc1[i >> 2], &a2 = acc2[i >> 2];
          const int g = (i & 3) * 4;
          *reinterpret_cast<f32x4*>(p.dk32 + at + i * 256) = f32x4{a1[g], a1[g + 1], a1[g + 2], a1[g + 3]};
          *reinterpret_cast<f32x4*>(p.dv32 + at + i * 256) = f32x4{a2[g], a2[g + 1], a2[g + 2], a2[g + 3]};
        }
      }
      // ---- dq ----
      if (last_phase) {
        lds_barrier();  // every wave is done with its part of the dS tiles
#pragma unroll
        for (int u = 0; u < STEPS; ++u) {
          vec4 o;
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] = (T)(dq[u][e] * p.scale);
          const uint32_t q = (u & 3) * 32 + 8 * ((ln & 15) >> 2) + 4 * qw + (ln & 3);
          lds_put<vec4>(DS + (u < 4 ? 0 : 2 * 16384) + q * 128 + (((2 * dw + (ln >> 5)) ^ (q & 7)) << 4) + ((ln >> 4) & 1) * 8, o);
        }
        uint32_t rows[4];  // behind the barrier other waves may put the next rows in their place
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) rows[j] = query_row(bl, wave * 32 + j * 8 + ln / 8);
        lds_barrier();
        if (wave < (uint32_t)n_waves) {
#pragma unroll
          for (uint32_t j = 0; j < 4; ++j) {
            const uint32_t r = (wave & 3) * 32 + j * 8 + ln / 8;
            vec8 o = lds_get<vec8>(DS + (wave < 4 ? 0 : 2 * 16384) + r * 128 + (((ln & 7) ^ (r & 7)) << 4));
            if constexpr (ACC) {
#pragma unroll
              for (int e = 0; e < 8; ++e) o[e] = (T)((float)o[e] + (float)old3[j][e]);
            }
            *reinterpret_cast<vec8*>(dqb + (uint32_t)(__umul24(rows[j], dq_rb) + (ln & 7) * 16)) = o;
          }
        }
      }
    }
  }
}

}  // namespace

// What the registers and LDS are laid out for: 256 keys and queries per block; with grouped queries a block's dk, dv would
// have to be kept over the query heads beside the sampled keys' sums.  Three passes | this kernel, the whole call in us where it
// writes the gradients: 256 samples (38 launches of 64 to 6144 blocks) 4 heads x 4096 rows 44 | 35, 24 x 4096 98 | 64, 24 x 8192
// 156 | 113, 32 x 16384 361 | 259, 24 x 65536 1038 | 735; without samples 20.4 | 19.3 to 692 | 424 (where it adds to them
// too, but for 16 x 2048 without samples, 22.8 | 23.2); 512: 2 x 512 43.7 | 39.5, 8 x 2048 50 | 48, 24 x 2048 79 | 56, 10 x 16384 165 | 132, 24 x
// 16384 350 | 297, 130 x 2048 296 | 263, 24 x 65536 1402 | 1099.  With more samples a workgroup's four or five phases are a chain that the passes spread over CUs
// which up to 64 blocks leave idle: 768: 1 x 1024 44.8 | 47.9, 2 x 4096 48.8 | 53.0, 8 x 2048 (64 blocks) 54.8 | 56.3, 4 x 4096 56.8 | 56.2, 18 x 1024 (72) 59.5 | 55.2, 24 x 2048 93 |
// 66, 24 x 8192 236 | 205, 24 x 65536 1737 | 1469; 1024: 1 x 1024 47.8 | 56.8, 2 x 4096 54.0 | 63.5, 8 x 2048 61.8 | 64.9, 2 x 8192 63.1 | 65.2, 3 x 6144 (72) 69.6 | 64.6, 5 x
// 4096 67.7 | 65.1, 24 x 2048 107 | 79, 130 x 2048 439 | 409, 24 x 65536 2079 | 1847.
// Head dims below 64, padded for the backward (O as it is): forward and backward of 24 x 16384, d = 48 476 | 418, 512 x 3072, d = 32
// 1570 | 1324, causal 24 x 65536, d = 40 5923 | 5340.
static int64_t fused_blocks(int64_t n) { return (n + FUSED_ROWS - 1) / FUSED_ROWS; }
bool ha_block_bwd_fused_shape(const ha_attn_operands& t, int64_t sample_size) {
  return t.d == FD && t.kv_group == 1 && t.n_q == t.n_k && sample_size % FUSED_ROWS == 0 && sample_size <= FUSED_MAX_SAMPLES &&
         (sample_size <= 512 || t.batch * t.heads * t.segs * fused_blocks(t.n_q) > 64);
}
bool ha_block_bwd_fused_takes(const ha_block_attn_args& a) {
  return !a.smooth_block && (a.block_size + 127) / 128 * 128 == FUSED_ROWS && ha_block_bwd_fused_shape(a.t, a.sample_size);
}

// Blocks per workgroup, one workgroup per CU: the run with the least time by the rounds of workgroups; starting and ending
// one takes as long as two thirds of a block.  Within 0.2 % of the best run of 1 to 8, 10 and 12 at every one of those
// launches, samples or not; as two fifths of a block it chose three rounds of one block for 24 x 8192, 175 us.
// Runs of more than 12 blocks, which save whole starts and shares where that leaves one round or two, forward and backward without mask,
// up to 12 | 64: 32 heads x 65536 1422 | 1399 us, 16 x 65536 727 | 714, 12 x 65536 575 | 557, 24 x 40960 703 | 682, 64 x 24576 1068 | 1057.
static int64_t fused_run(int64_t vseqs, int64_t n) {
  int64_t best = INT64_MAX, run = 1;
  const int64_t blocks = fused_blocks(n);
  for (int64_t r = 1; r <= std::min<int64_t>(blocks, 64); ++r) {
    const int64_t cost = (vseqs * ((blocks + r - 1) / r) + 255) / 256 * (3 * r + 2);
    if (cost < best) {
      best = cost;
      run = r;
    }
  }
  return run;
}
int64_t ha_block_bwd_fused_shares(int64_t vseqs, int64_t n) {
  const int64_t run = fused_run(vseqs, n);
  return (fused_blocks(n) + run - 1) / run;
}

int ha_launch_block_bwd_fused(ha_attn_bwd_params p, int is_f16, hipStream_t stream) {
  const int64_t vseqs = (int64_t)p.batch * p.heads * p.segs;
  p.run_blocks = (int)fused_run(vseqs, p.n_q);
  const int64_t grid = vseqs * ha_block_bwd_fused_shares(vseqs, p.n_q);
  if (grid >= (1ll << 31)) return ha_fail(HA_ERR_SHAPE, "ha_block_attn_bwd: grid of %lld workgroups", (long long)grid);
  auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(FUSED_THREADS), LDS_BYTES, stream, p); };
  auto launch_for = [&](auto short_o) {
    constexpr bool SHORT_O = decltype(short_o)::value;
    if (is_f16) p.accumulate ? launch(ha_block_bwd_fused_kernel<f16_t, true, SHORT_O>) : launch(ha_block_bwd_fused_kernel<f16_t, false, SHORT_O>);
    else p.accumulate ? launch(ha_block_bwd_fused_kernel<bf16_t, true, SHORT_O>) : launch(ha_block_bwd_fused_kernel<bf16_t, false, SHORT_O>);
  };
  if (p.out_last < FD / 8 - 1) launch_for(std::true_type{});
  else launch_for(std::false_type{});
  return ha_launch_status("ha_block_attn_bwd: blocks and sampled keys");
}
