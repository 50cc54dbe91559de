// dk, dv of exact attention, of plain blocks and of sampled keys at head dim 128, 256 keys per workgroup.
//
// Same sums as the passes of attn_bwd.hip, which keep 128 keys in 4 waves, one on each SIMD, with 480 registers each.
// There the 32 matrix products of a step of 32 queries (1080 cycles) and its soft-max and LDS reads (about 700) follow one
// another.  Here 8 waves of 32 keys alternate, two on each SIMD: a wave does products while the other has its vector
// stage, and a tile of queries is read by twice the keys.
//   - The wave's matrix stage: dk, dv of step t (P, dS in registers as B operands, q and dO transposed from LDS), then S,
//     dP of step t + 1, operands read 4 products ahead.  Its vector stage: P, dS of step t + 1 and the first operands.
//     Waves 0-3 pass the step's one barrier after the vector stage, waves 4-7 after the matrix stage, which keeps the two
//     waves of a SIMD (w, w + 4) in different stages.
//   - Registers: 128 accumulators, 64 for the keys' k and v, 64 for S, dP, P, dS, 32 operands: 256 (the sampled pass spills one, outside its loop).
//   - LDS, 136 KB: four tiles of 32 q and dO rows, filled three steps ahead by loads that bypass the registers, four
//     steps' statistics, eight steps' row numbers.  The compiler must not see those loads (it would wait for all of them at
//     every LDS access): assembly, counted by hand, the step's end waits for all but the last tile's two.
//     Another 64 KB hold the k rows at the start and the results at the end, turned to whole rows.
//   - Causal tiles one by one, the ones with the most queries first.
// Bound by the matrix cores and what does not overlap them: 32 products of 34 cycles and two waves on each SIMD are 0.9 us
// at 2.4 GHz of a step's 1.3 us (half the chip at work) to 1.9 us (all of it).  Measured, bf16, 128 -> 256 keys: exact
// causal, 8 segments of 2048 rows, 32 query heads on 8, 753 -> 540 us (540 to 577 on other boxes; 1.0 PFLOP/s of the visible pairs); 32 heads of 4096
// rows without mask 684 -> 477 (1.15); blocks of 256 of 16384 rows, 32 heads on 8, 225 -> 159; 256 sampled keys of 8192
// queries, 32 heads, 128 -> 75 (with atomic adds instead of stores at the end 122).
#include "ha_common.h"
#include "attn_tiles.h"
#include "attn_bwd_tiles.h"
#include "attn_bwd.h"

#include <algorithm>
#include <type_traits>

namespace {

constexpr int WD = 128;  // head dim
constexpr int WIDE_KEYS = 256, WIDE_THREADS = 512;
constexpr int RING = 4;  // tiles of 32 queries in LDS: two in use, two on their way
constexpr uint32_t TILE = 16384;  // 32 q rows, 32 dO rows
constexpr uint32_t STAGE = RING * TILE;  // 8 KB per wave: k rows at the start, results at the end
constexpr uint32_t LSE = STAGE + 65536, DELTA = LSE + 4 * 128, RAW = DELTA + 4 * 128, ROWS = RAW + 4 * 256, WIDE_LDS_BYTES = ROWS + 8 * 256;

template <typename T, int PASS, bool CAUSAL>
__global__ __launch_bounds__(WIDE_THREADS, 2) void ha_attn_bwd_wide_kernel(const ha_attn_bwd_params p) {
  ha_load_arguments<(int)sizeof(ha_attn_bwd_params)>();
  typedef typename ElemTraits<T>::vec8 vec8;
  typedef typename ElemTraits<T>::vec4 vec4;
  constexpr int KSTEPS = WD / 16, DB = WD / 32;
  constexpr bool EXACT = PASS == HA_BWD_DKV_EXACT, BLOCK = PASS == HA_BWD_DKV_BLOCK, SAMPLED = PASS == HA_BWD_DKV_SAMPLED;
  // in fp16 the exact pass rounds dS with its factor `scale`: see attn_bwd_tile.inc
  constexpr bool SCALE_DS = EXACT && std::is_same<T, f16_t>::value;
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds_block[];  // WIDE_LDS_BYTES, from address 0 on
  (void)lds_block;
  const uint32_t tid = threadIdx.x;
  uint32_t lane = tid & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  // ---- which keys, which queries ----
  const int st_total = SAMPLED ? p.sample_size : p.n_k, st_tiles = (st_total + WIDE_KEYS - 1) / WIDE_KEYS;
  const int splits = SAMPLED ? (p.n_q + p.q_split - 1) / p.q_split : 1;
  int tile, vseq, split = 0;
  if (EXACT && CAUSAL) {  // the tiles that stream the most queries first, over all sequences
    const int n_vseq = gridDim.x / st_tiles;
    tile = blockIdx.x / n_vseq;
    vseq = blockIdx.x - tile * n_vseq;
  } else {
    int rest = xcd_contiguous_id(blockIdx.x, gridDim.x);
    tile = rest % st_tiles;
    rest /= st_tiles;
    split = rest % splits;
    vseq = rest / splits;
  }
  const int seg = vseq % p.segs, bh = vseq / p.segs, kv_heads = p.heads / p.kv_group;
  // complete sums over the query heads of a group, or (sampled keys) the share of a range of one query head's queries
  const int n_group = SAMPLED ? 1 : p.kv_group;
  const int b = SAMPLED ? bh / p.heads : bh / kv_heads;
  const int h0 = SAMPLED ? bh - b * p.heads : (bh - b * kv_heads) * p.kv_group, hk = h0 / p.kv_group;

  const int64_t q_row0 = p.q_seg_off + (int64_t)seg * p.seg_stride, k_row0 = p.k_seg_off + (int64_t)seg * p.seg_stride;
  const unsigned char* const q0 = (const unsigned char*)((const T*)p.q + b * p.q_sb + h0 * p.q_sh + q_row0 * p.q_sn);
  const unsigned char* const do0 = (const unsigned char*)((const T*)p.dout + b * p.do_sb + h0 * p.do_sh + q_row0 * p.do_sn);
  const unsigned char* const kb = (const unsigned char*)((const T*)p.k + b * p.k_sb + hk * p.k_sh + k_row0 * p.k_sn);
  const unsigned char* const vb = (const unsigned char*)((const T*)p.v + b * p.v_sb + hk * p.v_sh + k_row0 * p.v_sn);
  const unsigned char* const stats0 = (const unsigned char*)(p.stats + ((int64_t)(b * p.heads + h0) * p.segs + seg) * p.n_q);
  const uint32_t k_rb = (uint32_t)p.k_sn * 2, v_rb = (uint32_t)p.v_sn * 2;
  const int idx_shift = p.idx64 ? 3 : 2;
  const unsigned char* const q_idx0 = (const unsigned char*)p.q_idx + ((b * p.qi_sb + h0 * p.qi_sh + (int64_t)seg * p.n_q * p.qi_sn) << idx_shift);
  const unsigned char* const k_idx = (const unsigned char*)p.k_idx + ((b * p.ki_sb + hk * p.ki_sh + (int64_t)seg * p.n_k * p.ki_sn) << idx_shift);
  const uint32_t qi_rb = (uint32_t)p.qi_sn << idx_shift, ki_rb = (uint32_t)p.ki_sn << idx_shift;

  // the queries of one head: y_first .. y_end - 1, in steps of 32
  int y_first = 0, y_end = p.n_q;
  if (EXACT && CAUSAL) y_first = tile * WIDE_KEYS;
  if (BLOCK) {
    const int block_id = 2 * tile / p.block_tiles;
    y_first = block_id * p.block_tiles * 128;
    y_end = min(y_first + p.block_tiles * 128, p.n_q);
  }
  if (SAMPLED) {
    y_first = split * p.q_split;
    y_end = min(y_first + p.q_split, p.n_q);
  }
  const int ns = y_end > y_first ? (y_end - y_first + 31) / 32 : 0, n_t = ns * n_group;

  // the wave's keys
  const int st_lo = tile * WIDE_KEYS + wave * 32;
  auto key_row = [&](uint32_t r) -> uint32_t {  // row of key r of the wave, clamped
    const int pos = min(st_lo + (int)r, st_total - 1);
    if (BLOCK) return *reinterpret_cast<const int*>(row_address(k_idx, pos, ki_rb, 0));
    if (SAMPLED && p.sampled_idx) return ha_load_idx(p.sampled_idx, b * p.si_sb + hk * p.si_sh + pos, p.idx64);
    return pos;
  };

  // ---- loads of the queries' side: into LDS, all of them unknown to the compiler, whose own loads stay out of the loop ----
  const unsigned char* const fill0 = wave < 4 ? q0 : do0;
  const int64_t fill_sh = (wave < 4 ? p.q_sh : p.do_sh) * 2;
  const uint32_t fill_rb = (uint32_t)(wave < 4 ? p.q_sn : p.do_sn) * 2;
  struct Cursor {  // a step: its number in its head, the head
    int j, g;
  };
  auto advance = [&](Cursor& c) {  // stays on the last step
    if (c.j + 1 < ns) ++c.j;
    else if (c.g + 1 < n_group) c.j = 0, ++c.g;
  };
  auto query_row = [&](const Cursor& c, int t, uint32_t r) -> uint32_t {
    if (BLOCK) return lds_get<int>(ROWS + (t & 7) * 256 + r * 4);
    return min(y_first + c.j * 32 + (int)r, p.n_q - 1);
  };
  auto load_rows = [&](const Cursor& c, int t) {  // row numbers of a step
    if (!BLOCK || (uint32_t)(t & 7) != wave) return;
    load_to_lds_4(q_idx0 + ((c.g * p.qi_sh) << idx_shift), __umul24(y_first + c.j * 32 + (lane & 31), qi_rb), ROWS + (t & 7) * 256);
  };
  auto load_stats = [&](const Cursor& c, int t) {
    if ((uint32_t)(t & 7) != wave) return;
    load_to_lds_4(stats0 + (int64_t)c.g * p.segs * p.n_q * 8, query_row(c, t, lane >> 1) * 8 + (lane & 1) * 4, RAW + (t & 3) * 256);
  };
  const float neg_inv = p.neg_inv_scale * (1.f / LOG2E);  // L arrives in log2 units
  auto keep_stats = [&](int j, int t) {
    if ((uint32_t)(t & 7) != wave) return;
    const f32x2 raw = lds_get<f32x2>(RAW + (t & 3) * 256 + (lane & 31) * 8);
    const bool past = y_first + j * 32 + (int)(lane & 31) >= y_end;  // L = inf: no weight
    if (lane < 32) {
      lds_put<float>(LSE + (t & 3) * 128 + lane * 4, (past ? __builtin_inff() : raw[0]) * neg_inv);
      lds_put<float>(DELTA + (t & 3) * 128 + lane * 4, raw[1]);
    }
  };
  auto load_tile = [&](const Cursor& c, int t) {
    const unsigned char* const base = fill0 + c.g * fill_sh;
#pragma unroll
    for (uint32_t j = 0; j < 2; ++j) {
      const uint32_t r = (wave & 3) * 8 + j * 4 + lane / 16;
      load_to_lds(base, __umul24(query_row(c, t, r), fill_rb) + (((lane & 15) ^ bwd_swizzle<WD>(r)) << 4),
                  (t & 3) * TILE + wave * 2048 + j * 1024);
    }
  };

  f32x16 acc1[DB], acc2[DB];  // dK^T, dV^T of the wave's keys
#pragma unroll
  for (int d2 = 0; d2 < DB; ++d2)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc1[d2][i] = acc2[d2][i] = 0.f;

  if (n_t > 0) {
    // ---- start: row numbers, then the first three steps, the keys ----
    Cursor c_idx = {0, 0}, c_tile = {0, 0}, c_keep = {0, 0};  // of step t+4, t+3, t+2 of the loop
    if (BLOCK) {
      for (int t = 0; t < 4; ++t, advance(c_idx)) load_rows(c_idx, t);
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
      lds_barrier();
    }
    const uint32_t stage = STAGE + wave * 8192;
    {
      uint32_t rows[8];
#pragma unroll
      for (uint32_t j = 0; j < 8; ++j) rows[j] = key_row(j * 4 + lane / 16);
#pragma unroll
      for (uint32_t j = 0; j < 8; ++j)
        load_to_lds(kb, __umul24(rows[j], k_rb) + (((lane & 15) ^ bwd_swizzle<WD>(j * 4 + lane / 16)) << 4), stage + j * 1024);
    }
    for (int t = 0; t < 3; ++t, advance(c_tile)) {
      load_stats(c_tile, t);
      load_tile(c_tile, t);
    }
    vec8 x1f[KSTEPS], x2f[KSTEPS];  // k, v rows of the wave's keys
    {
      const uint32_t row = key_row(lane & 31), hi = lane >> 5;
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ++ks) x2f[ks] = *reinterpret_cast<const vec8*>(row_address(vb, row, v_rb, (ks * 16 + hi * 8) * 2));
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);
    asm volatile("" ::: "memory");
    const uint32_t row_at = bwd_tile_offset<WD>(lane & 31, lane >> 5);
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) x1f[ks] = lds_get<vec8>(stage + (row_at ^ (ks << 5)));
    keep_stats(c_keep.j, 0);
    advance(c_keep);
    keep_stats(c_keep.j, 1);
    advance(c_keep);
    lds_barrier();

    uint32_t tr_at;
    {
      const uint32_t g = lane >> 4, sl = lane & 15, key = (g >> 1) * 4 + (sl >> 2), w = sl & 3;
      tr_at = bwd_tile_offset<WD>(key, (g & 1) * 2 + (w >> 1)) + (w & 1) * 8;  // rows 8 further on: 2048 further, another swizzle
    }
    auto in_order = [&]() { __builtin_amdgcn_sched_barrier(0); };
    // what a step asks for
    auto interval_loads = [&](int t) {
      asm volatile("" : "+v"(lane));  // what is made from it is not kept in registers
      load_rows(c_idx, t + 4);
      load_stats(c_tile, t + 3);
      keep_stats(c_keep.j, t + 2);
      load_tile(c_tile, t + 3);
      if (BLOCK) advance(c_idx);
      advance(c_tile);
      advance(c_keep);
    };
    // all but the last step's tile have landed for this wave; then for all
    auto interval_end = [&]() { asm volatile("s_waitcnt vmcnt(2) lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

    int t = 0;
    for (int g = 0; g < n_group; ++g) {
      // steps before the wave's own rows have no pairs with them (keys past the end have none at all)
      const int first = st_lo >= st_total ? ns : EXACT && CAUSAL ? min((int)wave, ns) : 0;
      for (int j = 0; j < first; ++j, ++t) {
        interval_loads(t);
        interval_end();
      }
      if (first < ns) {
        f32x16 s, dp;
        vec8 pn[2], dsn[2];
        vec8 op[8];  // operands read ahead
        uint32_t tr_base, row_base;
        constexpr int AHEAD = 4;
        // operand i of a step's products: 0..15 the transposed q (even) and dO rows of dk and dv, 16..23 the q and 24..31 the dO
        // rows of the next step's scores
        auto read_operand = [&](int i) {
          // (behind the empty assembly what is added stays an offset of the instruction and takes no register)
          if (i < 16) {
            const uint32_t at = (i >> 3) * 16 * WD * 2 + (i & 1) * 8192;
            uint32_t lo = tr_base ^ ((i >> 1 & 3) << 6), hi8 = tr_base ^ ((i >> 1 & 3) << 6 | 32);
            asm volatile("" : "+v"(lo), "+v"(hi8));
            op[i & 7] = lds_get_tr<T>(lo + at, hi8 + 2048 + at);
          } else if (i < 32) {
            uint32_t at = row_base ^ ((i & 7) << 5);
            asm volatile("" : "+v"(at));
            op[i & 7] = lds_get<vec8>(at + (i >= 24 ? 8192 : 0));
          }
        };
        auto read_statistics = [&](f32x16& c, uint32_t at, int t, int g) {
          const f32x4 v = lds_get<f32x4>(at + (t & 3) * 128 + (lane >> 5) * 16 + g * 32);
#pragma unroll
          for (int e = 0; e < 4; ++e) c[g * 4 + e] = v[e];
        };
        // P and dS of the step in s, dp; the first operands of its products are read
        auto weights = [&](int j, int t) {
          tr_base = tr_at + (t & 3) * TILE;
          const int y0 = y_first + j * 32;
          if (EXACT) {
            const bool touched = y0 + 31 >= p.n_q || (CAUSAL && y0 < st_lo + 31);
            if (__builtin_expect(touched, false)) {
              asm volatile("" ::);  // keeps this a branch
              const int last = p.n_q - 1 - y0 - 4 * (int)(lane >> 5), first = CAUSAL ? st_lo + (int)(lane & 31) - y0 - 4 * (int)(lane >> 5) : 0;
#pragma unroll
              for (int i = 0; i < 16; ++i) {
                const int r = 8 * (i >> 2) + (i & 3);
                if (r > last || (CAUSAL && r < first)) s[i] = -__builtin_inff();
              }
            }
          }
#pragma unroll
          for (int kk = 0; kk < 2; ++kk) {
            in_order();
#pragma unroll
            for (int i = 0; i < 8; ++i) {
              const float pv = __builtin_amdgcn_exp2f(s[kk * 8 + i] * p.scale_log2);
              pn[kk][i] = (T)pv;
              dsn[kk][i] = (T)(pv * (SCALE_DS ? dp[kk * 8 + i] * p.scale : dp[kk * 8 + i]));
            }
            asm volatile("" : "+v"(pn[kk]), "+v"(dsn[kk]));
          }
#pragma unroll
          for (int i = 0; i < AHEAD; ++i) read_operand(i);
          in_order();
        };
        // dk, dv of the step, then (more) the scores of the next one
        auto products = [&](int t, auto more) {
          __builtin_amdgcn_s_setprio(1);
          row_base = row_at + ((t + 1) & 3) * TILE;
          in_order();
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const int kk = i >> 3, d2 = i >> 1 & 3;
            if (i & 1) acc2[d2] = Mfma<T>::run(op[i & 7], pn[kk], acc2[d2]);
            else acc1[d2] = Mfma<T>::run(op[i & 7], dsn[kk], acc1[d2]);
            in_order();
            if (decltype(more)::value || i + AHEAD < 16) read_operand(i + AHEAD);
            if (decltype(more)::value && i >= 12) read_statistics(s, LSE, t + 1, i - 12);
            in_order();
          }
          if constexpr (decltype(more)::value) {
#pragma unroll
            for (int i = 16; i < 32; ++i) {
              if (i >= 24) dp = Mfma<T>::run(op[i & 7], x2f[i & 7], dp);
              else s = Mfma<T>::run(op[i & 7], x1f[i & 7], s);
              in_order();
              if (i < 20) read_statistics(dp, DELTA, t + 1, i - 16);
              read_operand(i + AHEAD);
              in_order();
            }
          }
          __builtin_amdgcn_s_setprio(0);
        };
        row_base = row_at + (t & 3) * TILE;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          read_statistics(s, LSE, t, i);
          read_statistics(dp, DELTA, t, i);
        }
#pragma unroll
        for (int i = 16; i < 32; ++i) {
          in_order();
          read_operand(i);
          if (i >= 24) dp = Mfma<T>::run(op[i & 7], x2f[i & 7], dp);
          else s = Mfma<T>::run(op[i & 7], x1f[i & 7], s);
        }
        in_order();
        weights(first, t);
        for (int j = first; j + 1 < ns; ++j, ++t) {
          interval_loads(t);
          products(t, std::true_type{});
          if (wave >= 4) interval_end();
          weights(j + 1, t + 1);
          if (wave < 4) interval_end();
        }
        interval_loads(t);
        products(t, std::false_type{});
        interval_end();
        ++t;
      }
    }
  }

  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): no load into this workgroup's LDS outlives it
  // ---- results ----
  const uint32_t hi = lane >> 5, col = lane & 31;
  if (!SCALE_DS) {
#pragma unroll
    for (int d2 = 0; d2 < DB; ++d2)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc1[d2][i] *= p.scale;
  }
  const uint32_t stage = STAGE + wave * 8192;
  if (st_lo >= st_total) return;
  // fp32 sums through the stage, 16 of the wave's keys at a time: rows [16][WD], 16-byte pieces XOR-ed with the row number
  auto turn = [&](const f32x16 (&acc)[DB], uint32_t part) {
    if (col >> 4 == part) {
#pragma unroll
      for (int d2 = 0; d2 < DB; ++d2)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          lds_put<f32x4>(stage + (col & 15) * (WD * 4) + (((8 * d2 + 2 * g + hi) ^ (col & 15)) << 4),
                         f32x4{acc[d2][g * 4], acc[d2][g * 4 + 1], acc[d2][g * 4 + 2], acc[d2][g * 4 + 3]});
    }
    wave_lds_order();
  };
  auto turned = [&](uint32_t r, uint32_t piece) { return lds_get<f32x4>(stage + r * (WD * 4) + ((piece ^ r) << 4)); };
  if (SAMPLED) {
    // this share's rows: [(batch, key head, segment)][share][slot], written whole
    const int shares = p.kv_group * splits, share = (h0 - hk * p.kv_group) * splits + split;
    const int64_t slot0 = (((((int64_t)b * kv_heads + hk) * p.segs + seg) * shares + share) * p.sample_size + st_lo) * WD;
#pragma unroll
    for (int which = 0; which < 2; ++which) {
      float* const dst = (which == 0 ? p.dk32 : p.dv32) + slot0;
#pragma unroll
      for (uint32_t part = 0; part < 2; ++part) {
        turn(which == 0 ? acc1 : acc2, part);
#pragma unroll
        for (uint32_t j = 0; j < 8; ++j) {
          const uint32_t r = j * 2 + hi;
          *reinterpret_cast<f32x4*>(dst + (part * 16 + r) * WD + col * 4) = turned(r, col);
        }
        wave_lds_order();
      }
    }
    return;
  }
  unsigned char* const dkb = (unsigned char*)((T*)p.dk + b * p.dk_sb + hk * p.dk_sh + k_row0 * p.dk_sn);
  unsigned char* const dvb = (unsigned char*)((T*)p.dv + b * p.dv_sb + hk * p.dv_sh + k_row0 * p.dv_sn);
  // turned around in LDS: 16 lanes write a whole row
  uint32_t rows[8];
#pragma unroll
  for (uint32_t j = 0; j < 8; ++j) rows[j] = key_row(j * 4 + lane / 16);
  auto store = [&](const f32x16 (&acc)[DB], unsigned char* base, int64_t row_bytes) {
    // What is there and the fp32 sum are rounded once, together, as in the passes of 128 keys (rounded to 16 bits for the
    // turn first, 320 heads of 256 causal rows take 95 us instead of 97 for all gradients, 256 of 1280 rows 753 and 759).
    if (p.accumulate) {
      vec8 old[8];
#pragma unroll
      for (uint32_t j = 0; j < 8; ++j) old[j] = *reinterpret_cast<const vec8*>(base + rows[j] * row_bytes + (lane & 15) * 16);
#pragma unroll
      for (uint32_t part = 0; part < 2; ++part) {
        turn(acc, part);
#pragma unroll
        for (uint32_t j = part * 4; j < part * 4 + 4; ++j) {
          const uint32_t r = j * 4 + lane / 16;
          const f32x4 lo = turned(r & 15, 2 * (lane & 15)), up = turned(r & 15, 2 * (lane & 15) + 1);
          vec8 o;
#pragma unroll
          for (int e = 0; e < 8; ++e) o[e] = (T)((e < 4 ? lo[e & 3] : up[e & 3]) + (float)old[j][e]);
          if (st_lo + (int)r < st_total) *reinterpret_cast<vec8*>(base + rows[j] * row_bytes + (lane & 15) * 16) = o;
        }
        wave_lds_order();
      }
      return;
    }
#pragma unroll
    for (int d2 = 0; d2 < DB; ++d2)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        vec4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = (T)acc[d2][g * 4 + e];
        lds_put<vec4>(stage + col * 256 + (((4 * d2 + g) ^ (col & 15)) << 4) + hi * 8, o);
      }
    wave_lds_order();
#pragma unroll
    for (uint32_t j = 0; j < 8; ++j) {
      const uint32_t r = j * 4 + lane / 16;
      if (st_lo + (int)r < st_total)
        *reinterpret_cast<vec8*>(base + rows[j] * row_bytes + (lane & 15) * 16) = lds_get<vec8>(stage + r * 256 + (((lane & 15) ^ (r & 15)) << 4));
    }
    wave_lds_order();
  };
  if (n_t > 0 || !p.accumulate) {
    store(acc1, dkb, p.dk_sn * 2);
    store(acc2, dvb, p.dv_sn * 2);
  }
}

}  // namespace

int ha_launch_bwd_wide(const ha_attn_bwd_params& p, int pass, bool causal, int is_f16, int64_t grid, hipStream_t stream, const char* what) {
  if (grid <= 0) return HA_OK;
  if (grid >= (1ll << 31)) return ha_fail(HA_ERR_SHAPE, "%s: grid of %lld workgroups", what, (long long)grid);
  auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(WIDE_THREADS), WIDE_LDS_BYTES, stream, p); };
  auto typed = [&](auto t) {
    typedef decltype(t) T;
    if (pass == HA_BWD_DKV_BLOCK) launch(ha_attn_bwd_wide_kernel<T, HA_BWD_DKV_BLOCK, false>);
    else if (pass == HA_BWD_DKV_SAMPLED) launch(ha_attn_bwd_wide_kernel<T, HA_BWD_DKV_SAMPLED, false>);
    else if (causal) launch(ha_attn_bwd_wide_kernel<T, HA_BWD_DKV_EXACT, true>);
    else launch(ha_attn_bwd_wide_kernel<T, HA_BWD_DKV_EXACT, false>);
  };
  if (is_f16) typed(f16_t{});
  else typed(bf16_t{});
  return ha_launch_status(what);
}
