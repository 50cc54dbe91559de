// dq of exact attention at head dim 128, 256 queries per workgroup.
//
// The two alternating stages of attn_bwd_wide.hip with queries and keys exchanged: a wave's matrix stage is dq of step t
// (dS in registers as the B operand, k transposed from LDS) and S, dP of step t + 1, 24 products; its vector stage dS of
// step t + 1.  Barriers, ring and loads as there.  S starts from zero and L enters with the scale of the exponent; dP
// starts from -D, which 16 registers hold.  206 registers, no spills.
// Start: q to the wave's stage, then dO to the same place (from the cache by then: D has been made from its rows and O's,
// whole rows per 16 lanes; a 16-byte piece of 32 rows at a time took 5 us more).
// Bound by the start and the end of a workgroup and the matrix cores: 1.15 to 1.25 us a step, of which the 24 products of
// two waves take 0.7 at 2.4 GHz, and 13 us a workgroup outside its loop, 6 to 7 of them for 240 KB of first loads of every CU
// at once.  (Workgroups that take tile after tile and load the next one's rows beside the loop lost: their loop got as
// much slower as the start got shorter, 493 against 467 us.  So did touching the next workgroup's rows, 513.)
// Measured, bf16, 128 -> 256 queries: causal, 8 segments of 2048 rows, 32 heads, 480 -> 453 us (444 to 456 on other boxes); 32 heads of 4096 223 -> 190;
// without mask 376 -> 342 (1.2 PFLOP/s).
#include "ha_common.h"
#include "attn_tiles.h"
#include "attn_bwd_tiles.h"
#include "attn_bwd.h"

#include <algorithm>
#include <type_traits>

namespace {

constexpr int WD = 128;  // head dim
constexpr int WIDE_QUERIES = 256, WIDE_THREADS = 512;
constexpr int RING = 4;  // tiles of 32 keys in LDS: two in use, two on their way
constexpr uint32_t TILE = 16384;  // 32 k rows, 32 v rows
constexpr uint32_t STAGE = RING * TILE;  // 8 KB per wave: q rows at the start, results at the end
constexpr uint32_t WIDE_LDS_BYTES = STAGE + 65536;

template <typename T, bool CAUSAL>
__global__ __launch_bounds__(WIDE_THREADS, 2) void ha_attn_bwd_wide_dq_kernel(const ha_attn_bwd_params p) {
  ha_load_arguments<(int)sizeof(ha_attn_bwd_params)>();
  typedef typename ElemTraits<T>::vec8 vec8;
  typedef typename ElemTraits<T>::vec4 vec4;
  constexpr int KSTEPS = WD / 16, DB = WD / 32;
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds_block[];  // WIDE_LDS_BYTES, from address 0 on
  (void)lds_block;
  const uint32_t tid = threadIdx.x;
  uint32_t lane = tid & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  // ---- which queries, which keys ----
  const int tiles = (p.n_q + WIDE_QUERIES - 1) / WIDE_QUERIES;
  int tile, vseq;
  if (CAUSAL) {  // the tiles that see the most keys first, over all sequences
    const int n_vseq = gridDim.x / tiles, place = blockIdx.x / n_vseq;
    tile = tiles - 1 - place;
    vseq = blockIdx.x - place * n_vseq;
  } else {
    const int id = xcd_contiguous_id(blockIdx.x, gridDim.x);
    vseq = id / tiles;
    tile = id - vseq * tiles;
  }
  const int seg = vseq % p.segs, bh = vseq / p.segs, b = bh / p.heads, h = bh - b * p.heads, hk = h / p.kv_group;

  const int64_t q_row0 = p.q_seg_off + (int64_t)seg * p.seg_stride, k_row0 = p.k_seg_off + (int64_t)seg * p.seg_stride;
  const int64_t o_row0 = p.o_seg_off + (int64_t)seg * p.o_seg_stride;
  const unsigned char* const qb = (const unsigned char*)((const T*)p.q + b * p.q_sb + h * p.q_sh + q_row0 * p.q_sn);
  const unsigned char* const dob = (const unsigned char*)((const T*)p.dout + b * p.do_sb + h * p.do_sh + q_row0 * p.do_sn);
  const unsigned char* const ob = (const unsigned char*)((const T*)p.out + b * p.o_sb + h * p.o_sh + o_row0 * p.o_sn);
  const unsigned char* const kb = (const unsigned char*)((const T*)p.k + b * p.k_sb + hk * p.k_sh + k_row0 * p.k_sn);
  const unsigned char* const vb = (const unsigned char*)((const T*)p.v + b * p.v_sb + hk * p.v_sh + k_row0 * p.v_sn);
  const uint32_t q_rb = (uint32_t)p.q_sn * 2, do_rb = (uint32_t)p.do_sn * 2, o_rb = (uint32_t)p.o_sn * 2;

  const int ns = ((CAUSAL ? min((tile + 1) * WIDE_QUERIES, p.n_k) : p.n_k) + 31) / 32;  // steps of 32 keys
  const int st_lo = tile * WIDE_QUERIES + wave * 32;  // the wave's queries
  const int own = st_lo >= p.n_q ? 0 : CAUSAL ? min(ns, st_lo / 32 + 1) : ns;  // steps with pairs of the wave

  // ---- loads of the keys' side: into LDS, all of them unknown to the compiler, whose own loads stay out of the loop ----
  const unsigned char* const fill0 = wave < 4 ? kb : vb;
  const uint32_t fill_rb = (uint32_t)(wave < 4 ? p.k_sn : p.v_sn) * 2;
  auto load_tile = [&](int t) {  // past the last step: that one once more
    const int c = min(t, ns - 1);
#pragma unroll
    for (uint32_t j = 0; j < 2; ++j) {
      const uint32_t r = (wave & 3) * 8 + j * 4 + lane / 16;
      const uint32_t row = min(c * 32 + (int)r, p.n_k - 1);
      load_to_lds(fill0, __umul24(row, fill_rb) + (((lane & 15) ^ bwd_swizzle<WD>(r)) << 4), (t & 3) * TILE + wave * 2048 + j * 1024);
    }
  };

  f32x16 acc[DB];  // dQ^T of the wave's queries
#pragma unroll
  for (int d2 = 0; d2 < DB; ++d2)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[d2][i] = 0.f;

  // ---- start: the first three steps, the queries and their statistics ----
  const uint32_t stage = STAGE + wave * 8192;
  auto query_row = [&](uint32_t r) -> uint32_t { return min(st_lo + (int)r, p.n_q - 1); };
  const uint32_t q_row = query_row(lane & 31);  // of the lane's column
  auto load_rows_of = [&](const unsigned char* base, uint32_t rb) {  // the wave's rows to its stage
#pragma unroll
    for (uint32_t j = 0; j < 8; ++j) {
      const uint32_t r = j * 4 + lane / 16;
      load_to_lds(base, __umul24(query_row(r), rb) + (((lane & 15) ^ bwd_swizzle<WD>(r)) << 4), stage + j * 1024);
    }
  };
  const uint32_t row_at = bwd_tile_offset<WD>(lane & 31, lane >> 5);
  load_rows_of(qb, q_rb);
  for (int t = 0; t < 3; ++t) load_tile(t);
  vec8 x1f[KSTEPS], x2f[KSTEPS];  // q, dO rows of the wave's queries
  float lse2;                     // L of the lane's query in log2 units
  f32x16 neg_d;                   // -D in every element: what the dP of a step start from
  {
    // D = sum_c dO * O: whole rows per 16 lanes, whose shares meet in a part of the ring that is not in use yet
    const uint32_t shares = 3 * TILE + wave * 2048;
    {
      vec8 of[8], df[8];
#pragma unroll
      for (uint32_t j = 0; j < 8; ++j) {
        const uint32_t row = query_row(j * 4 + lane / 16);
        of[j] = *reinterpret_cast<const vec8*>(row_address(ob, row, o_rb, min((int)lane & 15, p.out_last) * 16));  // (shorter rows: zeros of dO)
        df[j] = *reinterpret_cast<const vec8*>(row_address(dob, row, do_rb, (lane & 15) * 16));
      }
      lse2 = p.lse[b * p.lse_sb + h * p.lse_sh + o_row0 + q_row] * LOG2E;
#pragma unroll
      for (uint32_t j = 0; j < 8; ++j) {
        float part = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) part = __builtin_fmaf((float)of[j][e], (float)df[j][e], part);
        lds_put<float>(shares + j * 256 + lane * 4, part);
      }
    }
    wave_lds_order();
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): q
    asm volatile("" ::: "memory");
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) x1f[ks] = lds_get<vec8>(stage + (row_at ^ (ks << 5)));
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // q is out of the stage
    load_rows_of(dob, do_rb);
    float part = 0.f;
#pragma unroll
    for (uint32_t i = 0; i < 2; ++i) {
      const f32x4 v = lds_get<f32x4>(shares + (lane & 31) * 64 + (lane >> 5) * 32 + i * 16);
      part += (v[0] + v[1]) + (v[2] + v[3]);
    }
    const float d_row = ha_sum_xor32(part);
#pragma unroll
    for (int i = 0; i < 16; ++i) neg_d[i] = -d_row;
    // the dk, dv passes of the call read both statistics
    if (lane < 32 && st_lo + (int)lane < p.n_q) p.stats[((int64_t)(b * p.heads + h) * p.segs + seg) * p.n_q + q_row] = f32x2{lse2, -d_row};
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);
  asm volatile("" : "+v"(neg_d)::"memory");

#pragma unroll
  for (int ks = 0; ks < KSTEPS; ++ks) x2f[ks] = lds_get<vec8>(stage + (row_at ^ (ks << 5)));
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
    load_tile(t + 3);
  };
  // all but the last step's tile have landed for this wave; then for all
  auto interval_end = [&]() { asm volatile("s_waitcnt vmcnt(2) lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

  int t = 0;
  if (own > 0) {
    f32x16 s, dp;
    vec8 dsn[2];
    vec8 op[8];  // operands read ahead
    uint32_t tr_base, row_base;
    constexpr int AHEAD = 4;
    // operand i of a step's products: 0..7 the transposed k rows of dq, 8..15 the k and 16..23 the v rows of the next
    // step's scores
    auto read_operand = [&](int i) {
      // (behind the empty assembly what is added stays an offset of the instruction and takes no register)
      if (i < 8) {
        const uint32_t at = (i >> 2) * 16 * WD * 2;
        uint32_t lo = tr_base ^ ((i & 3) << 6), hi8 = tr_base ^ ((i & 3) << 6 | 32);
        asm volatile("" : "+v"(lo), "+v"(hi8));
        op[i & 7] = lds_get_tr<T>(lo + at, hi8 + 2048 + at);
      } else if (i < 24) {
        uint32_t at = row_base ^ ((i & 7) << 5);
        asm volatile("" : "+v"(at));
        op[i & 7] = lds_get<vec8>(at + (i >= 16 ? 8192 : 0));
      }
    };
    auto score = [&](int i) {
      const f32x16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      if (i < 16) s = Mfma<T>::run(op[i & 7], x1f[i & 7], i == 8 ? zero : s);
      else dp = Mfma<T>::run(op[i & 7], x2f[i & 7], i == 16 ? neg_d : dp);
    };
    // dS of step t in s, dp; the first operands of its products are read
    auto weights = [&](int t) {
      tr_base = tr_at + (t & 3) * TILE;
      const int y0 = t * 32;
      const bool touched = y0 + 31 >= p.n_k || (CAUSAL && y0 + 31 > st_lo);
      if (__builtin_expect(touched, false)) {
        asm volatile("" ::);  // keeps this a branch
        int last = p.n_k - 1 - y0 - 4 * (int)(lane >> 5);
        if (CAUSAL) last = min(last, st_lo + (int)(lane & 31) - y0 - 4 * (int)(lane >> 5));
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (8 * (i >> 2) + (i & 3) > last) s[i] = -__builtin_inff();
      }
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        in_order();
#pragma unroll
        for (int i = 0; i < 8; ++i)
          dsn[kk][i] = (T)(__builtin_amdgcn_exp2f(__builtin_fmaf(s[kk * 8 + i], p.scale_log2, -lse2)) * dp[kk * 8 + i]);
        asm volatile("" : "+v"(dsn[kk]));
      }
#pragma unroll
      for (int i = 0; i < AHEAD; ++i) read_operand(i);
      in_order();
    };
    // dq of step t, then (more) the scores of the next one
    auto products = [&](int t, auto more) {
      __builtin_amdgcn_s_setprio(1);
      row_base = row_at + ((t + 1) & 3) * TILE;
      in_order();
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        acc[i & 3] = Mfma<T>::run(op[i & 7], dsn[i >> 2], acc[i & 3]);
        in_order();
        if (decltype(more)::value || i + AHEAD < 8) read_operand(i + AHEAD);
        in_order();
      }
      if constexpr (decltype(more)::value) {
#pragma unroll
        for (int i = 8; i < 24; ++i) {
          score(i);
          in_order();
          read_operand(i + AHEAD);
          in_order();
        }
      }
      __builtin_amdgcn_s_setprio(0);
    };
    row_base = row_at;
#pragma unroll
    for (int i = 8; i < 24; ++i) {
      in_order();
      read_operand(i);
      score(i);
    }
    in_order();
    weights(0);
    for (; t + 1 < own; ++t) {
      interval_loads(t);
      products(t, std::true_type{});
      if (wave >= 4) interval_end();
      weights(t + 1);
      if (wave < 4) interval_end();
    }
    interval_loads(t);
    products(t, std::false_type{});
    interval_end();
    ++t;
  }
  for (; t < ns; ++t) {  // steps after the wave's last one
    interval_loads(t);
    interval_end();
  }

  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): no load into this workgroup's LDS outlives it
  // ---- results, turned around in LDS: 16 lanes write a whole row ----
  if (st_lo >= p.n_q) return;
  const uint32_t hi = lane >> 5, col = lane & 31;
  unsigned char* const dqb = (unsigned char*)((T*)p.dq + b * p.dq_sb + h * p.dq_sh + q_row0 * p.dq_sn);
  const int64_t dq_rb = p.dq_sn * 2;
  uint32_t rows[8];
#pragma unroll
  for (uint32_t j = 0; j < 8; ++j) rows[j] = query_row(j * 4 + lane / 16);
  if (p.accumulate) {
    // what is there and the fp32 sum are rounded once, together: 16 rows at a time, [16][WD] fp32, 16-byte pieces XOR-ed
    // with the row number
    vec8 old[8];
#pragma unroll
    for (uint32_t j = 0; j < 8; ++j) old[j] = *reinterpret_cast<const vec8*>(dqb + rows[j] * dq_rb + (lane & 15) * 16);
#pragma unroll
    for (uint32_t part = 0; part < 2; ++part) {
      if (col >> 4 == part) {
#pragma unroll
        for (int d2 = 0; d2 < DB; ++d2)
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            f32x4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = acc[d2][g * 4 + e] * p.scale;
            lds_put<f32x4>(stage + (col & 15) * (WD * 4) + (((8 * d2 + 2 * g + hi) ^ (col & 15)) << 4), o);
          }
      }
      wave_lds_order();
#pragma unroll
      for (uint32_t j = part * 4; j < part * 4 + 4; ++j) {
        const uint32_t r = j * 4 + lane / 16, at = stage + (r & 15) * (WD * 4), piece = 2 * (lane & 15);
        const f32x4 lo = lds_get<f32x4>(at + ((piece ^ (r & 15)) << 4)), up = lds_get<f32x4>(at + (((piece + 1) ^ (r & 15)) << 4));
        vec8 o;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = (T)((e < 4 ? lo[e & 3] : up[e & 3]) + (float)old[j][e]);
        if (st_lo + (int)r < p.n_q) *reinterpret_cast<vec8*>(dqb + rows[j] * dq_rb + (lane & 15) * 16) = o;
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
      for (int e = 0; e < 4; ++e) o[e] = (T)(acc[d2][g * 4 + e] * p.scale);
      lds_put<vec4>(stage + col * 256 + (((4 * d2 + g) ^ (col & 15)) << 4) + hi * 8, o);
    }
  wave_lds_order();
#pragma unroll
  for (uint32_t j = 0; j < 8; ++j) {
    const uint32_t r = j * 4 + lane / 16;
    if (st_lo + (int)r < p.n_q)
      *reinterpret_cast<vec8*>(dqb + rows[j] * dq_rb + (lane & 15) * 16) = lds_get<vec8>(stage + r * 256 + (((lane & 15) ^ (r & 15)) << 4));
  }
}

}  // namespace

int ha_launch_bwd_wide_dq(const ha_attn_bwd_params& p, bool causal, int is_f16, int64_t grid, hipStream_t stream, const char* what) {
  if (grid <= 0) return HA_OK;
  if (grid >= (1ll << 31)) return ha_fail(HA_ERR_SHAPE, "%s: grid of %lld workgroups", what, (long long)grid);
  auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(WIDE_THREADS), WIDE_LDS_BYTES, stream, p); };
  auto typed = [&](auto t) {
    typedef decltype(t) T;
    if (causal) launch(ha_attn_bwd_wide_dq_kernel<T, true>);
    else launch(ha_attn_bwd_wide_dq_kernel<T, false>);
  };
  if (is_f16) typed(f16_t{});
  else typed(bf16_t{});
  return ha_launch_status(what);
}
