// Bucket ids and bucket order of one unit of a sequence's rows by one workgroup of an attention launch: the work of the hash
// launch (lsh_hash.hip) and of rank_units_kernel (bucket_sort.hip) on a unit, without the ids' way through memory.
//
// The exact causal launch of a forward pass needs neither, so its grid carries these workgroups along (ha_rank_beside in
// attn_fwd.h) and the two launches with their start-up and their idle CUs are gone from the chain.  A unit is bound by the time
// its rows take to arrive, 4 waves asking for 16 or 32 KB each at a time; a launch of nothing but these workgroups would
// be slower than the two launches that it replaces.  The exact tiles hide it where they are about one round (24 heads of 4096 rows: launch 36 -> 42 us, hash
// and ranking 10); a launch of several rounds grows by what hashing takes alone (16 of 20479, d = 96: 177 -> 205 us, hash and ranking 27; 32 on 2 of
// 32768, d = 128: 545 -> 611, 67), and what is saved is the launches themselves (rank_beside_leaves in api.hip).
#pragma once

#include "attn_fwd.h"
#include "lsh_tiles.h"
#include "rank_tiles.h"

namespace {

// Units of up to HA_SORT_CHUNK rows, or HA_SORT_BESIDE where a unit is a whole segment and no placement launch follows.
// LDS: the order (2 bytes a row), the waves' bucket counts (WAVES KB and 4 bytes per wave), the ids (a byte a row), the projection
template <typename T, int PARTS, int WAVES, int ORDER_BYTES, int COUNT_BYTES, int ID_BYTES, int PROJ_BYTES>
__device__ __forceinline__ void hash_and_rank_unit(const ha_attn_kernel_params& p, const ha_rank_beside& a, int local, unsigned char (&lds_order)[ORDER_BYTES],
                                                   unsigned char (&lds_counts)[COUNT_BYTES], unsigned char (&lds_ids)[ID_BYTES],
                                                   unsigned char (&lds_proj)[PROJ_BYTES]) {
  typedef typename ElemTraits<T>::vec8 vec8;
  typedef Projection<T, PARTS> P;
  constexpr int THREADS = 64 * WAVES;
  static_assert(ORDER_BYTES >= 2 * HA_SORT_BESIDE && COUNT_BYTES >= WAVES * 1028 && ID_BYTES >= HA_SORT_BESIDE &&
                PROJ_BYTES >= P::LDS_BYTES && WAVES >= 4);
  const ha_unit_grid& g = a.grid;
  uint16_t* const order = reinterpret_cast<uint16_t*>(lds_order);
  uint32_t* const counts = reinterpret_cast<uint32_t*>(lds_counts);
  uint32_t* const wave_totals = counts + WAVES * 256;
  uint8_t* const ids = lds_ids;
  T* const proj = reinterpret_cast<T*>(lds_proj);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  // ---- which unit, and where its rows are ----
  const int which = local >= a.units0 ? 1 : 0;
  local -= which ? a.units0 : 0;
  const int seq = local / a.num_units, u = a.first_unit[which] + local % a.num_units;
  const int gran = u / g.units_per_granule, w = u % g.units_per_granule;
  const int64_t unit_row = (int64_t)gran * g.granule + (int64_t)w * g.unit;  // in its sequence
  const int len = (int)min((int64_t)g.unit, g.granule - (int64_t)w * g.unit);
  const int real = (int)min((int64_t)len, a.n_read - unit_row);  // rows from there on are the appended zero row
  const int heads = which ? p.heads / p.kv_group : p.heads, b = seq / heads, h = seq - b * heads;
  const unsigned char* const base = which ? (const unsigned char*)((const T*)p.k + b * p.k_sb + h * p.k_sh + unit_row * p.k_sn)
                                          : (const unsigned char*)((const T*)p.q + b * p.q_sb + h * p.q_sh + unit_row * p.q_sn);
  const uint32_t row_bytes = (uint32_t)(which ? p.k_sn : p.q_sn) * 2;
  const int per_wave = ((len + THREADS - 1) / THREADS) * HA_WAVE;  // rows per wave, whole steps
  const int wave_start = wave * per_wave, wave_end = min(wave_start + per_wave, len);

  // ---- bucket ids, 64 rows a step, the next step's rows in flight ----
  const int m = lane & 15, kg = lane >> 4;
  uint32_t piece[PARTS];
#pragma unroll
  for (int pt = 0; pt < PARTS; ++pt) piece[pt] = pt * 4 + kg < p.qk_pieces ? pt * 64 + 16 * kg : 0;
  vec8 rows[2][2][2][PARTS];  // [buffer][pair of tiles][tile]
  auto load_step = [&](vec8 (&x)[2][2][PARTS], int i0) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int pt = 0; pt < PARTS; ++pt)
        x[t >> 1][t & 1][pt] = *reinterpret_cast<const vec8*>(
            base + (uint32_t)(__umul24((uint32_t)min(i0 + t * 16 + m, real - 1), row_bytes) + piece[pt]));
  };
  load_step(rows[0], wave_start);
  load_step(rows[1], wave_start + HA_WAVE);
#pragma unroll
  for (int k = 0; k < 4; ++k) counts[wave * 256 + k * 64 + lane] = 0;
  if (tid < 256) P::stage((const T*)a.proj, a.num_projs, p.qk_pieces * 8, proj, tid);
  __syncthreads();
  const P projection(proj, a.num_projs, lane);
  auto hash_step = [&](vec8 (&x)[2][2][PARTS], int i0) {
    if (p.qk_pieces < PARTS * 4 || i0 + HA_WAVE > real) {
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int pt = 0; pt < PARTS; ++pt)
          if (pt * 4 + kg >= p.qk_pieces || i0 + t * 16 + m >= real) x[t >> 1][t & 1][pt] = vec8{};
    }
    uint32_t id[2];
#pragma unroll
    for (int pair = 0; pair < 2; ++pair) {
      uint32_t nib[2];
      projection_signs<T, PARTS, 2>(x[pair], projection, a.num_projs, lane, nib);
      id[pair] = bucket_ids(nib[0], nib[1], a.num_projs);
    }
    // the lower halves of the two, side by side
    const uint32_t bucket = __builtin_amdgcn_permlane32_swap(id[0], id[1], false, false)[0];
    if (i0 + lane < wave_end) {
      ids[i0 + lane] = (uint8_t)bucket;
      atomicAdd(&counts[wave * 256 + bucket], 1u);
    }
  };
#pragma unroll 1
  for (int i0 = wave_start; i0 < wave_end; i0 += 2 * HA_WAVE) {
    hash_step(rows[0], i0);
    load_step(rows[0], i0 + 2 * HA_WAVE);
    if (i0 + HA_WAVE < wave_end) hash_step(rows[1], i0 + HA_WAVE);
    load_step(rows[1], i0 + 3 * HA_WAVE);
  }
  __syncthreads();

  // ---- the unit's order, as rank_units_kernel makes it ----
  const bool whole = a.out[which] != nullptr;
  uint32_t total = 0;
  if (tid < 256) {
#pragma unroll
    for (int k = 0; k < WAVES; ++k) total += counts[k * 256 + tid];
    if (!whole) a.hist[which][((int64_t)seq * g.units_per_seq + u) * 256 + tid] = total;
  }
  uint32_t run = block_exclusive_scan(total, wave_totals);
  if (tid < 256) {
#pragma unroll
    for (int k = 0; k < WAVES; ++k) {
      const uint32_t c = counts[k * 256 + tid];
      counts[k * 256 + tid] = run;
      run += c;
    }
  }
  __syncthreads();
#pragma unroll 1
  for (int i0 = wave_start; i0 < wave_end; i0 += HA_WAVE) {
    const int i = i0 + lane;
    const bool valid = i < wave_end;
    const int digit = ids[valid ? i : i0];
    const uint64_t same = match_digit(digit, valid);
    const uint32_t below = rank_below(same);
    if (valid) order[counts[wave * 256 + digit] + below] = (uint16_t)i;
    __builtin_amdgcn_wave_barrier();
    if (valid && below == 0) counts[wave * 256 + digit] += (uint32_t)__popcll(same);
    __builtin_amdgcn_wave_barrier();
  }
  __syncthreads();
  if (whole) {
    int32_t* const out = a.out[which] + (int64_t)seq * len;
    for (int pos = tid; pos < len; pos += THREADS) out[pos] = (int32_t)order[pos];
  } else {
    uint32_t* const out = a.sorted[which] + (int64_t)seq * g.n + unit_row;
    for (int pos = tid; pos < len; pos += THREADS) out[pos] = (uint32_t)ids[order[pos]] << 16 | order[pos];
  }
}

}  // namespace
