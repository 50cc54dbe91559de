// Signs of the random projections of rows, 16 rows at a time on the matrix cores: shared by the hash launch (lsh_hash.hip) and
// by the workgroups that hash and rank beside the exact causal kernel (unit_ranking.h).  What decides a sign is the exact dot
// product: fp32 MFMA sums within their error bound of zero are redone in fp64 (lsh_hash.hip has the definition and the bound).
#pragma once

#include "ha_common.h"

namespace {

template <typename T>
struct HashMfma;
template <>
struct HashMfma<f16_t> {
  static __device__ __forceinline__ f32x4 run(f16x8 a, f16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};
template <>
struct HashMfma<bf16_t> {
  static __device__ __forceinline__ f32x4 run(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};

// the bits of c's signs, c[0]'s lowest
__device__ __forceinline__ uint32_t sign_bits(f32x4 c) {
  uint32_t bits = 0;
#pragma unroll
  for (int i = 3; i >= 0; --i) {
    const float ci = c[i];
    bits = __builtin_amdgcn_alignbit(bits, __builtin_bit_cast(uint32_t, ci), 31);
  }
  return bits;
}

// The projection matrix (d_real rows of r <= 16) as MFMA operands: in LDS transposed, projection j's elements side by side
// from j * PITCH on, zeros for the missing rows and projections.
template <typename T, int PARTS>
struct Projection {
  typedef typename ElemTraits<T>::vec8 vec8;
  static constexpr int D = PARTS * 32;
  static constexpr int PITCH = D + 8;  // 16 bytes more, so that the 16 projections' pieces lie on different banks
  static constexpr int LDS_BYTES = 16 * PITCH * (int)sizeof(T);

  const T* lds;
  vec8 pf[PARTS], pa[PARTS];  // P and |P| for every part: slot m, group kg holds P[part*32 + 8*kg + e][m]
  f32x4 c_first;              // a slot past the last projection starts at -1 and its products are zeros: never in doubt

  // by the first 256 threads; a barrier belongs between this and the constructor
  static __device__ __forceinline__ void stage(const T* proj, int r, int d_real, T* lds, int tid) {
    const int j = tid & 15, k0 = tid >> 4;
    // selects, not branches: behind one the compiler waits for the loads ahead of it, the rows'
    T v[D / 16];
    bool wanted[D / 16];
#pragma unroll
    for (int i = 0; i < D / 16; ++i) {
      const int k = k0 + 16 * i, at = __mul24(k, r) + j;
      wanted[i] = (j < r) & (k < d_real);
      v[i] = proj[wanted[i] ? at : 0];
    }
#pragma unroll
    for (int i = 0; i < D / 16; ++i) lds[j * PITCH + k0 + 16 * i] = wanted[i] ? v[i] : (T)0.f;
  }
  __device__ __forceinline__ Projection(const T* staged, int r, int lane) : lds(staged) {
    const int m = lane & 15, kg = lane >> 4;
#pragma unroll
    for (int pt = 0; pt < PARTS; ++pt) {
      pf[pt] = *reinterpret_cast<const vec8*>(&lds[m * PITCH + pt * 32 + 8 * kg]);
      pa[pt] = __builtin_bit_cast(vec8, __builtin_bit_cast(u32x4, pf[pt]) & 0x7fff7fffu);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) c_first[i] = 4 * kg + i < r ? 0.f : -1.f;
  }
};

// Signs of GROUP tiles of 16 rows: lane (m = lane % 16, kg = lane / 16) holds elements 32*part + 8*kg .. +7 of row m of each and
// gets the bits of slots 4*kg .. +3 of that row, set where the projection is negative.
template <typename T, int PARTS, int GROUP>
__device__ __forceinline__ void projection_signs(const typename ElemTraits<T>::vec8 (&xf)[GROUP][PARTS], const Projection<T, PARTS>& p,
                                                 int r, int lane, uint32_t (&nib)[GROUP]) {
  typedef typename ElemTraits<T>::vec8 vec8;
  typedef Projection<T, PARTS> P;
  const int kg = lane >> 4;
  const float tol = (float)(P::D + 8) * 4.76837158203125e-07f;  // 2 * (d + 8) * 2^-23
  f32x4 c[GROUP], ca[GROUP];
#pragma unroll
  for (int u = 0; u < GROUP; ++u) {
    c[u] = p.c_first;
    ca[u] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
#pragma unroll
  for (int pt = 0; pt < PARTS; ++pt)
#pragma unroll
    for (int u = 0; u < GROUP; ++u) {
      const vec8 abs_x = __builtin_bit_cast(vec8, __builtin_bit_cast(u32x4, xf[u][pt]) & 0x7fff7fffu);
      c[u] = HashMfma<T>::run(p.pf[pt], xf[u][pt], c[u]);
      ca[u] = HashMfma<T>::run(p.pa[pt], abs_x, ca[u]);
    }
#pragma unroll
  for (int u = 0; u < GROUP; ++u) {
    nib[u] = sign_bits(c[u]);
    // what is left of |projection| above the bound of its error; a NaN stays one
    float left[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) left[i] = __builtin_fmaf(-tol, ca[u][i], __builtin_fabsf(c[u][i]));
    const float least = __builtin_elementwise_minimum(__builtin_elementwise_minimum(left[0], left[1]),
                                                      __builtin_elementwise_minimum(left[2], left[3]));
    if (__builtin_expect(__any(!(least > 0.f)), false)) {
      uint32_t unsure = 0;
#pragma unroll
      for (int i = 0; i < 4; ++i) unsure |= left[i] > 0.f ? 0u : 1u << (4 * kg + i);
      for (int jj = 0; jj < r; ++jj) {
        if (!__any((unsure >> jj) & 1u)) continue;
        // this lane's elements of row m, then the sum over the four lanes that share the row
        double part = 0.0;
#pragma unroll
        for (int pt = 0; pt < PARTS; ++pt) {
          // converted where they are used (ahead of the loop, the doubles took 64 registers that are waves in flight)
          u32x4 raw = __builtin_bit_cast(u32x4, xf[u][pt]);
          asm volatile("" : "+v"(raw));
          const vec8 x = __builtin_bit_cast(vec8, raw);
          const vec8 p8 = *reinterpret_cast<const vec8*>(&p.lds[jj * P::PITCH + pt * 32 + 8 * kg]);
#pragma unroll
          for (int e = 0; e < 8; ++e)
            part = __builtin_fma((double)ha_to_float(x[e]), (double)ha_to_float(p8[e]), part);
          __builtin_amdgcn_sched_barrier(0);
        }
        part += __shfl_xor(part, 16);
        part += __shfl_xor(part, 32);
        const uint32_t bit = 1u << (jj & 3);
        if (kg == jj >> 2) nib[u] = part > 0.0 ? nib[u] & ~bit : nib[u] | bit;
      }
    }
  }
}

// Bucket ids of two tiles from their signs, rows in order over the lanes 0 .. 31 (the upper half holds copies of use to nobody):
// a row's nibbles meet in one lane.  After the swap groups of 16 lanes hold (tile 0, tile 1) of slots 0..3 | 8..11, and of slots
// 4..7 | 12..15.
__device__ __forceinline__ uint32_t bucket_ids(uint32_t tile0, uint32_t tile1, int r) {
  const auto sw = __builtin_amdgcn_permlane16_swap(tile0, tile1, false, false);
  uint32_t bin = sw[0] | sw[1] << 4;
  if (r > 8) bin |= (uint32_t)__shfl_xor((int)bin, 32) << 8;  // of use in the lower half of the lanes
  bin = ~bin & ((1u << r) - 1u);
  return bin ^ (bin >> 1);
}

}  // namespace
