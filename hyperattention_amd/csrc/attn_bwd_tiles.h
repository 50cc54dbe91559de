// Layout of the tiles that the attention backward kernels read both ways, and their transposing operand read.
#pragma once

#include "attn_tiles.h"

namespace {

// LDS layout of a streamed tile: row-major [64][D] 2-byte elements, the 16-byte pieces of a row XOR-ed
// with a function of the row number chosen so that BOTH ways the tile is read are free of bank
// conflicts (the LDS serves 16 lanes, 64 banks of 4 bytes, at a time):
//   row reads (ds_read_b128): 16 lanes read the same piece of 16 consecutive rows -> the 16 rows
//     must land in 16 different 16-byte slots of the 256-byte bank window;
//   transposing reads (ds_read_b64_tr_b16): 16 lanes read 2 adjacent pieces of 4 consecutive rows
//     (starting at a multiple of 4) -> the four pairs must differ in a bit above the lowest.
// d = 64 (a row is half a bank window, so rows of equal parity compete for 8 slots): the bits 1,2,3
// of the row number, in reversed order.  d = 128 (16 slots per row): the low four bits of the row
// number with the two pairs of bits exchanged.
template <int D>
__device__ __forceinline__ int bwd_swizzle(int row) {
  if (D == 64) return (((row >> 1) & 1) << 2) | (((row >> 2) & 1) << 1) | ((row >> 3) & 1);
  return ((row & 3) << 2) | ((row >> 2) & 3);
}
template <int D>
__device__ __forceinline__ int bwd_tile_offset(int row, int piece) {
  return row * D * 2 + ((piece ^ bwd_swizzle<D>(row)) << 4);
}

// 8 streamed rows x 1 column, transposed by the LDS unit: rows 0..3 and 8..11 (+4 for the upper lane
// half) relative to the row the offsets were computed for
template <typename T>
__device__ __forceinline__ typename ElemTraits<T>::vec8 bwd_read_tr(const unsigned char* tile, int off_lo, int off_hi) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  typedef short s16x8 __attribute__((ext_vector_type(8)));
  typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
  const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(tile + off_lo));
  const s16x4 hi8 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(tile + off_hi));
  const s16x8 both = __builtin_shufflevector(lo, hi8, 0, 1, 2, 3, 4, 5, 6, 7);
  return __builtin_bit_cast(typename ElemTraits<T>::vec8, both);
#else
  return typename ElemTraits<T>::vec8{};
#endif
}

// ---- LDS by address: kernels whose whole LDS is one dynamic block from address 0 on ----
// A barrier that waits for this wave's LDS operations but not for its loads and stores in memory
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// What lanes of one wave write to LDS and others read: the wave's LDS operations stay in this order
__device__ __forceinline__ void wave_lds_order() { asm volatile("" ::: "memory"); }

template <typename V>
__device__ __forceinline__ V lds_get(uint32_t address) {
#if defined(__HIP_DEVICE_COMPILE__)
  return *(const __attribute__((address_space(3))) V*)address;
#else
  return V{};
#endif
}
template <typename V>
__device__ __forceinline__ void lds_put(uint32_t address, V value) {
#if defined(__HIP_DEVICE_COMPILE__)
  *(__attribute__((address_space(3))) V*)address = value;
#endif
}
// 8 rows x 1 column, transposed by the LDS unit, from two blocks of 4 rows
template <typename T>
__device__ __forceinline__ typename ElemTraits<T>::vec8 lds_get_tr(uint32_t lo, uint32_t hi) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  typedef short s16x8 __attribute__((ext_vector_type(8)));
  typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
  const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)lo), b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)hi);
  return __builtin_bit_cast(typename ElemTraits<T>::vec8, (s16x8)__builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
#else
  return typename ElemTraits<T>::vec8{};
#endif
}

// 16 bytes per lane from base + offset to LDS at lds_dst + 16 * lane.  In assembly: the compiler, which does not know what
// such a load writes, would wait for it before LDS accesses that have nothing to do with it.  It also does not count it, so
// a wait that it puts in for one of its own loads waits for these loads too if they were issued later.
__device__ __forceinline__ void load_to_lds(const unsigned char* base, uint32_t offset, uint32_t lds_dst) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" 
               ::"s"(__builtin_amdgcn_readfirstlane(lds_dst)), "v"(offset), "s"(base) : "memory", "m0");
#endif
}

// As load_to_lds, 4 bytes per lane to lds_dst + 4 * lane
__device__ __forceinline__ void load_to_lds_4(const unsigned char* base, uint32_t offset, uint32_t lds_dst) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2"
               ::"s"(__builtin_amdgcn_readfirstlane(lds_dst)), "v"(offset), "s"(base) : "memory", "m0");
#endif
}

}  // namespace
