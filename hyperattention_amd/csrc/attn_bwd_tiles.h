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

}  // namespace
