// What the kernels that hold a LayerNorm-quantiser share: elements of a row as they lie in memory, the rounding of a stored
// value, and the sums in the reference order (chunk c, elements 4c .. 4c + 3, belongs to lane c % 256 of four waves, a lane adds
// in ascending order, a wave by a xor butterfly, the four waves left to right).
#pragma once
#include <type_traits>

#include "ti_common.h"

namespace ti {

// s of this lane and of the lane whose number differs in one bit, added; bits 5, 4, .. 0 in turn.  All on the vector ALU: LDS
// permutes are six dependent round trips, twice a row (24 rows of 4096 fp16: 4.7 -> 4.4 us).
__device__ __forceinline__ float wave_butterfly_sum(float s) {
  // a swap of a value with a copy of itself leaves this lane's value in one result and its partner's in the other
  auto swapped = [](float v, auto swap) {
    auto both = swap(__builtin_bit_cast(unsigned, v), __builtin_bit_cast(unsigned, v));
    const unsigned a = both[0], b = both[1];  // plain values: the casts must not see vector elements
    return __builtin_bit_cast(float, a) + __builtin_bit_cast(float, b);
  };
  s = swapped(s, [](unsigned a, unsigned b) { return __builtin_amdgcn_permlane32_swap(a, b, false, false); });
  s = swapped(s, [](unsigned a, unsigned b) { return __builtin_amdgcn_permlane16_swap(a, b, false, false); });
  // rotations inside a row of 16: by 8 the partner of bit 3; by 4 that of bit 2, as lanes 8 apart hold the same by then
  s = s + __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, s), 0x128, 0xf, 0xf, true));
  s = s + __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, s), 0x124, 0xf, 0xf, true));
  s = s + __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, s), 0x4E, 0xf, 0xf, true));
  s = s + __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, s), 0xB1, 0xf, 0xf, true));
  return s;
}

// `red`: four floats that nothing else uses
__device__ __forceinline__ float block_sum_256(float s, float* red) {
  s = wave_butterfly_sum(s);
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) red[wave] = s;
  __syncthreads();
  return ((red[0] + red[1]) + red[2]) + red[3];
}

typedef _Float16 v4h __attribute__((ext_vector_type(4)));

// four consecutive elements as they lie in memory; chunk c of a row as fp32 / stored from fp32
template <class T> struct Chunk;
template <> struct Chunk<float> { typedef v4f type; };
template <> struct Chunk<_Float16> { typedef v4h type; };
__device__ __forceinline__ v4f to_f32(v4f v) { return v; }
__device__ __forceinline__ v4f to_f32(v4h h) { return v4f{(float)h[0], (float)h[1], (float)h[2], (float)h[3]}; }
__device__ __forceinline__ v4f load4(const float* row, int c) { return reinterpret_cast<const v4f*>(row)[c]; }
__device__ __forceinline__ v4f load4(const _Float16* row, int c) {
  const v4h h = reinterpret_cast<const v4h*>(row)[c];
  return v4f{(float)h[0], (float)h[1], (float)h[2], (float)h[3]};
}
__device__ __forceinline__ void store4(float* row, int c, v4f v) { reinterpret_cast<v4f*>(row)[c] = v; }
__device__ __forceinline__ void store4(_Float16* row, int c, v4f v) {
  reinterpret_cast<v4h*>(row)[c] = v4h{(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
}
// The value a tensor of element type T holds after the fp32 value `x` is stored to it (round to nearest even
// for fp16).  The empty asm keeps the fp32 result of the preceding operation a value of its own: without it the
// compiler merges an fma and the conversion into one mixed-precision instruction that rounds the exact sum
// straight to fp16, which differs from "fp32 operation, then conversion" when the fp32 result is a tie.
template <class T>
__device__ __forceinline__ float as_stored(float x) {
  if constexpr (sizeof(T) == 2) asm volatile("" : "+v"(x));
  return (float)(T)x;
}

__device__ __forceinline__ int pack_s8x4(float y0, float y1, float y2, float y3) {
  unsigned b0 = (unsigned char)(int8_t)rne_s8(y0);
  unsigned b1 = (unsigned char)(int8_t)rne_s8(y1);
  unsigned b2 = (unsigned char)(int8_t)rne_s8(y2);
  unsigned b3 = (unsigned char)(int8_t)rne_s8(y3);
  return (int)(b0 | (b1 << 8) | (b2 << 16) | (b3 << 24));
}

}  // namespace ti
