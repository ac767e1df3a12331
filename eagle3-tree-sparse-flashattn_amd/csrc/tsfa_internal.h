// Internal declarations shared by the libtsfa HIP sources (gfx950 only).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/tsfa.h"
#include "tsfa_plan.h"

namespace tsfa {

// ------------------------------------------------------------------ vectors
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef short i16x8 __attribute__((ext_vector_type(8)));

#define TSFA_LDS __attribute__((address_space(3)))

// Per-dtype MFMA 32x32x16 (fp32 accumulate).  Lane layouts (verified on
// gfx950): A[m][k] lane m + 32*(k/8), element k%8; B[k][n] lane n + 32*(k/8),
// element k%8; C[m][n] lane n + 32*((m/4)%2), element 4*(m/8) + m%4.
template <typename T> struct Mma;
template <> struct Mma<__bf16> {
  typedef bf16x8 vec8;
  __device__ static inline f32x16 run(vec8 a, vec8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
};
template <> struct Mma<_Float16> {
  typedef f16x8 vec8;
  __device__ static inline f32x16 run(vec8 a, vec8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
};

// ------------------------------------------------------------- mask packing
// Nonzero bytes of x (4 mask bytes, first byte lowest) as bits 0-3: the
// high bit of each byte of (x & 0x7f7f7f7f) + 0x7f7f7f7f | x is set iff the
// byte is nonzero; the multiply moves bits 7, 15, 23, 31 to 28..31 (its other
// partial products land on distinct positions below 28, so no carry reaches
// them).
__device__ inline uint32_t nonzero_nibble(uint32_t x) {
  const uint32_t t = ((((x & 0x7f7f7f7fu) + 0x7f7f7f7fu) | x) & 0x80808080u);
  return (t * 0x00204081u) >> 28;
}

// 32 mask bytes from p (any alignment) as bits.
__device__ inline uint32_t pack32(const uint8_t* p) {
  uint32_t x[8];
  __builtin_memcpy(x, p, 32);
  uint32_t word = 0;
#pragma unroll
  for (int i = 0; i < 8; ++i) word |= nonzero_nibble(x[i]) << (4 * i);
  return word;
}

// Columns [c0, c0 + 32) of a mask row of n columns as bits, columns past its
// end 0 (c0 < n).  A cut last word takes the 32 bytes that end at column n; a
// row of fewer than 32 columns comes whole, 8 bytes at a time (32 loads at
// once spill the fp32 head_dim 256 kernel).
__device__ inline uint32_t mask_word(const uint8_t* row, int c0, int n) {
  const int valid = min(32, n - c0);
  if (c0 + valid >= 32) return pack32(row + c0 + valid - 32) >> (32 - valid);
  uint32_t word = 0;
  for (int i0 = 0; i0 < n; i0 += 8) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int c = min(i0 + i, n - 1);  // past the end: the last byte again
      word |= (uint32_t)(row[c] != 0) << c;
    }
  }
  return word >> c0;
}

// ---------------------------------------------------------- host utilities
int device_cu_count(int* out);            // cached per device
int device_max_lds_per_block(int* out);   // cached per device


}  // namespace tsfa
