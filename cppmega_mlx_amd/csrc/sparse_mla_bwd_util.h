// Operand reads and products shared by the sparse-MLA backward kernels (gfx950).
#pragma once

#include "common.h"
#include "mfma_util.h"

namespace cm {

__device__ __forceinline__ bf16x8 lds_b128(const unsigned short* p) { return *reinterpret_cast<const bf16x8*>(p); }

// Transposing read: within a group of 16 lanes, lane i points at 4 consecutive elements
// (row i / 4, columns 4 * (i % 4) ..) of a 4 x 16 block and receives column i of rows 0..3.
__device__ __forceinline__ bf16x4 lds_tr16(const unsigned short* p) {
  typedef __attribute__((ext_vector_type(4))) short s16x4;
  const s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)p);
  return __builtin_bit_cast(bf16x4, v);
}
__device__ __forceinline__ bf16x8 join(const bf16x4 a, const bf16x4 b) {
  bf16x8 r;
  r[0] = a[0]; r[1] = a[1]; r[2] = a[2]; r[3] = a[3];
  r[4] = b[0]; r[5] = b[1]; r[6] = b[2]; r[7] = b[3];
  return r;
}
__device__ __forceinline__ bf16x8 zero8() {
  return __builtin_bit_cast(bf16x8, make_uint4(0u, 0u, 0u, 0u));
}

// float16 planes of P and dS are kept at 16 times their value: a float16 is flushed below 6e-8 and overflows above
// 65504, so entries down to 4e-9 survive and |dS| may reach 4000
template <bool F16>
struct PlaneScale {
  static constexpr float up = F16 ? 16.0f : 1.0f, down = F16 ? 1.0f / 16.0f : 1.0f;
};

}  // namespace cm
