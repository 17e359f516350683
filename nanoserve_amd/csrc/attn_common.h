// Device helpers shared by the matrix-core attention kernels (head size 128): buffer-to-LDS loads of
// K / V rows and the transposed LDS read of V.
#pragma once
#include "w4_common.h"

namespace ns {

typedef __attribute__((__vector_size__(2 * sizeof(uint32_t)))) uint32_t u32x2_t;
typedef short s16x4_t __attribute__((ext_vector_type(4)));

// 16 bytes per lane into LDS at dst + 16 lane (a plain function: the builtin inside a lambda of a
// kernel template keeps the host pass from emitting the launch stub).
__device__ __forceinline__ void attn_lds_load16(__amdgpu_buffer_rsrc_t r, uint16_t* dst, uint32_t voff,
                                                uint32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 16, voff,
                                           soff, 0, 0);
}

// ds_read_b64_tr_b16: the 16 lanes of a group read a 4 x 16 block of 16-bit values, lane l at row
// l / 4, columns 4 (l % 4) .. + 3, and lane l receives column l, rows 0 .. 3.
__device__ __forceinline__ u32x2_t lds_read_tr16(const uint16_t* p) {
  return __builtin_bit_cast(
      u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                   (__attribute__((address_space(3))) s16x4_t*)const_cast<uint16_t*>(p)));
}

}  // namespace ns
