// LDS tile helpers shared by the attention kernels (attn.hip, xattn_mfma.hip).
#pragma once
#include "md_common.h"

constexpr int kVSub = 1056;  // bytes per [32 keys][16 d] V sub-tile (+32 B pad: conflict-free ds_write_b128)

typedef bf16x8 bf16x8_a8 __attribute__((aligned(8)));      // of rows that start at 8 bytes

// Place of 16-byte piece `ch` in row `row` of an LDS image of rows of N pieces: 16 rows' pieces of one number lie in different banks.
template <int N>
__device__ __forceinline__ int lds_place(int ch, int row) {
    return ch ^ (N % 16 == 0 ? row & 15 : N % 8 == 0 ? (row >> 1) & 7 : (row >> 2) & 3);
}
__device__ __forceinline__ bf16x8 lds_read_b128(const unsigned char* p) {
    return *reinterpret_cast<const bf16x8*>(p);
}
__device__ __forceinline__ bf16x4 lds_read_tr(const unsigned char* p) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
        (__attribute__((address_space(3))) bf16x4*)(p));
}
