// Shared by the dynamic-quantization kernels (dq_kernels.hip: quantizers, few-row and plain products; dq_tile.hip: the
// tiled product): the code families and the conversions of packed codes into matrix operands.
#pragma once
#include "a16_common.h"
#include "internal.h"

namespace mi {

typedef __attribute__((ext_vector_type(4))) int i32x4;

// dq_type families: integer codes (INT4 / INT8), E4M3 codes in 8-bit storage (F8E4M3), E2M1 codes in 4-bit storage (F4)
constexpr int FLAV_INT = 0, FLAV_F8 = 1, FLAV_F4 = 2;

// E2M1 magnitude codes are {0, .5, 1, 1.5, 2, 3, 4, 6}; as E4M3 bytes:
constexpr uint32_t F4_AS_F8_LO = 0x3C383000u;  // 0, 0.5, 1, 1.5
constexpr uint32_t F4_AS_F8_HI = 0x4C484440u;  // 2, 3, 4, 6
__device__ __forceinline__ uint32_t f4_code_as_f8(uint32_t c) {
  const uint32_t m = c & 7u;
  const uint32_t tbl = m < 4 ? F4_AS_F8_LO : F4_AS_F8_HI;
  return ((tbl >> (8 * (m & 3u))) & 0xffu) | ((c & 8u) << 4);
}
// four nibbles held one per byte (0..15 each) -> four E4M3 bytes
__device__ __forceinline__ uint32_t f4x4_as_f8(uint32_t nib) {
  return __builtin_amdgcn_perm(F4_AS_F8_HI, F4_AS_F8_LO, nib & 0x07070707u) | ((nib & 0x08080808u) << 4);
}

// position of element e (0..7) of a packed dword inside the 8 operand bytes it unpacks to: the low-nibble bytes of
// the dword are elements 0,4,1,5 and the high-nibble bytes elements 2,6,3,7 (see unpack below)
__device__ __forceinline__ int dq_slot(int e) { return ((e & 1) << 1) | ((e & 2) << 1) | (e >> 2); }

// nibbles of a packed dword as bytes: low nibbles (elements 0,4,1,5), high nibbles (elements 2,6,3,7)
__device__ __forceinline__ void unpack_bytes(uint32_t d, int &lo, int &hi) {
  lo = (int)(d & 0x0F0F0F0Fu);
  hi = (int)((d >> 4) & 0x0F0F0F0Fu);
}

__device__ __forceinline__ long pack64(uint32_t lo, uint32_t hi) { return (long)(((uint64_t)hi << 32) | lo); }

// eight E4M3 bytes -> eight bf16 values (exact: 4 significant bits into 8).  The fp8 matrix instructions align their
// products to the largest one and drop low bits (about 2^-14 of the group sum here); the bf16 instruction fed with the
// same values adds the exact products with fp32 rounding, which is what the reference's f32 matmul does.
__device__ __forceinline__ bf16x8 f8x8_as_bf16(uint32_t lo, uint32_t hi) {
  typedef __attribute__((ext_vector_type(2))) float f32x2;
  const f32x2 p0 = __builtin_amdgcn_cvt_pk_f32_fp8((int)lo, false), p1 = __builtin_amdgcn_cvt_pk_f32_fp8((int)lo, true);
  const f32x2 p2 = __builtin_amdgcn_cvt_pk_f32_fp8((int)hi, false), p3 = __builtin_amdgcn_cvt_pk_f32_fp8((int)hi, true);
  const u32x4 r = {__builtin_amdgcn_perm(__float_as_uint(p0[1]), __float_as_uint(p0[0]), 0x07060302u),
                   __builtin_amdgcn_perm(__float_as_uint(p1[1]), __float_as_uint(p1[0]), 0x07060302u),
                   __builtin_amdgcn_perm(__float_as_uint(p2[1]), __float_as_uint(p2[0]), 0x07060302u),
                   __builtin_amdgcn_perm(__float_as_uint(p3[1]), __float_as_uint(p3[0]), 0x07060302u)};
  return __builtin_bit_cast(bf16x8, r);
}

// tiled product of quantized fragments (dq_tile.hip)
enum { DQB_W4 = 0, DQB_W8 = 1, DQB_ACT = 2 };  // right operand: packed 4- / 8-bit weight tiles, or quantized activations
struct DqTileArgs {
  const uint8_t *aq;        // left codes [m_blocks][K / 64][64 lanes][16 B]
  const uint8_t *bq;        // right operand, DQB_W4: [n_blocks][K / 128][64][16 B], else [n_blocks][K / 64][64][16 B]
  const float *as_t;        // [m_blocks][G][16]: amax / imax of the left rows
  const int32_t *asum_t;    // [m_blocks][G][16]: sums of their codes (not read for DQB_ACT)
  const void *bscale;       // [n_blocks][G][16]: scale | zero point words, 16-bit scales, or floats (amax / imax)
  const float *nzs;         // DQB_W8: [n_blocks][G][16]
  const float *bias;        // [N] or null
  uint16_t *y;
  float *y32;
  int64_t M, N;
  int halves;               // K / 64
  int G, g;
  int dtype, chip;
};
int dq_tile_launch(const DqTileArgs &a, int b_kind, int flavor, hipStream_t stream);

}  // namespace mi
