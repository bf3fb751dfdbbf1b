// Rewriting of 8-bit matmul operands into the layout the tile kernels read (i8_kernels.hip, f8_kernels.hip).
#include "internal.h"

namespace mi {

typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

// Operands that the tile kernels cannot take as they lie in memory are rewritten once, both in one launch: a [K, N]
// right operand becomes [N, K], a K that is not a whole number of K stages is padded to one, and (for the kernel that
// cannot do it on the way to the matrix cores) unsigned bytes are re-biased to signed.  HBM / launch bound: every
// byte is read and written once, in 16-byte pieces whatever the row alignment (the piece that would reach past its
// row is shifted into place).  1000 x 3000 transposed + 333 x 1000 padded: 6.4 us, both operands; the 64 x 64
// byte-wise transpose it replaces took 10 us for the right operand alone, and the register-staged kernel that took any
// K without padding 182 us for that product where the ring kernel below takes 8.3 (437 us at 333 x 3000 x 1000, now 15.5).

// 16 bytes of a row of `len` bytes from position `at`: bytes past the end are `pad`.  The last piece of a row is the
// row's last 16 bytes shifted into place, so that it costs one request like any other; only a row shorter than that is
// read byte by byte.
__device__ __forceinline__ u32x4 load16_ragged(const uint8_t *row, int64_t at, int64_t len, uint32_t pad4) {
  u32x4 v = {pad4, pad4, pad4, pad4};
  const int64_t over = at + 16 - len;
  if (over <= 0) {
    __builtin_memcpy(&v, row + at, 16);
  } else if (over < 16 && len >= 16) {
    uint64_t q[2];
    __builtin_memcpy(q, row + len - 16, 16);
    const uint64_t pad8 = ((uint64_t)pad4 << 32) | pad4;
    const int s = (int)(over & 7) * 8;  // pad4 is one byte repeated: whole words of it shift in from above
    if (over >= 8) {
      q[0] = q[1];
      q[1] = pad8;
    }
    if (s) {
      q[0] = (q[0] >> s) | (q[1] << (64 - s));
      q[1] = (q[1] >> s) | (pad8 << (64 - s));
    }
    v = u32x4{(uint32_t)q[0], (uint32_t)(q[0] >> 32), (uint32_t)q[1], (uint32_t)(q[1] >> 32)};
  } else if (over < 16) {
    uint32_t w[4] = {pad4, pad4, pad4, pad4};
    for (int i = 0; i < 16 && at + i < len; ++i) {
      const int sh = 8 * (i & 3);
      w[i >> 2] = (w[i >> 2] & ~(0xffu << sh)) | ((uint32_t)row[at + i] << sh);
    }
    v = u32x4{w[0], w[1], w[2], w[3]};
  }
  return v;
}

__device__ __forceinline__ void copy_rows(const OperandCopy &c, int64_t block) {
  const uint32_t cpr = (uint32_t)(c.Kp / 16);
  const int64_t i = block * 256 + threadIdx.x;
  const int64_t r = c.rows * c.Kp < ((int64_t)1 << 36) ? (int64_t)((uint32_t)i / cpr) : i / cpr;  // a 64-bit division costs more than the copy
  if (r >= c.rows)
    return;
  const int64_t k = (i - r * cpr) * 16;
  u32x4 v = load16_ragged(c.src + r * c.K, k, c.K, c.pad4 ^ c.flip4);
#pragma unroll
  for (int e = 0; e < 4; ++e)
    v[e] ^= c.flip4;
  *(u32x4 *)(c.dst + r * c.Kp + k) = v;
}

// 128 k x 128 n per workgroup: a thread reads 16 bytes of each of four consecutive k rows, turns them into 16 dwords
// of four k each (two byte permutes per dword) and leaves those in LDS, from where rows of n go out 128 bytes at a time
__device__ __forceinline__ void copy_transposed(const OperandCopy &c, int64_t block, uint32_t (*tile)[33]) {
  const int tid = threadIdx.x;
  const int64_t nb = (c.rows + 127) / 128;
  const int64_t n0 = block % nb * 128, k0 = block / nb * 128;
  {
    const int nc = tid & 7, kq = tid >> 3;
    const int64_t n = n0 + nc * 16, k = k0 + kq * 4;
    u32x4 w[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const uint32_t raw = c.pad4 ^ c.flip4;
      w[u] = k + u < c.K ? load16_ragged(c.src + (k + u) * c.rows, n, c.rows, raw) : u32x4{raw, raw, raw, raw};
    }
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const uint32_t a = __builtin_amdgcn_perm(w[1][d], w[0][d], 0x05010400u), b = __builtin_amdgcn_perm(w[3][d], w[2][d], 0x05010400u);
      const uint32_t e = __builtin_amdgcn_perm(w[1][d], w[0][d], 0x07030602u), f = __builtin_amdgcn_perm(w[3][d], w[2][d], 0x07030602u);
      tile[nc * 16 + 4 * d + 0][kq] = __builtin_amdgcn_perm(b, a, 0x05040100u) ^ c.flip4;
      tile[nc * 16 + 4 * d + 1][kq] = __builtin_amdgcn_perm(b, a, 0x07060302u) ^ c.flip4;
      tile[nc * 16 + 4 * d + 2][kq] = __builtin_amdgcn_perm(f, e, 0x05040100u) ^ c.flip4;
      tile[nc * 16 + 4 * d + 3][kq] = __builtin_amdgcn_perm(f, e, 0x07060302u) ^ c.flip4;
    }
  }
  __syncthreads();
#pragma unroll
  for (int it = 0; it < 4; ++it) {
    const int r = it * 32 + (tid >> 3), ch = tid & 7;
    const int64_t n = n0 + r, k = k0 + ch * 16;
    if (n < c.rows && k < c.Kp)
      *(u32x4 *)(c.dst + n * c.Kp + k) = u32x4{tile[r][4 * ch], tile[r][4 * ch + 1], tile[r][4 * ch + 2], tile[r][4 * ch + 3]};
  }
}

__global__ __launch_bounds__(256) void operand_copy_kernel(OperandCopy a, OperandCopy b, int64_t b_blocks) {
  __shared__ uint32_t tile[128][33];
  if ((int64_t)blockIdx.x < b_blocks) {
    if (b.transpose)
      copy_transposed(b, blockIdx.x, tile);
    else
      copy_rows(b, blockIdx.x);
  } else {
    copy_rows(a, (int64_t)blockIdx.x - b_blocks);
  }
}

static int64_t copy_blocks(const OperandCopy &c) {
  if (!c.src)
    return 0;
  return c.transpose ? ((c.rows + 127) / 128) * ((c.Kp + 127) / 128) : (c.rows * (c.Kp / 16) + 255) / 256;
}

int operand_copy_launch(const OperandCopy &a, const OperandCopy &b, hipStream_t stream) {
  const int64_t na = copy_blocks(a), nb = copy_blocks(b);
  MI_REQUIRE(na + nb < (1ll << 31) && !a.transpose, MI_BAD_ARGUMENT, "matmul: operands too large");
  if (na + nb == 0)
    return MI_SUCCESS;
  operand_copy_kernel<<<dim3((unsigned)(na + nb)), dim3(256), 0, stream>>>(a, b, nb);
  MI_HIP(hipGetLastError());
  return MI_SUCCESS;
}

}  // namespace mi
