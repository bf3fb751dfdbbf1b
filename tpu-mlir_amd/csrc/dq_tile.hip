// The tiled product of dynamic quantization, for many rows: tpu.A16MatMul (A16MatMul.cpp:135-160) on quantized
// activations and packed weights, and tpu.MatMul (MatMul.cpp:560-583) on two quantized activations.  Both operands come
// as matrix fragments (dq_kernels.hip).
//
// 64 x 64 outputs per workgroup, eight waves of 32 x 16.  A wave keeps its outputs in registers over all of K: per
// quantization group it forms the group's sums on the matrix cores and adds  sum * (amax / imax) * scale  to them, in
// group order and with every fp32 operation rounded on its own, which is the reference's order, so the result is its
// result bit for bit (integer codes and E2M1; E4M3 group sums round in the matrix core's order).
//
// What bounds it is that addition: five vector instructions per output and group (zero point, conversion, two products,
// sum), 8.5 us of vector issue for 512 x 4096 x 4096 with groups of 128, and as much again for unpacking and addresses,
// beside 3.4 us of matrix time.  The 16 x 16 blocks of the kernel for few rows re-read both operands and send every
// group's terms through LDS: 77 us there, 25 us here; 2048 rows 268 -> 99 us; two activations 2048 x 128 x 2048
// 33 -> 9.8 us.
// Measured against this shape: four waves of 32 x 32 are 7 % slower up to 512 rows and 8 % faster from 1024 on; four
// waves of 64 x 32 (a quarter fewer instructions, 220 registers) 15 to 30 % slower: occupancy is worth more.
//
// Fragments, row parameters and column parameters of 128 (or 64) k travel through a four-stage LDS ring filled by
// direct-to-LDS loads; a fragment is 16 consecutive bytes of 64 consecutive lanes on both sides, so neither the loads
// nor the reads need a swizzle.
#include "dq_common.h"

#include <type_traits>

#pragma clang fp contract(off)

namespace mi {

typedef const __attribute__((address_space(1))) void *gptr_t;
typedef __attribute__((address_space(3))) void *lptr_t;

constexpr int dqt_waitcnt_vm(int n) { return (n & 0xF) | ((n >> 4) << 14) | 0x0F70; }

constexpr int DQT_NST = 4;                     // ring stages
constexpr int DQT_OUT_STRIDE = 72;             // 16-bit outputs per row of the store tile (16-byte aligned rows)
// A fragments | B fragments | four parameter kinds x groups x 64 rows or columns
constexpr int dqt_a_bytes(int sh) { return 4 * sh * 1024; }
constexpr int dqt_b_bytes(int b, int sh) { return 4 * (b == DQB_W4 ? 1 : sh) * 1024; }
constexpr int dqt_stage(int b, int gps, int sh) { return dqt_a_bytes(sh) + dqt_b_bytes(b, sh) + 4 * gps * 256; }

struct DqTileGrid {
  int tiles_m, tiles_n, per_xcd;
  int m_blocks, n_blocks;
  int stages, stages_per_group;
  unsigned spg_recip;  // stage / stages_per_group == the high word of stage * spg_recip (below 2^16 stages)
};

// a half stage (64 k) of a fragment as the matrix instructions take it
template <int FLAV>
struct DqFrag {
  u32x4 v;
  __device__ __forceinline__ void set(u32x4 x) { v = x; }
};
template <>
struct DqFrag<FLAV_F8> {
  bf16x8 lo, hi;
  __device__ __forceinline__ void set(u32x4 x) {
    lo = f8x8_as_bf16(x[0], x[1]);
    hi = f8x8_as_bf16(x[2], x[3]);
  }
};

// 32 k (q: which half of the fragment) or all 64 (q < 0)
template <int FLAV, int Q, typename ACC>
__device__ __forceinline__ ACC dqt_mfma(const DqFrag<FLAV> &a, const DqFrag<FLAV> &b, ACC c) {
  if constexpr (FLAV == FLAV_INT) {
    if constexpr (Q < 0)
      return __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(i32x4, a.v), __builtin_bit_cast(i32x4, b.v), c, 0, 0, 0);
    else
      return __builtin_amdgcn_mfma_i32_16x16x32_i8(pack64(a.v[2 * Q], a.v[2 * Q + 1]), pack64(b.v[2 * Q], b.v[2 * Q + 1]), c, 0,
                                                   0, 0);
  } else if constexpr (FLAV == FLAV_F4) {
    if constexpr (Q != 1)
      c = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(pack64(a.v[0], a.v[1]), pack64(b.v[0], b.v[1]), c, 0, 0, 0);
    if constexpr (Q != 0)
      c = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(pack64(a.v[2], a.v[3]), pack64(b.v[2], b.v[3]), c, 0, 0, 0);
    return c;
  } else {
    if constexpr (Q != 1)
      c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.lo, b.lo, c, 0, 0, 0);
    if constexpr (Q != 0)
      c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.hi, b.hi, c, 0, 0, 0);
    return c;
  }
}

// B: what the right operand is.  SH: 64-wide halves of K per stage.  GPS: groups per stage (1: a group is one or more
// whole stages).  PIPE: a group is exactly one stage; the sums of a group are added to the outputs while the next
// group's are formed, from the other of two register sets, so that a wave's matrix instructions, its LDS reads and its
// vector instructions do not wait for one another in turn (with several groups in a stage they have each other).
template <int B, int FLAV, int GPS, int SH, bool PIPE>
__global__ __launch_bounds__(512, 2) void dq_tile_kernel(DqTileArgs a, DqTileGrid t) {
  static_assert(B != DQB_W4 || SH == 2, "4-bit tiles are 128 wide");
  static_assert(!PIPE || GPS == 1, "one group per stage");
  using acc_t = typename std::conditional<FLAV == FLAV_INT, i32x4, f32x4>::type;
  constexpr int STAGE = dqt_stage(B, GPS, SH), OFF_B = dqt_a_bytes(SH), OFF_P = OFF_B + dqt_b_bytes(B, SH);
  constexpr int BH = B == DQB_W4 ? 1 : SH;  // kilobytes of a block's right operand per stage
  constexpr bool SUMS = B != DQB_ACT;       // weight zero points meet the sums of the codes
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 2, wn = wave & 3, col = lane & 15, kq = lane >> 4;
  // each XCD gets a contiguous run of the tile order: four tile rows, column by column
  const int L = (blockIdx.x & 7) * t.per_xcd + (blockIdx.x >> 3);
  if (L >= t.tiles_m * t.tiles_n)
    return;
  constexpr int GM = 4;
  const int group = L / (GM * t.tiles_n);
  const int gm = (t.tiles_m - group * GM) < GM ? (t.tiles_m - group * GM) : GM;
  const int in_group = L - group * GM * t.tiles_n;
  const int tm = group * GM + in_group % gm, tn = in_group / gm;

  // request plan: waves 0 .. 3 fetch a block of left fragments each, waves 4 .. 7 a block of right ones and a parameter
  // kind (left scales, left sums, right words, 8-bit scales; a kind that does not exist repeats the one before it).
  // Blocks past the matrix repeat the last one; what comes of them is never stored.  Addresses are a uniform pointer,
  // moved on by stage, plus a lane's 32-bit offset.
  auto clampi = [](int v, int n) { return v < n ? v : n - 1; };
  const bool fetch_a = wave < 4;
  const int w4 = wave & 3;
  const uint8_t *gx = fetch_a ? a.aq + (int64_t)clampi(tm * 4 + w4, t.m_blocks) * a.halves * 1024
                              : a.bq + (int64_t)clampi(tn * 4 + w4, t.n_blocks) * a.halves * (B == DQB_W4 ? 512 : 1024);
  const uint32_t lane16 = lane * 16;
  const bool left_kind = w4 < 2;
  const int pb0 = left_kind ? tm * 4 : tn * 4, pbs = left_kind ? t.m_blocks : t.n_blocks;
  const bool narrow = B == DQB_W8 && w4 == 3;  // 16-bit scales: a dword holds two channels; lanes 32 .. 63 repeat
  const uint8_t *gp;
  if (w4 == 0 || (w4 == 1 && !SUMS))
    gp = (const uint8_t *)a.as_t;
  else if (w4 == 1)
    gp = (const uint8_t *)a.asum_t;
  else if (B == DQB_W8 && w4 == 2)
    gp = (const uint8_t *)a.nzs;
  else
    gp = (const uint8_t *)a.bscale;
  const int gp_step = narrow ? 32 : 64;  // bytes from a group's 16 values to the next group's
  gp += (int64_t)pb0 * a.G * gp_step;
  const uint32_t poff = (uint32_t)(clampi(pb0 + (narrow ? (lane & 31) >> 3 : lane >> 4), pbs) - pb0) * (uint32_t)a.G * (uint32_t)gp_step +
                        (narrow ? (lane & 7) : col) * 4;
  auto issue = [&](int stage, int slot) {
    const int k = stage < t.stages ? stage : t.stages - 1;  // past the end: harmless re-loads of the last stage
    uint8_t *st = lds + slot * STAGE;
    if (fetch_a) {
      const uint8_t *g = gx + (int64_t)k * (SH * 1024);
#pragma unroll
      for (int h = 0; h < SH; ++h)
        __builtin_amdgcn_global_load_lds((gptr_t)(g + h * 1024 + lane16), (lptr_t)(st + (w4 * SH + h) * 1024), 16, 0, 0);
    } else {
      const uint8_t *g = gx + (int64_t)k * (BH * 1024);
#pragma unroll
      for (int h = 0; h < BH; ++h)
        __builtin_amdgcn_global_load_lds((gptr_t)(g + h * 1024 + lane16), (lptr_t)(st + OFF_B + (w4 * BH + h) * 1024), 16, 0, 0);
      // the stage's first group: k * GPS, or k / stages_per_group as a product with its reciprocal
      const int first = PIPE ? k : GPS > 1 ? k * GPS : (int)__umulhi((unsigned)k, t.spg_recip);
      const uint8_t *q = gp + (int64_t)first * gp_step;
#pragma unroll
      for (int p = 0; p < GPS; ++p)
        __builtin_amdgcn_global_load_lds((gptr_t)(q + p * gp_step + poff), (lptr_t)(st + OFF_P + (w4 * GPS + p) * 256), 4, 0, 0);
    }
  };

  constexpr int SETS = PIPE ? 2 : 1;
  float out[2][4];
  acc_t acc[SETS][GPS][2];
  float sc[SETS][GPS];      // of this lane's column
  int zp[SETS][GPS];
  f32x4 as4[SETS][GPS][2];  // of this lane's rows
  i32x4 sum4[SETS][GPS][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      out[i][r] = 0.0f;
  const int64_t m0 = (int64_t)tm * 64, n0 = (int64_t)tn * 64;
  const int64_t n_lane = n0 + wn * 16 + col;
  const float bias = a.bias ? a.bias[n_lane < a.N ? n_lane : a.N - 1] : 0.0f;

  const uint8_t *rd_a = lds + wm * 2 * SH * 1024 + lane * 16, *rd_b = lds + OFF_B + wn * BH * 1024 + lane * 16;
  const uint8_t *rd_row = lds + OFF_P + (wm * 32 + 4 * kq) * 4;
  const uint8_t *rd_col = lds + OFF_P + 2 * GPS * 256 + (wn * 16 + col) * 4;
  const uint8_t *rd_col2 = lds + OFF_P + 3 * GPS * 256 + (wn * 16 + col) * 2;
  u32x4 ra[2][SH], rb[BH];  // the stage's fragments as they lie in LDS
  uint32_t word[GPS];       // and its column parameters
  uint16_t half[GPS];
  auto read_params = [&](int slot, int set) {
#pragma unroll
    for (int p = 0; p < GPS; ++p) {
      word[p] = *(const uint32_t *)(rd_col + slot * STAGE + p * 256);
      if constexpr (B == DQB_W8)
        half[p] = *(const uint16_t *)(rd_col2 + slot * STAGE + p * 256);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        as4[set][p][i] = *(const f32x4 *)(rd_row + slot * STAGE + p * 256 + i * 64);
        if constexpr (SUMS)
          sum4[set][p][i] = *(const i32x4 *)(rd_row + slot * STAGE + (GPS + p) * 256 + i * 64);
      }
    }
  };
  auto read_fragments = [&](int slot) {
#pragma unroll
    for (int h = 0; h < BH; ++h)
      rb[h] = *(const u32x4 *)(rd_b + slot * STAGE + h * 1024);
#pragma unroll
    for (int h = 0; h < SH; ++h)
#pragma unroll
      for (int i = 0; i < 2; ++i)
        ra[i][h] = *(const u32x4 *)(rd_a + slot * STAGE + (i * SH + h) * 1024);
  };
  // the starting values of a group's sums: -zp * sum(codes) for integer codes, zero otherwise
  auto begin_group = [&](int set) {
#pragma unroll
    for (int p = 0; p < GPS; ++p) {
      if constexpr (B == DQB_ACT) {
        sc[set][p] = __uint_as_float(word[p]);
        zp[set][p] = 0;
      } else if constexpr (B == DQB_W4) {
        const uint16_t h = (uint16_t)(word[p] >> 16);
        sc[set][p] = a.dtype == MI_DT_F16 ? f16_bits_to_f32(h) : bf16_bits_to_f32(h);
        zp[set][p] = (int)(word[p] & 0xffu);
      } else {
        const float s = a.dtype == MI_DT_F16 ? f16_bits_to_f32(half[p]) : bf16_bits_to_f32(half[p]);
        // exact: the word is -(zp') * scale without rounding; integer codes were flipped to signed, E4M3 bytes not
        constexpr int OFFSET = FLAV == FLAV_INT ? 128 : 0;
        zp[set][p] = (s != 0.0f ? (int)rintf(-__uint_as_float(word[p]) / s) : OFFSET) - OFFSET;
        sc[set][p] = s;
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if constexpr (SUMS && FLAV == FLAV_INT)
            acc[set][p][i][r] = __mul24(-zp[set][p], sum4[set][p][i][r]);  // both below 2^23
          else
            acc[set][p][i][r] = 0;
        }
    }
  };
  auto multiply = [&](int set) {
    DqFrag<FLAV> fa[2][SH], fb[SH];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int h = 0; h < SH; ++h)
        fa[i][h].set(ra[i][h]);
    if constexpr (B == DQB_W4) {
      uint32_t lo[4], hi[4];
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        lo[d] = rb[0][d] & 0x0F0F0F0Fu;
        hi[d] = (rb[0][d] >> 4) & 0x0F0F0F0Fu;
        if constexpr (FLAV == FLAV_F4) {
          lo[d] = f4x4_as_f8(lo[d]);
          hi[d] = f4x4_as_f8(hi[d]);
        }
      }
      fb[0].set(u32x4{lo[0], hi[0], lo[1], hi[1]});
      fb[SH - 1].set(u32x4{lo[2], hi[2], lo[3], hi[3]});
    } else {
#pragma unroll
      for (int h = 0; h < SH; ++h) {
        u32x4 w = rb[h];
        if constexpr (B == DQB_W8 && FLAV == FLAV_INT) {
#pragma unroll
          for (int d = 0; d < 4; ++d)
            w[d] ^= 0x80808080u;
        }
        fb[h].set(w);
      }
    }
#pragma unroll
    for (int h = 0; h < SH; ++h)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        if constexpr (GPS == 2 * SH) {  // 32-wide groups: one per half of the fragment
          acc[set][2 * h][i] = dqt_mfma<FLAV, 0>(fa[i][h], fb[h], acc[set][2 * h][i]);
          acc[set][2 * h + 1][i] = dqt_mfma<FLAV, 1>(fa[i][h], fb[h], acc[set][2 * h + 1][i]);
        } else {
          constexpr int STEP = GPS == SH && GPS > 1 ? 1 : 0;  // 64-wide groups: one per fragment
          acc[set][h * STEP][i] = dqt_mfma<FLAV, -1>(fa[i][h], fb[h], acc[set][h * STEP][i]);
        }
      }
  };
  auto add_group = [&](int set, bool first) {
#pragma unroll
    for (int p = 0; p < GPS; ++p)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float v = (float)acc[set][p][i][r];  // integer sums are below 2^24 (checked on the host): exact
          if constexpr (SUMS && FLAV != FLAV_INT)
            v = zp[set][p] != 0 ? v - (float)zp[set][p] * __int_as_float(sum4[set][p][i][r]) : v;
          v = v * as4[set][p][i][r];  // A16MatMul.cpp:153-156, MatMul.cpp:577-581: left to right
          v = v * sc[set][p];
          out[i][r] = out[i][r] + v;
        }
        if (first && p == 0 && a.bias)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            out[i][r] = out[i][r] + bias;  // A16MatMul.cpp:157-159, after the first group
      }
  };
  auto arrive = [&](int kt, int slot) {  // stage kt, in `slot`, is complete and the slot before it free: request into that
    if (fetch_a)
      __builtin_amdgcn_s_waitcnt(dqt_waitcnt_vm((DQT_NST - 2) * SH));
    else
      __builtin_amdgcn_s_waitcnt(dqt_waitcnt_vm((DQT_NST - 2) * (BH + GPS)));
    __builtin_amdgcn_s_barrier();
    issue(kt + DQT_NST - 1, (slot + DQT_NST - 1) % DQT_NST);
  };
#pragma unroll
  for (int s = 0; s < DQT_NST - 1; ++s)
    issue(s, s);
  if constexpr (PIPE) {
    for (int kt = 0; kt < t.stages; kt += 4) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {  // slot u, register set u % 2
        if (kt + u >= t.stages)
          break;
        arrive(kt + u, u);
        // the stage's LDS reads are on their way while the previous group is added, and its matrix instructions
        // finish under the next stage's wait
        read_fragments(u);
        read_params(u, u & 1);
        __builtin_amdgcn_sched_barrier(0);
        if (kt + u > 0)
          add_group((u & 1) ^ 1, kt + u == 1);
        __builtin_amdgcn_sched_barrier(0);
        begin_group(u & 1);
        multiply(u & 1);
      }
    }
    if (t.stages & 1)
      add_group(0, t.stages == 1);
    else
      add_group(1, false);
  } else {
    int left = t.stages_per_group;
    bool first = true;
    for (int kt = 0; kt < t.stages; ++kt) {
      const int slot = kt % DQT_NST;
      arrive(kt, slot);
      read_fragments(slot);
      if (left == t.stages_per_group) {
        read_params(slot, 0);
        begin_group(0);
      }
      multiply(0);
      if (--left == 0) {
        left = t.stages_per_group;
        add_group(0, first);
        first = false;
      }
    }
  }
  __builtin_amdgcn_s_waitcnt(dqt_waitcnt_vm(0));  // the re-loads issued past the end
  __builtin_amdgcn_s_barrier();                   // every wave is done reading the ring

  // 16-bit outputs leave through LDS as whole 128-byte rows of the tile
  uint16_t *tile = (uint16_t *)lds + (wm * 32 + 4 * kq) * DQT_OUT_STRIDE + wn * 16 + col;
  auto to_tile = [&](auto round16) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        tile[(i * 16 + r) * DQT_OUT_STRIDE] = round16(out[i][r]);
  };
  if (a.chip == MI_CHIP_CV18XX && a.dtype == MI_DT_F16)
    to_tile([](float v) { return round_out16<MI_DT_F16, MI_CHIP_CV18XX>(v); });
  else if (a.chip == MI_CHIP_CV18XX)
    to_tile([](float v) { return round_out16<MI_DT_BF16, MI_CHIP_CV18XX>(v); });
  else if (a.dtype == MI_DT_F16)
    to_tile([](float v) { return round_out16<MI_DT_F16, MI_CHIP_BM168X>(v); });
  else
    to_tile([](float v) { return round_out16<MI_DT_BF16, MI_CHIP_BM168X>(v); });
  if (a.y32) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t m = m0 + wm * 32 + i * 16 + 4 * kq + r;
        if (m < a.M && n_lane < a.N)
          a.y32[m * a.N + n_lane] = out[i][r];
      }
  }
  __syncthreads();
  const int row = tid >> 3, c = (tid & 7) * 8;
  const int64_t m = m0 + row, n = n0 + c;
  if (m >= a.M)
    return;
  uint16_t *dst = a.y + m * a.N + n;
  const uint16_t *src = (const uint16_t *)lds + row * DQT_OUT_STRIDE + c;
  const u32x4 v = *(const u32x4 *)src;
  if (n + 8 <= a.N) {
    __builtin_memcpy(dst, &v, 16);
  } else {
    for (int e = 0; e < 8; ++e)
      if (n + e < a.N)
        dst[e] = src[e];
  }
}

int dq_tile_launch(const DqTileArgs &a, int b_kind, int flavor, hipStream_t stream) {
  DqTileGrid t;
  t.m_blocks = (int)((a.M + 15) / 16);
  t.n_blocks = (int)((a.N + 15) / 16);
  t.tiles_n = (t.n_blocks + 3) / 4;
  t.tiles_m = (t.m_blocks + 3) / 4;
  MI_REQUIRE((int64_t)t.tiles_m * t.tiles_n < (1ll << 30), MI_BAD_ARGUMENT, "dynamic quantization: too many outputs");
  t.per_xcd = (t.tiles_m * t.tiles_n + 7) / 8;
  // 128 k per stage where K and the groups divide into such stages, 64 otherwise (two activations only)
  const bool wide = a.halves % 2 == 0 && (a.g == 32 || a.g == 64 || a.g % 128 == 0);
  const int sh = wide ? 2 : 1;
  const int gps = a.g >= 64 * sh ? 1 : 64 * sh / a.g;
  t.stages = a.halves / sh;
  t.stages_per_group = a.g >= 64 * sh ? a.g / (64 * sh) : 1;
  t.spg_recip = t.stages_per_group > 1 ? (unsigned)((1ull << 32) / t.stages_per_group + 1) : 0;
  const dim3 grid((unsigned)(t.per_xcd * 8));
  const bool pipe = gps == 1 && t.stages_per_group == 1;
#define MI_DQT(B, FLAV, GPS, SH, PIPE)                                                                        \
  if (gps == GPS && sh == SH && pipe == PIPE) {                                                               \
    static LdsLimitOnce lds_limit;                                                                            \
    lds_limit.ensure((const void *)dq_tile_kernel<B, FLAV, GPS, SH, PIPE>, 160 * 1024);                       \
    dq_tile_kernel<B, FLAV, GPS, SH, PIPE><<<grid, dim3(512), DQT_NST * dqt_stage(B, GPS, SH), stream>>>(a, t); \
  }
#define MI_DQT_WIDE(B, FLAV)                                                                                  \
  MI_DQT(B, FLAV, 1, 2, true)                                                                                 \
  MI_DQT(B, FLAV, 1, 2, false)                                                                                \
  MI_DQT(B, FLAV, 2, 2, false)                                                                                \
  MI_DQT(B, FLAV, 4, 2, false)
#define MI_DQT_ANY(FLAV)                                                                                      \
  MI_DQT_WIDE(DQB_ACT, FLAV)                                                                                  \
  MI_DQT(DQB_ACT, FLAV, 1, 1, true)                                                                           \
  MI_DQT(DQB_ACT, FLAV, 1, 1, false)                                                                          \
  MI_DQT(DQB_ACT, FLAV, 2, 1, false)
  if (b_kind == DQB_W4 && flavor == FLAV_INT) {
    MI_DQT_WIDE(DQB_W4, FLAV_INT)
  } else if (b_kind == DQB_W4) {
    MI_DQT_WIDE(DQB_W4, FLAV_F4)
  } else if (b_kind == DQB_W8 && flavor == FLAV_INT) {
    MI_DQT_WIDE(DQB_W8, FLAV_INT)
  } else if (b_kind == DQB_W8) {
    MI_DQT_WIDE(DQB_W8, FLAV_F8)
  } else if (flavor == FLAV_INT) {
    MI_DQT_ANY(FLAV_INT)
  } else if (flavor == FLAV_F4) {
    MI_DQT_ANY(FLAV_F4)
  } else {
    MI_DQT_ANY(FLAV_F8)
  }
#undef MI_DQT
#undef MI_DQT_WIDE
#undef MI_DQT_ANY
  MI_HIP(hipGetLastError());
  return MI_SUCCESS;
}

}  // namespace mi
