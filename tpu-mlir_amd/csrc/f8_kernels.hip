// tpu.MatMul on F8E4M3 operands with the F8 output requantization, for gfx950:
//   acc[m,n] = sum_k A[m,k] * B[n,k] + bias[n]          (E4M3 codes in, fp32 out of v_mfma_f32_32x32x64_f8f6f4)
//   v        = relu / clip
//   out      = E4M3( v / step ),  step = 1 / scale (one scale: narrowed to fp32 first, as the reference's array routine
//              does; per channel: the double)                lib/Dialect/Tpu/Interfaces/Common/MatMul.cpp:598-629
//
// 128 x 128 outputs per workgroup, 4 waves (2 x 2), each wave 64 x 64 as 2 x 2 blocks of 32 x 32.  K advances 64 bytes per
// stage; one matrix instruction consumes a whole stage of a block (64 k: lane l holds two 16-byte pieces of row l % 32
// for both operands -- the contraction order inside an instruction is free as long as both sides agree).
//   f8_gemm_ring_kernel   a ring of LDS stages filled by direct-to-LDS loads (no staging registers, several stages of
//                         requests in flight), 16-byte chunks XOR-swizzled against bank conflicts, workgroups renumbered
//                         so that each XCD's L2 sees a compact block of tiles.
//   f8_gemm_large_kernel  the same for 256 x 256 tiles.
// A [K, N] right operand, and a K that is no whole number of stages, is rewritten first (operand_copy.hip; code 0 = +0:
// padding adds nothing).
//
// The fp8 matrix pipeline aligns the products of one instruction to the largest and drops low bits, so a long sum
// carries a relative error of about 2^-13 where an fp32 FMA chain has 2^-24; after the E4M3 rounding (2^-4 steps) that
// moves a result across a rounding boundary about once in a thousand outputs.  The reference's own fp32 matmul fixes
// no summation order either; tests bound the fp32 value and count the differing codes.
#include <cstdlib>

#include "device_math.h"
#include "internal.h"

namespace mi {

typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
typedef __attribute__((ext_vector_type(8))) int i32x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;

constexpr int F8_BM = 128, F8_BN = 128, F8_BK = 64;

struct F8Args {
  const uint8_t *A;     // [M, K] E4M3 codes
  const uint8_t *B;     // [N, K] E4M3 codes
  const float *bias;    // [N] or null
  void *out;
  float *acc_out;       // fp32 value before requantization, or null
  int64_t M, K, N;
  int do_relu;
  float relu_limit;
  int out_kind;         // MI_F8_OUT_*
  double step;          // one scale: (double)(float)(1 / scale)
  float inv_step;       // one scale: fl32(1 / step)
  const double *scales; // per channel [N], or null
  // few-row kernel only: K shared by 2^split_shift workgroups per 32-column block (0: none of the below is touched)
  int split_shift;
  float *part;          // [workgroup][16 registers][64 lanes]
  unsigned *counters;   // [block], zero between launches
};

// operand format of v_mfma_f32_32x32x64_f8f6f4 (its cbsz / blgp fields): 0 = E4M3, 1 = E5M2
constexpr int F8_FMT_E4M3 = 0, F8_FMT_E5M2 = 1;

// The output arms of a product of E5M2 operands (MatMul.cpp:630-635): F8E5M2(v, 1.0, true) for an E5M2 result (as
// codes or as the values in f32), F16(v) / BF16(v) for a 16-bit result.
__device__ __forceinline__ void f8_store_e5m2(const F8Args &a, int64_t o, float v) {
  if (a.out_kind == MI_F8_OUT_CODES)
    ((uint8_t *)a.out)[o] = (uint8_t)f8e5m2_from_f32(v);
  else if (a.out_kind == MI_F8_OUT_F32)
    ((float *)a.out)[o] = f8e5m2_to_f32(f8e5m2_from_f32(v));
  else if (a.out_kind == MI_F8_OUT_BF16)
    ((uint16_t *)a.out)[o] = f32_to_bf16_bm(v);
  else
    ((uint16_t *)a.out)[o] = f32_to_f16_ref(v);
}

// One output: bias added by the caller; ReLU, the fp32 side output, the requantization and the store.
template <int FMT>
__device__ __forceinline__ void f8_finish_one(const F8Args &a, int64_t o, float v, double step, double inv_step) {
  if (a.do_relu) {  // post_relu, lib/Support/Dnnl/DnnlUtils.cpp:15-25
    v = v > 0.0f ? v : 0.0f;
    if (a.relu_limit > 0.0f && v > a.relu_limit)
      v = a.relu_limit;
  }
  if (a.acc_out)
    a.acc_out[o] = v;
  if constexpr (FMT == F8_FMT_E5M2) {
    f8_store_e5m2(a, o, v);
    return;
  }
  // F8E4M3(v, step, true): the quotient in double, narrowed to fp32, rounded to E4M3 (Float8.cpp:259-261).
  // v * (1 / step) is within two double ulps of that quotient, so the narrowing can come out differently
  // only when the 29 bits it drops sit next to the halfway pattern; only then is the division carried out.
  double qd = (double)v * inv_step;
  const int32_t low = (int32_t)((uint32_t)__double_as_longlong(qd) & 0x1fffffffu);
  if (low >= 0x10000000 - 4 && low <= 0x10000000 + 4)
    qd = (double)v / step;
  const uint32_t code = f8e4m3_from_f32((float)qd);
  if (a.out_kind == MI_F8_OUT_CODES)
    ((uint8_t *)a.out)[o] = (uint8_t)code;
  else if (a.out_kind == MI_F8_OUT_F32)
    ((float *)a.out)[o] = f8e4m3_to_f32(code);
  else if (a.out_kind == MI_F8_OUT_BF16)  // exact: E4M3 values fit both 16-bit types
    ((uint16_t *)a.out)[o] = (uint16_t)(__float_as_uint(f8e4m3_to_f32(code)) >> 16);
  else
    ((uint16_t *)a.out)[o] = __builtin_bit_cast(uint16_t, (_Float16)f8e4m3_to_f32(code));
}

// The reference's requantization is E4M3((float)((double)v / step)), Float8.cpp:259-261.  With inv an fp32 number within
// 2^-23 of 1 / step (per channel: the scale itself rounded to fp32, since step = 1 / scale; one scale: fl32(1 / step)
// from the host), v * inv is within 3.01 fp32 ulps of the real quotient v / step and the reference's fp32 quotient
// within 0.51, so the two can only round to different E4M3 codes when a rounding boundary lies within 4 ulps of v * inv.
// The test: v times inv shrunk and grown by 2^-20 (7 ulps or more after their own roundings) must convert to the same
// code; conversion is monotonic, so then every value in between does, the reference's included.  Otherwise (about 6
// outputs in 10^5) the division is carried out as written, four outputs at a time.  The hardware conversion
// (v_cvt_pk_fp8_f32: round to nearest even, subnormals included) runs on values clamped to +-448, which is the
// reference's saturation; NaN goes down the slow path.
// four columns' requantization as the reference writes it; out of line, so that the call sites of the fast path do not
// each carry copies of the double divisions and the software conversion
__device__ __attribute__((noinline)) uint32_t f8_requant_exact4(float v0, float v1, float v2, float v3, const double *scales,
                                                                int64_t n, int64_t last, double step) {
  const float v[4] = {v0, v1, v2, v3};
  uint32_t w = 0;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const double st = scales ? 1.0 / scales[n + e < last ? n + e : last] : step;
    w |= f8e4m3_from_f32((float)((double)v[e] / st)) << (8 * e);
  }
  return w;
}

// what a lane keeps of the 16 consecutive columns it finishes
struct F8Cols {
  int64_t n0;
  bool whole;                          // all 16 exist: 16-byte accesses, of output rows at any alignment
  float bias[16], inv_lo[16], inv_hi[16];  // inv_lo / inv_hi: fl32(1 / step) shrunk / grown by 2^-20
};
__device__ __forceinline__ void f8_load_cols(const F8Args &a, F8Cols &c, int64_t n0) {
  constexpr float DN = 1.0f - 0x1p-20f, UP = 1.0f + 0x1p-20f;
  c.n0 = n0;
  c.whole = n0 + 16 <= a.N;
  // every load of an array is on its way before the first is used
  auto at = [&](int e) { return (n0 + e) < a.N ? (n0 + e) : (a.N - 1); };
#pragma unroll
  for (int e = 0; e < 16; ++e)
    c.bias[e] = 0.0f;
  if (a.bias) {
#pragma unroll
    for (int e = 0; e < 16; ++e)
      c.bias[e] = a.bias[at(e)];
  }
  float inv[16];
#pragma unroll
  for (int e = 0; e < 16; ++e)
    inv[e] = a.inv_step;
  if (a.scales) {
#pragma unroll
    for (int e = 0; e < 16; ++e)
      inv[e] = (float)a.scales[at(e)];
  }
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    c.inv_lo[e] = inv[e] * DN;
    c.inv_hi[e] = inv[e] * UP;
  }
}
template <typename V>
__device__ __forceinline__ void f8_store16(void *p, V v) {
  static_assert(sizeof(V) == 16, "16 bytes");
  __builtin_memcpy(p, &v, 16);
}

// The output kinds and row ends that are not 16 whole codes: n codes as codes or as the values they stand for (exact in
// all three types).  Out of line: the finishing loop is instantiated several times.
__device__ __attribute__((noinline)) void f8_store_codes(void *out, int kind, int64_t o, int n, uint32_t w0, uint32_t w1,
                                                         uint32_t w2, uint32_t w3) {
  const uint32_t w[4] = {w0, w1, w2, w3};
  auto code = [&](int e) { return (w[e >> 2] >> (8 * (e & 3))) & 0xffu; };
  if (kind == MI_F8_OUT_CODES) {
#pragma unroll
    for (int e = 0; e < 16; ++e)
      if (e < n)
        ((uint8_t *)out)[o + e] = (uint8_t)code(e);
    return;
  }
  if (kind == MI_F8_OUT_F32) {
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        v[e] = f8e4m3_to_f32(code(q4 * 4 + e));
      if (q4 * 4 + 4 <= n) {
        f8_store16((float *)out + o + q4 * 4, f32x4{v[0], v[1], v[2], v[3]});
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (q4 * 4 + e < n)
            ((float *)out)[o + q4 * 4 + e] = v[e];
      }
    }
    return;
  }
#pragma unroll
  for (int q8 = 0; q8 < 2; ++q8) {
    uint32_t h[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float v = f8e4m3_to_f32(code(q8 * 8 + e));
      h[e] = kind == MI_F8_OUT_BF16 ? __float_as_uint(v) >> 16 : __builtin_bit_cast(uint16_t, (_Float16)v);
    }
    if (q8 * 8 + 8 <= n) {
      f8_store16((uint16_t *)out + o + q8 * 8,
                 u32x4{h[0] | (h[1] << 16), h[2] | (h[3] << 16), h[4] | (h[5] << 16), h[6] | (h[7] << 16)});
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (q8 * 8 + e < n)
          ((uint16_t *)out)[o + q8 * 8 + e] = (uint16_t)h[e];
    }
  }
}

// One row of a lane's 16 columns, read from the strip: bias, ReLU, side output, requantization, store.
template <int FMT>
__device__ __forceinline__ void f8_finish_row(const F8Args &a, const F8Cols &c, const float *src, int64_t m) {
  float v[16];
#pragma unroll
  for (int q4 = 0; q4 < 4; ++q4) {
    const f32x4 t = *(const f32x4 *)(src + q4 * 4);
#pragma unroll
    for (int e = 0; e < 4; ++e)
      v[q4 * 4 + e] = t[e] + c.bias[q4 * 4 + e];
  }
  if (a.do_relu) {  // post_relu, lib/Support/Dnnl/DnnlUtils.cpp:15-25 (its comparison sends a NaN to 0 as well)
    const float relu_hi = a.relu_limit > 0.0f ? a.relu_limit : __builtin_inff();
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      v[e] = v[e] > 0.0f ? v[e] : 0.0f;
      v[e] = v[e] > relu_hi ? relu_hi : v[e];
    }
  }
  if (m >= a.M || c.n0 >= a.N)
    return;
  const int64_t o = m * a.N + c.n0;
  if (a.acc_out) {
    if (c.whole) {
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4)
        f8_store16(a.acc_out + o + q4 * 4, f32x4{v[q4 * 4], v[q4 * 4 + 1], v[q4 * 4 + 2], v[q4 * 4 + 3]});
    } else {
#pragma unroll
      for (int e = 0; e < 16; ++e)
        if (c.n0 + e < a.N)
          a.acc_out[o + e] = v[e];
    }
  }
  if constexpr (FMT == F8_FMT_E5M2) {
    if (c.whole && a.out_kind == MI_F8_OUT_CODES) {
      uint32_t w[4];
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4)
        w[q4] = f8e5m2_from_f32(v[q4 * 4]) | (f8e5m2_from_f32(v[q4 * 4 + 1]) << 8) |
                (f8e5m2_from_f32(v[q4 * 4 + 2]) << 16) | (f8e5m2_from_f32(v[q4 * 4 + 3]) << 24);
      f8_store16((uint8_t *)a.out + o, u32x4{w[0], w[1], w[2], w[3]});
      return;
    }
#pragma unroll
    for (int e = 0; e < 16; ++e)
      if (c.n0 + e < a.N)
        f8_store_e5m2(a, o + e, v[e]);
    return;
  } else {
    uint32_t w[4];  // four codes each
    uint32_t differ = 0;
    bool nan = false;
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      auto clamped = [](float q) { return __builtin_amdgcn_fmed3f(q, -448.0f, 448.0f); };
      int lo = 0, hi = 0;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int e = q4 * 4 + u * 2;
        const float l0 = clamped(v[e] * c.inv_lo[e]), l1 = clamped(v[e + 1] * c.inv_lo[e + 1]);
        const float h0 = clamped(v[e] * c.inv_hi[e]), h1 = clamped(v[e + 1] * c.inv_hi[e + 1]);
        lo = u ? __builtin_amdgcn_cvt_pk_fp8_f32(l0, l1, lo, true) : __builtin_amdgcn_cvt_pk_fp8_f32(l0, l1, lo, false);
        hi = u ? __builtin_amdgcn_cvt_pk_fp8_f32(h0, h1, hi, true) : __builtin_amdgcn_cvt_pk_fp8_f32(h0, h1, hi, false);
        nan |= __builtin_isunordered(v[e], v[e + 1]);
      }
      w[q4] = (uint32_t)lo;
      differ |= (uint32_t)(lo != hi) << q4;
    }
    if (differ != 0 || nan) {
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4)
        if (nan || ((differ >> q4) & 1))
          w[q4] = f8_requant_exact4(v[q4 * 4], v[q4 * 4 + 1], v[q4 * 4 + 2], v[q4 * 4 + 3], a.scales, c.n0 + q4 * 4, a.N - 1,
                                    a.step);
    }
    if (c.whole && a.out_kind == MI_F8_OUT_CODES) {
      f8_store16((uint8_t *)a.out + o, u32x4{w[0], w[1], w[2], w[3]});
      return;
    }
    const int64_t left = a.N - c.n0;
    f8_store_codes(a.out, a.out_kind, o, left < 16 ? (int)left : 16, w[0], w[1], w[2], w[3]);
  }
}

// Epilogue of NBI x NBJ blocks of a wave through its own strip of LDS: the accumulators (register r of lane l = row
// 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32 of block (i, j)) are laid out row-major (NBJ * 32 + 4 dwords a row:
// 16-byte aligned, staggered banks) so that a lane owns 16 consecutive columns of a row -- per-column parameters are
// fetched once per lane, results leave as 16-byte stores.
template <int NBJ>
__device__ __forceinline__ int f8_strip_col(int lane) { return lane % (NBJ * 2) * 16; }
template <int FMT, int NBI, int NBJ>
__device__ __forceinline__ void f8_strip_epilogue(const F8Args &a, const f32x16 (&acc)[NBI][NBJ], const F8Cols &cols, float *strip,
                                                  int64_t m0, int lane) {
  constexpr int STRIDE = NBJ * 32 + 4, CPR = NBJ * 2, RPP = 64 / CPR, PASSES = NBI * 32 / RPP;
#pragma unroll
  for (int i = 0; i < NBI; ++i)
#pragma unroll
    for (int j = 0; j < NBJ; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        strip[(i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)) * STRIDE + j * 32 + (lane & 31)] = acc[i][j][r];
  // a wave only reads what it wrote: no barrier, the LDS counter orders it
#pragma unroll 1
  for (int p = 0; p < PASSES; ++p) {
    const int row = p * RPP + lane / CPR;
    f8_finish_row<FMT>(a, cols, strip + row * STRIDE + f8_strip_col<NBJ>(lane), m0 + row);
  }
}

typedef const __attribute__((address_space(1))) void *f8_gptr_t;
typedef __attribute__((address_space(3))) void *f8_lptr_t;
constexpr int f8_stage_bytes(int bt) { return 2 * bt * F8_BK; }  // 16 KiB (128-tiles) / 8 KiB (64-tiles)
constexpr int f8_waitcnt_vm(int n) { return (n & 0xF) | ((n >> 4) << 14) | 0x0F70; }  // s_waitcnt vmcnt(n) only
// the ring, or the four epilogue strips that reuse its memory, whichever is larger
constexpr int f8_ring_lds_bytes(int nst, int bt = 128) {
  return nst * f8_stage_bytes(bt) > 4 * (bt / 2) * (bt / 2 + 4) * 4 ? nst * f8_stage_bytes(bt)
                                                                      : 4 * (bt / 2) * (bt / 2 + 4) * 4;
}

// NST = stages in the LDS ring: 4 (two workgroups per CU) when there are more tiles than CUs, 8 when every workgroup
// has a CU to itself
// BT = tile edge: 128 (a wave 64 x 64), or 64 (a wave one 32 x 32 block) for grids of up to 128 tiles of 128 x 128:
// four times the workgroups, several per CU hiding each other's waits (the INT8 kernel's measured crossover)
template <int NST, int FMT, int BT = 128>
__global__ __launch_bounds__(256) void f8_gemm_ring_kernel(F8Args a, int tiles_m, int tiles_n, int per_xcd) {
  constexpr int WT = BT / 2, NB = WT / 32;
  constexpr int F8_STAGE = f8_stage_bytes(BT);
  constexpr int LOADS = BT * (F8_BK / 16) / 256;  // direct-to-LDS instructions per operand, stage and thread: 2 or 1
  constexpr int LPS = 2 * LOADS;
  extern __shared__ __attribute__((aligned(16))) uint8_t f8_lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int bid = blockIdx.x;
  const int L = (bid & 7) * per_xcd + (bid >> 3);  // each XCD gets a contiguous run of the tile order
  if (L >= tiles_m * tiles_n)
    return;
  constexpr int GM = 4;  // tiles are ordered in groups of 4 tile rows, column-major inside a group
  const int group = L / (GM * tiles_n);
  const int gm = (tiles_m - group * GM) < GM ? (tiles_m - group * GM) : GM;
  const int in_group = L - group * GM * tiles_n;
  const int tm = group * GM + in_group % gm, tn = in_group / gm;
  const int64_t m_base = (int64_t)tm * BT, n_base = (int64_t)tn * BT;

  // the 16-byte chunk c of row r is stored at position c ^ ((r >> 2) & 3): the 32 rows of a fragment read hit distinct
  // bank groups
  const uint8_t *ga[LOADS], *gb[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int slot = (i * 4 + wave) * 64 + lane;
    const int row = slot >> 2, pos = slot & 3;
    const int chunk = pos ^ ((row >> 2) & 3);
    int64_t ra = m_base + row, rb = n_base + row;
    ra = ra < a.M ? ra : a.M - 1;  // rows past the matrix re-read the last one; their results are never stored
    rb = rb < a.N ? rb : a.N - 1;
    ga[i] = a.A + ra * a.K + chunk * 16;
    gb[i] = a.B + rb * a.K + chunk * 16;
  }
  const int kt_total = (int)(a.K / F8_BK);
  auto issue = [&](int kt) {
    const int64_t koff = (int64_t)(kt < kt_total ? kt : kt_total - 1) * F8_BK;  // past the end: harmless re-load
    uint8_t *sa = f8_lds + (kt % NST) * F8_STAGE, *sb = sa + BT * F8_BK;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      __builtin_amdgcn_global_load_lds((f8_gptr_t)(ga[i] + koff), (f8_lptr_t)(sa + (i * 4 + wave) * 1024), 16, 0, 0);
      __builtin_amdgcn_global_load_lds((f8_gptr_t)(gb[i] + koff), (f8_lptr_t)(sb + (i * 4 + wave) * 1024), 16, 0, 0);
    }
  };

  f32x16 acc[NB][NB];
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        acc[i][j][r] = 0.0f;

  const int frow = lane & 31, kh = lane >> 5;
  int a_off[NB], b_off[NB];
  const int f_sw = (frow >> 2) & 3;  // (row >> 2) & 3 with row = 32-aligned base + frow
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    a_off[i] = (wm * WT + i * 32 + frow) * F8_BK;
    b_off[i] = BT * F8_BK + (wn * WT + i * 32 + frow) * F8_BK;
  }
#pragma unroll
  for (int s0 = 0; s0 < NST - 1; ++s0)
    issue(s0);
  for (int kt = 0; kt < kt_total; ++kt) {
    // requests complete in order: at most (NST - 2) stages' worth outstanding means stage kt has landed
    __builtin_amdgcn_s_waitcnt(f8_waitcnt_vm((NST - 2) * LPS));
    __builtin_amdgcn_s_barrier();  // everyone's share of stage kt is in LDS; everyone is done with stage kt - 1
    issue(kt + NST - 1);
    const uint8_t *st = f8_lds + (kt % NST) * F8_STAGE;
    // lane (row, kh) takes chunks kh and 2 + kh of its row for both operands
    i32x8 fa[NB], fb[NB];
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const u32x4 a0 = *(const u32x4 *)(st + a_off[i] + ((kh ^ f_sw) << 4));
      const u32x4 a1 = *(const u32x4 *)(st + a_off[i] + (((2 + kh) ^ f_sw) << 4));
      const u32x4 b0 = *(const u32x4 *)(st + b_off[i] + ((kh ^ f_sw) << 4));
      const u32x4 b1 = *(const u32x4 *)(st + b_off[i] + (((2 + kh) ^ f_sw) << 4));
      fa[i] = i32x8{(int)a0[0], (int)a0[1], (int)a0[2], (int)a0[3], (int)a1[0], (int)a1[1], (int)a1[2], (int)a1[3]};
      fb[i] = i32x8{(int)b0[0], (int)b0[1], (int)b0[2], (int)b0[3], (int)b1[0], (int)b1[1], (int)b1[2], (int)b1[3]};
    }
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fa[i], fb[j], acc[i][j], FMT, FMT, 0, 0, 0, 0);
  }
  __builtin_amdgcn_s_waitcnt(f8_waitcnt_vm(0));  // drain the re-loads issued past the end
  __builtin_amdgcn_s_barrier();                  // every wave is done reading the ring
  F8Cols cols;
  f8_load_cols(a, cols, n_base + wn * WT + f8_strip_col<NB>(lane));
  f8_strip_epilogue<FMT, NB, NB>(a, acc, cols, (float *)f8_lds + wave * (WT * (WT + 4)), m_base + wm * WT, lane);
}

// ---- 256 x 256 outputs per workgroup, eight waves (2 x 4, two per SIMD: one wave's waits run under the other's matrix
// instructions), each 128 x 64 as 4 x 2 blocks of 32 x 32 (128 fp32 accumulators per lane).  K advances 64 bytes per
// stage, one matrix instruction per block; five stages of 32 KiB fill all of LDS.  As in the INT8 kernel of this tile
// (i8_kernels.hip) stages are requested in pairs, the two halves of every 128-byte line back to back, so that the vector
// cache asks L2 for each line once.  Requires K % 128 == 0.  4096^3, per-channel scales: 61.5 us (2.23 PFLOP/s; four
// waves of 128 x 128 with single-stage requests and the longer epilogue: 84.8); the vendor's fp8 product without
// requantization reaches 2.77 at this size.
//
// A stage is a batch of eight matrix instructions with the next stage's twelve fragment reads and, in every second
// batch, the eight requests of a pair of stages pinned between them.  The left fragments of the next stage take the
// registers of this stage's as soon as their two instructions are issued; the right ones alternate between two sets.
// One barrier per stage, at its start: by then every wave has received the stage's fragments (its LDS buffer is free)
// and its own share of the next stage, and so after it the next stage is complete.  The pair (2p + 4, 2p + 5) takes
// the buffers of stages 2p - 1 and 2p, is requested in batch 2p and first read in batch 2p + 3.
constexpr int F8L_M = 256, F8L_N = 256;
constexpr int F8L_STAGE = (F8L_M + F8L_N) * F8_BK;  // 32 KiB
constexpr int F8L_NST = 5;
constexpr int F8_WAITCNT_LGKM0 = 0xC07F;

template <int FMT>
__global__ __launch_bounds__(512, 1) void f8_gemm_large_kernel(F8Args a, int tiles_m, int tiles_n, int per_xcd) {
  constexpr int NST = F8L_NST;
  constexpr int LOADS = F8L_M * (F8_BK / 16) / 512;  // direct-to-LDS instructions per operand, stage and thread: 2
  constexpr int PAIR = 4 * LOADS;                    // requests per thread and pair of stages
  extern __shared__ __attribute__((aligned(16))) uint8_t f8_lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 2, wn = wave & 3;
  const int bid = blockIdx.x;
  const int L = (bid & 7) * per_xcd + (bid >> 3);  // each XCD gets a contiguous run of the tile order
  if (L >= tiles_m * tiles_n)
    return;
  constexpr int GM = 4;
  const int group = L / (GM * tiles_n);
  const int gm = (tiles_m - group * GM) < GM ? (tiles_m - group * GM) : GM;
  const int in_group = L - group * GM * tiles_n;
  const int tm = group * GM + in_group % gm, tn = in_group / gm;
  const int64_t m_base = (int64_t)tm * F8L_M, n_base = (int64_t)tn * F8L_N;

  // a lane's address is a uniform tile base plus a 32-bit offset (rows past the matrix re-read the last one; their
  // results are never stored); the 16-byte chunk c of row r is stored at position c ^ ((r >> 2) & 3)
  const uint8_t *Abase = a.A + m_base * a.K, *Bbase = a.B + n_base * a.K;
  uint32_t va[LOADS], vb[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int slot = (i * 8 + wave) * 64 + lane;
    const int row = slot >> 2, chunk = (slot & 3) ^ ((row >> 2) & 3);
    int64_t ra = m_base + row, rb = n_base + row;
    ra = ra < a.M ? ra : a.M - 1;
    rb = rb < a.N ? rb : a.N - 1;
    va[i] = (uint32_t)((ra - m_base) * a.K + chunk * 16);
    vb[i] = (uint32_t)((rb - n_base) * a.K + chunk * 16);
  }
  const int pairs = (int)(a.K / (2 * F8_BK));
  // one operand (half = 0: A, 1: B), one of its LOADS pieces of a pair of stages; s0, s1: their buffers
  auto issue = [&](int pair, int half, int i, int s0, int s1) {
    const int64_t koff = (int64_t)(pair < pairs ? pair : pairs - 1) * (2 * F8_BK);  // past the end: harmless re-load
    const uint8_t *pg = (half ? Bbase : Abase) + koff;
    const uint32_t v = half ? vb[i] : va[i];
    uint8_t *l0 = f8_lds + s0 * F8L_STAGE + half * (F8L_M * F8_BK) + (i * 8 + wave) * 1024;
    uint8_t *l1 = f8_lds + s1 * F8L_STAGE + half * (F8L_M * F8_BK) + (i * 8 + wave) * 1024;
    __builtin_amdgcn_global_load_lds((f8_gptr_t)(pg + v), (f8_lptr_t)l0, 16, 0, 0);
    __builtin_amdgcn_global_load_lds((f8_gptr_t)(pg + v + F8_BK), (f8_lptr_t)l1, 16, 0, 0);
  };

  f32x16 acc[4][2];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        acc[i][j][r] = 0.0f;

  const int frow = lane & 31, kh = lane >> 5;
  const int f_sw = (frow >> 2) & 3;
  const int c0 = (kh ^ f_sw) << 4, c1 = ((2 + kh) ^ f_sw) << 4;  // this lane's two chunks of a row, swizzled
  const int a_row = (wm * 128 + frow) * F8_BK, b_row = F8L_M * F8_BK + (wn * 64 + frow) * F8_BK;
  auto read_frag = [&](i32x8 &f, const uint8_t *st, int off) {
    const u32x4 lo = *(const u32x4 *)(st + off + c0), hi = *(const u32x4 *)(st + off + c1);
    f = i32x8{(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
  };

  i32x8 fa[4], fb[2][2];
  // batch kt: its fragments are in fa and fb[cur]; pair >= 0: that pair of stages is requested on the way
  auto batch = [&](int cur, int kt, int pair) {
    __builtin_amdgcn_s_waitcnt(F8_WAITCNT_LGKM0);
    __builtin_amdgcn_s_waitcnt(f8_waitcnt_vm(PAIR));  // all but the newest pair of stages
    __builtin_amdgcn_s_barrier();
    const uint8_t *st = f8_lds + (kt + 1) % NST * F8L_STAGE;
    const int s0 = (kt + 4) % NST, s1 = kt % NST;  // pair: the buffers of stages kt + 4 and kt + 5
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const int i = t >> 1, j = t & 1;
      acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fa[i], fb[cur][j], acc[i][j], FMT, FMT, 0, 0, 0, 0);
      if (j)
        read_frag(fa[i], st, a_row + i * 32 * F8_BK);
      else if (i < 2)
        read_frag(fb[cur ^ 1][i], st, b_row + i * 32 * F8_BK);
      if (pair >= 0 && t >= 4)
        issue(pair, (t - 4) >> 1, (t - 4) & 1, s0, s1);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int i = 0; i < LOADS; ++i)
        issue(p, half, i, 2 * p, 2 * p + 1);
  __builtin_amdgcn_s_waitcnt(f8_waitcnt_vm(PAIR));  // stages 0 and 1 landed
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int i = 0; i < 4; ++i)
    read_frag(fa[i], f8_lds, a_row + i * 32 * F8_BK);
#pragma unroll
  for (int j = 0; j < 2; ++j)
    read_frag(fb[0][j], f8_lds, b_row + j * 32 * F8_BK);
  for (int p = 0; p < pairs; ++p) {
    batch(0, 2 * p, p + 2);
    batch(1, 2 * p + 1, -1);
  }
  __builtin_amdgcn_s_waitcnt(f8_waitcnt_vm(0));  // drain the re-loads issued past the end
  __syncthreads();                               // every wave is done with the ring

  F8Cols cols;
  f8_load_cols(a, cols, n_base + wn * 64 + f8_strip_col<2>(lane));
  float *strip = (float *)f8_lds + wave * (32 * 68);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const f32x16 sub[1][2] = {{acc[i][0], acc[i][1]}};
    f8_strip_epilogue<FMT, 1, 2>(a, sub, cols, strip, m_base + wm * 128 + i * 32, lane);
  }
}

// ------------------------------------------------------------------------------------------------
// Few rows (M <= 32): a stream over the right operand, HBM-bound; the INT8 few-row kernel (i8_kernels.hip) on F8
// codes.  A workgroup owns 32 output columns, its eight waves take the 128-byte K tiles round-robin (with the waves of
// the block's other K parts, when K is split over workgroups), each multiplies all rows against its tiles (a lane's 64
// bytes of its row feed two K = 64 MFMAs; the K order inside a tile is permuted alike for both operands).  As there,
// the right operand comes in whole cache lines through the wave's own two-tile LDS ring and the left one straight into
// registers by untracked loads, one tile ahead, both waited for by request count.  Partial sums are added in wave
// order, then in part order: fp32 sums in another order than the tiled kernels', inside the same bound.  Requires
// K % 128 == 0.
// ------------------------------------------------------------------------------------------------
__device__ __forceinline__ u32x4 f8_load16_untracked(const void *p) {
  u32x4 v;
  asm volatile("global_load_dwordx4 %0, %1, off" : "=v"(v) : "v"(p) : "memory");
  return v;
}
template <int FMT>
__global__ __launch_bounds__(512) void f8_rows32_kernel(F8Args a) {
  constexpr int WAVES = 8;
  constexpr int RING_BYTES = WAVES * 2 * 4096;  // per wave: two tiles of 32 rows x 128 bytes of the right operand
  __shared__ __attribute__((aligned(16))) uint8_t smem[RING_BYTES];
  float (*red)[16][64] = reinterpret_cast<float (*)[16][64]>(smem);  // overlays the rings after the loop
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c32 = lane & 31, h = lane >> 5;
  const int parts = 1 << a.split_shift, part = blockIdx.x & (parts - 1);
  const int64_t block = blockIdx.x >> a.split_shift;
  const int64_t n = block * 32 + c32;
  const int64_t ma = c32 < a.M ? c32 : a.M - 1;
  const uint8_t *pa = a.A + ma * a.K + h * 64;
  // request q of a tile: rows 8 q + lane / 8 of the block, the lane's 16-byte chunk (lane % 8, swizzled by the row)
  const uint8_t *pb[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int r = 8 * q + (lane >> 3);
    int64_t nb = block * 32 + r;
    nb = nb < a.N ? nb : a.N - 1;  // columns past N repeat the last one; never stored
    pb[q] = a.B + nb * a.K + (((lane & 7) ^ ((r >> 1) & 7)) << 4);
  }
  uint8_t *ring = smem + wave * 8192;
  const uint8_t *bfrag = ring + c32 * 128;
  const int k_tiles = (int)(a.K / 128);
  const int first = part * WAVES + wave, stride = WAVES << a.split_shift;
  const int count = (k_tiles - first + stride - 1) / stride;

  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r)
    acc[r] = 0.0f;
  u32x4 xa[2][4];
  auto issue_tile = [&](int i, int slot) {  // eight requests: four into LDS, four into registers
    const int64_t off = (int64_t)(first + (i < count ? i : count - 1) * stride) * 128;  // past the end: a re-load
#pragma unroll
    for (int q = 0; q < 4; ++q)
      __builtin_amdgcn_global_load_lds((f8_gptr_t)(pb[q] + off), (f8_lptr_t)(ring + slot * 4096 + q * 1024), 16, 0, 0);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      xa[slot][j] = f8_load16_untracked(pa + off + j * 16);
  };
  if (count > 0) {
    issue_tile(0, 0);
    for (int t0 = 0; t0 < count; t0 += 2) {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        if (t0 + u >= count)
          break;
        issue_tile(t0 + u + 1, u ^ 1);
        __builtin_amdgcn_s_waitcnt(f8_waitcnt_vm(8));  // all but the tile just asked for
        asm volatile("" ::: "memory");                 // the tile is in LDS from here on, not before
#pragma unroll
        for (int j = 0; j < 4; ++j)
          asm volatile("" : "+v"(xa[u][j]));           // ... and in its registers
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const u32x4 a0 = xa[u][2 * j], a1 = xa[u][2 * j + 1];
          const u32x4 b0 = *(const u32x4 *)(bfrag + u * 4096 + (((4 * h + 2 * j) ^ ((c32 >> 1) & 7)) << 4));
          const u32x4 b1 = *(const u32x4 *)(bfrag + u * 4096 + (((4 * h + 2 * j + 1) ^ ((c32 >> 1) & 7)) << 4));
          const i32x8 fa = {(int)a0[0], (int)a0[1], (int)a0[2], (int)a0[3], (int)a1[0], (int)a1[1], (int)a1[2], (int)a1[3]};
          const i32x8 fb = {(int)b0[0], (int)b0[1], (int)b0[2], (int)b0[3], (int)b1[0], (int)b1[1], (int)b1[2], (int)b1[3]};
          acc = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fa, fb, acc, FMT, FMT, 0, 0, 0, 0);
        }
      }
    }
    __builtin_amdgcn_s_waitcnt(f8_waitcnt_vm(0));  // the re-loads issued past the end
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        asm volatile("" : "+v"(xa[u][j]));  // their registers stay taken until here
  }
  __syncthreads();  // the partial blocks overlay the rings: every wave is done with its tiles
  // cross-wave sum, in wave order.  Register r of lane l is row 8 * (r / 4) + 4 * (l / 32) + r % 4, column l % 32.
#pragma unroll
  for (int r = 0; r < 16; ++r)
    red[wave][r][lane] = acc[r];
  __syncthreads();
  float sum[2] = {0.0f, 0.0f};
#pragma unroll
  for (int q = 0; q < 2; ++q)
#pragma unroll
    for (int wv = 0; wv < WAVES; ++wv)
      sum[q] += red[wv][wave * 2 + q][lane];
  if (a.split_shift != 0) {
    // the block's other K parts: see i8_rows32_kernel (device-scope relaxed atomics ordered by waiting for them)
    __shared__ int last_flag;
    float *slab = a.part + block * parts * 1024;
    const int idx = wave * 128 + lane;
    __hip_atomic_store(slab + part * 1024 + idx, sum[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(slab + part * 1024 + idx + 64, sum[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __builtin_amdgcn_s_waitcnt(f8_waitcnt_vm(0));
    __syncthreads();
    if (tid == 0) {
      const unsigned before = __hip_atomic_fetch_add(a.counters + block, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const int last = before == (unsigned)(parts - 1);
      if (last)
        __hip_atomic_store(a.counters + block, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      last_flag = last;
    }
    __syncthreads();
    if (!last_flag)
      return;
    sum[0] = sum[1] = 0.0f;
    for (int p = 0; p < parts; ++p) {
      sum[0] += __hip_atomic_load(slab + p * 1024 + idx, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      sum[1] += __hip_atomic_load(slab + p * 1024 + idx + 64, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  const bool n_ok = n < a.N;
  const float bias_n = (a.bias && n_ok) ? a.bias[n] : 0.0f;
  const double step = (a.scales && n_ok) ? 1.0 / a.scales[n] : a.step;
  const double inv_step = 1.0 / step;
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int r = wave * 2 + q;
    const int64_t m = 8 * (r >> 2) + 4 * h + (r & 3);
    if (n_ok && m < a.M)
      f8_finish_one<FMT>(a, m * a.N + n, sum[q] + bias_n, step, inv_step);
  }
}

int f8mm_launch(const uint8_t *d_a, const uint8_t *d_b, int right_transpose, const float *d_bias, int64_t M, int64_t K,
                int64_t N, int do_relu, double relu_limit, double out_scale, const double *d_out_scales, int out_kind,
                void *d_out, float *d_acc, hipStream_t stream, int f8_type) {
  MI_REQUIRE(f8_type == MI_F8_E4M3 || f8_type == MI_F8_E5M2, MI_BAD_ARGUMENT, "mi_f8mm_launch: f8_type");
  if (f8_type == MI_F8_E5M2) {  // MatMul.cpp:630-635: no scales on these arms
    d_out_scales = nullptr;
    out_scale = 1.0;
  }
  MI_REQUIRE(M >= 0 && K > 0 && N > 0, MI_BAD_ARGUMENT, "mi_f8mm_launch: bad shape");
  MI_REQUIRE(M == 0 || (d_a && d_b && d_out), MI_BAD_ARGUMENT, "mi_f8mm_launch: null argument");
  MI_REQUIRE(out_kind >= MI_F8_OUT_CODES && out_kind <= MI_F8_OUT_F16, MI_BAD_ARGUMENT, "mi_f8mm_launch: out_kind");
  MI_REQUIRE(d_out_scales || (out_scale == out_scale && out_scale != 0.0), MI_BAD_ARGUMENT,
             "mi_f8mm_launch: the output scale must be a nonzero number");
  if (M == 0)
    return MI_SUCCESS;
  // kernel by size: the streaming kernel up to 32 rows, by the INT8 product's rule (same bytes per element; plan: f8_tile
  // = 32 asks for it, any other value rules it out; 4096 x 4096 (N x K) M = 1: 15.2 us on 64 x 64 tiles, 4096 x 11008:
  // 38.7), 256 x 256 tiles from the INT8 kernels' measured crossover on, 64 x 64 tiles up to 128 tiles of 128 x 128
  const int e = plan().f8_tile;
  const bool few_pays = M * N <= 45056 || (N <= 8192 && (M <= 24 || K > 4096));
  const bool few = M <= 32 && (K % 128) == 0 && (e == 32 || (e == 0 && few_pays));
  const int64_t tiles_m = (M + F8_BM - 1) / F8_BM, tiles_n = (N + F8_BN - 1) / F8_BN;
  const int64_t tl_m = (M + F8L_M - 1) / F8L_M, tl_n = (N + F8L_N - 1) / F8L_N;
  MI_REQUIRE(tiles_m * tiles_n < (int64_t(1) << 28), MI_UNSUPPORTED, "mi_f8mm_launch: too many outputs for one launch");
  const bool large = !few && (e > 0 && e != 32 ? e == 256 : tl_m * tl_n >= 144);
  const bool small = !few && !large && (e > 0 && e != 32 ? e == 64 : tiles_m * tiles_n <= 128);
  const int64_t stage = large ? 2 * F8_BK : F8_BK, Kp = few ? K : (K + stage - 1) / stage * stage;
  const bool rewrite_a = Kp != K, rewrite_b = Kp != K || !right_transpose;
  ScratchBytes scratch;
  const uint8_t *a_mk = d_a, *b_nk = d_b;
  if (rewrite_b) {
    const size_t a_bytes = rewrite_a ? (size_t)((M * Kp + 255) & ~(int64_t)255) : 0;
    int rc = scratch.get(stream, WS_F8_OPERANDS, a_bytes + (size_t)(N * Kp));
    if (rc != MI_SUCCESS)
      return rc;
    uint8_t *t = (uint8_t *)scratch.ptr;
    OperandCopy ca = {}, cb = {d_b, t + a_bytes, N, K, Kp, !right_transpose, 0, 0};
    if (rewrite_a) {
      ca = OperandCopy{d_a, t, M, K, Kp, 0, 0, 0};
      a_mk = t;
    }
    b_nk = t + a_bytes;
    if ((rc = operand_copy_launch(ca, cb, stream)))
      return rc;
  }
  F8Args a;
  a.A = a_mk;
  a.B = b_nk;
  a.bias = d_bias;
  a.out = d_out;
  a.acc_out = d_acc;
  a.M = M;
  a.K = Kp;
  a.N = N;
  a.do_relu = do_relu;
  a.relu_limit = (float)relu_limit;
  a.out_kind = out_kind;
  a.step = (double)(float)(1 / out_scale);  // MatMul.cpp:613-615 into the float parameter of Float8.cpp:267
  a.inv_step = (float)(1.0 / a.step);
  a.scales = d_out_scales;
  a.split_shift = 0;
  a.part = nullptr;
  a.counters = nullptr;
  const bool e5m2 = f8_type == MI_F8_E5M2;
  if (few) {
    const int64_t blocks = (N + 31) / 32;
    MI_REQUIRE(blocks < (1ll << 29), MI_BAD_ARGUMENT, "mi_f8mm_launch: too many output columns");
    while (a.split_shift < 2 && (blocks << (a.split_shift + 1)) <= R32_SPLIT_MAX_WGS &&
           K / 128 >= (32 << (a.split_shift + 1)))
      ++a.split_shift;
    if (a.split_shift != 0) {
      void *p = nullptr;
      // (a stream under capture that never ran such a shape gets the error: an unsplit launch would add the partial
      // sums in another order)
      const int rc = stream_workspace(stream, WS_ROWS32_SPLIT, R32_SPLIT_COUNTER_BYTES + (size_t)R32_SPLIT_MAX_WGS * 4096,
                                      &p, /*zero_fresh=*/true);
      if (rc != MI_SUCCESS)
        return rc;
      a.counters = (unsigned *)p;
      a.part = (float *)((uint8_t *)p + R32_SPLIT_COUNTER_BYTES);
    }
    const dim3 grid((unsigned)(blocks << a.split_shift));
    if (e5m2)
      f8_rows32_kernel<F8_FMT_E5M2><<<grid, dim3(512), 0, stream>>>(a);
    else
      f8_rows32_kernel<F8_FMT_E4M3><<<grid, dim3(512), 0, stream>>>(a);
  } else if (large) {
    static LdsLimitOnce lim_a, lim_b;
    lim_a.ensure((const void *)f8_gemm_large_kernel<F8_FMT_E4M3>, F8L_NST * F8L_STAGE);
    lim_b.ensure((const void *)f8_gemm_large_kernel<F8_FMT_E5M2>, F8L_NST * F8L_STAGE);
    const int per_xcd = (int)((tl_m * tl_n + 7) / 8);
    const dim3 grid((unsigned)(per_xcd * 8));
    if (e5m2)
      f8_gemm_large_kernel<F8_FMT_E5M2><<<grid, dim3(512), F8L_NST * F8L_STAGE, stream>>>(a, (int)tl_m, (int)tl_n, per_xcd);
    else
      f8_gemm_large_kernel<F8_FMT_E4M3><<<grid, dim3(512), F8L_NST * F8L_STAGE, stream>>>(a, (int)tl_m, (int)tl_n, per_xcd);
  } else {
    const int bt = small ? 64 : 128;
    const int tm = (int)((M + bt - 1) / bt), tn = (int)((N + bt - 1) / bt), per_xcd = (tm * tn + 7) / 8;
    const dim3 grid((unsigned)(per_xcd * 8));
#define MI_F8_RING(NST, BT)                                                                                             \
  {                                                                                                                     \
    static LdsLimitOnce lim_a, lim_b;                                                                                   \
    lim_a.ensure((const void *)f8_gemm_ring_kernel<NST, F8_FMT_E4M3, BT>, f8_ring_lds_bytes(NST, BT));                  \
    lim_b.ensure((const void *)f8_gemm_ring_kernel<NST, F8_FMT_E5M2, BT>, f8_ring_lds_bytes(NST, BT));                  \
    if (e5m2)                                                                                                           \
      f8_gemm_ring_kernel<NST, F8_FMT_E5M2, BT><<<grid, dim3(256), f8_ring_lds_bytes(NST, BT), stream>>>(a, tm, tn, per_xcd); \
    else                                                                                                                \
      f8_gemm_ring_kernel<NST, F8_FMT_E4M3, BT><<<grid, dim3(256), f8_ring_lds_bytes(NST, BT), stream>>>(a, tm, tn, per_xcd); \
  }
    if (small)
      MI_F8_RING(4, 64)
    else if (tiles_m * tiles_n <= 256)
      MI_F8_RING(8, 128)
    else
      MI_F8_RING(4, 128)
#undef MI_F8_RING
  }
  MI_HIP(hipGetLastError());
  return scratch.release();
}

}  // namespace mi
