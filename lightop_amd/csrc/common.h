// Shared device/host helpers of the gfx950 block-INT8 fused-MoE kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/lightop_mi355.h"

namespace lo {

constexpr int kWave = 64;   // CDNA wavefront
constexpr int kGroup = 128; // quantisation group along K and weight block edge

// Order of the 2 KB blocks (16 rows x 128 K-bytes) of a pre-shuffled expert weight:
// K-block-major, i.e. [K/128][N/16]: the blocks that neighbouring waves read at the same
// step of their K loops are contiguous in memory.  (Row-block-major order puts them
// K*16 bytes apart, which for K = 2048 is a 32 KB stride and piles the concurrent reads
// onto a few memory channels.)
#ifndef LO_SHUF_KB_MAJOR
#define LO_SHUF_KB_MAJOR 1
#endif
// byte offset of block (row block nb, K block kb) inside one expert
__host__ __device__ __forceinline__ int64_t shuf_block_off(int64_t nb, int64_t kb, int64_t NBLK, int64_t KB) {
  return (LO_SHUF_KB_MAJOR ? kb * NBLK + nb : nb * KB + kb) * 2048;
}
// the two strides of that formula, for kernels that advance kb with a scalar offset
__host__ __device__ __forceinline__ int shuf_nb_stride(int KB) { return LO_SHUF_KB_MAJOR ? 2048 : KB * 2048; }
__host__ __device__ __forceinline__ int shuf_kb_stride(int NBLK) { return LO_SHUF_KB_MAJOR ? NBLK * 2048 : 2048; }

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v2i __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef unsigned short v4u16 __attribute__((ext_vector_type(4)));
typedef unsigned short v8u16 __attribute__((ext_vector_type(8)));

// ---- error reporting (host) -------------------------------------------------
void set_error(const char *fmt, ...);
int check_launch(const char *what);
// bf16(silu(g)) for all 65536 bf16 patterns g, built on first use (per device).
int silu_table(hipStream_t stream, const uint16_t **table);
// T(act(g)) for all 65536 patterns g of the 16-bit type T (LO_BF16 / LO_F16), act = LO_ACT_SILU / LO_ACT_GELU.
int act_table(hipStream_t stream, int act, int dtype, const uint16_t **table);
// The gated activation of c1 [rows, 2I] from its table, followed by the 1x128 group quantisation
// (q [rows, I], s [rows, I/128]) or by the per-token quantisation (s [rows]; SiLU without a floor
// under the row maximum, as fuse_silu_mul_quant, GELU with per_token_quant_int8's), one launch each.
// row_mask (optional, [rows] bytes): rows whose byte is 0 are skipped.
int launch_act_mul_group_quant(const void *c1, int dtype, int act, int64_t rows, int64_t I, int8_t *q, float *s,
                               const uint8_t *row_mask, hipStream_t stream);
// fp32 rows (elementwise_f32.hip)
int launch_group_quant_f32(const float *x, int64_t groups, float eps, int8_t *q, float *s, hipStream_t stream);
int launch_act_mul_f32(const float *c1, int64_t rows, int64_t I, int act, float *out, hipStream_t stream);
int launch_act_mul_group_quant_f32(const float *c1, int act, int64_t rows, int64_t I, int8_t *q, float *s,
                                   const uint8_t *row_mask, hipStream_t stream);
int launch_moe_sum_f32(const float *in, float *out, const float *bias, const uint8_t *mask, int64_t M, int32_t topk,
                       int64_t H, float factor, const int32_t *num_local_tokens, hipStream_t stream);
int launch_act_mul_row_quant(const void *c1, int dtype, int act, int64_t rows, int64_t I, int8_t *q, float *s,
                             const int32_t *num_local_tokens, int32_t top_k, const int32_t *row_ids,
                             const uint8_t *row_mask, hipStream_t stream);

// The per-token quantisation alone, of activations [rows, I] that a gated first stage left; floored as above.
int launch_act_rows_quant(const void *act, int dtype, bool floored, int64_t rows, int64_t I, int8_t *q, float *s,
                          const uint8_t *row_mask, hipStream_t stream);

// Raises a kernel's dynamic-LDS limit once per device instead of on every launch (kernels that use
// more than the default 64 KB).  `done` is the call site's own static flag set, one bit per device.
int reserve_lds_once(const void *kernel, int bytes, unsigned long long *done);

#define LO_REQUIRE(cond, code, ...)  \
  do {                               \
    if (!(cond)) {                   \
      ::lo::set_error(__VA_ARGS__);  \
      return (code);                 \
    }                                \
  } while (0)

// ---- 16-bit float helpers (device) ------------------------------------------
__device__ __forceinline__ float bf16_to_f32(uint16_t h) {
  return __uint_as_float(static_cast<uint32_t>(h) << 16);
}

// Round-to-nearest-even (gfx950 has the conversion in hardware: v_cvt_pk_bf16_f32).
__device__ __forceinline__ uint16_t f32_to_bf16(float f) {
  return __builtin_bit_cast(uint16_t, static_cast<__bf16>(f));
}

__device__ __forceinline__ float f16_to_f32(uint16_t h) {
  return static_cast<float>(__builtin_bit_cast(_Float16, h));
}
// The conversion is kept opaque: written as a cast, the compiler folds a preceding fp32
// multiplication into v_fma_mixlo_f16 (a * b + 0 rounded straight to half), which rounds once where
// the definition rounds twice and turns a -0 product into +0.
__device__ __forceinline__ uint16_t f32_to_f16(float f) {
  uint32_t r;
  asm("v_cvt_f16_f32 %0, %1" : "=v"(r) : "v"(f));
  return static_cast<uint16_t>(r);
}

template <int DT> __device__ __forceinline__ float to_f32(uint16_t h) {
  if constexpr (DT == LO_BF16) return bf16_to_f32(h);
  else return f16_to_f32(h);
}
template <int DT> __device__ __forceinline__ uint16_t from_f32(float f) {
  if constexpr (DT == LO_BF16) return f32_to_bf16(f);
  else return f32_to_f16(f);
}

// exp(x) as a fixed sequence of IEEE single operations (Cody-Waite reduction,
// degree-7 polynomial, exact power-of-two scaling), so that the result does not
// depend on a math library.  Used for SiLU: g / (1 + exp(-g)).
__device__ __forceinline__ float det_expf(float x) {
  const float x_in = x;
  x = fminf(fmaxf(x, -87.0f), 88.72283f); // straight-line code: the ends are patched below
  float n = __builtin_rintf(x * 1.44269504088896341f);
  float r = __builtin_fmaf(n, -0.693145751953125f, x);
  r = __builtin_fmaf(n, -1.42860682030941723212e-6f, r);
  float p = 1.9841270114e-4f;
  p = __builtin_fmaf(p, r, 1.3888889225e-3f);
  p = __builtin_fmaf(p, r, 8.3333337680e-3f);
  p = __builtin_fmaf(p, r, 4.1666667908e-2f);
  p = __builtin_fmaf(p, r, 1.6666667163e-1f);
  p = __builtin_fmaf(p, r, 5.0000000000e-1f);
  p = __builtin_fmaf(p, r, 1.0f);
  p = __builtin_fmaf(p, r, 1.0f);
  int ni = static_cast<int>(n);
  int h = ni / 2;
  float a = __uint_as_float(static_cast<uint32_t>(h + 127) << 23);
  float b = __uint_as_float(static_cast<uint32_t>(ni - h + 127) << 23);
  float e = (p * a) * b;
  e = x_in > 88.72283f ? __uint_as_float(0x7f800000u) : e;
  return x_in < -87.0f ? 0.0f : e;
}

// act = T( T(silu(g)) * u ), everything in fp32 between the roundings.
template <int DT> __device__ __forceinline__ uint16_t silu_mul(uint16_t g16, uint16_t u16) {
  float g = to_f32<DT>(g16);
  float e = det_expf(-g);
  float sg = to_f32<DT>(from_f32<DT>(g / (1.0f + e)));
  return from_f32<DT>(sg * to_f32<DT>(u16));
}

// Any gated activation whose T(act(g)) sits in a 64K-entry table: act = T(T(act(g)) * u).
template <int DT>
__device__ __forceinline__ uint16_t act_mul_tab(const uint16_t *__restrict__ table, uint16_t g16, uint16_t u16) {
  return from_f32<DT>(to_f32<DT>(table[g16]) * to_f32<DT>(u16));
}

// ---- SiLU of bf16 gates on the transcendental unit ---------------------------------------------------------
// Two floats rounded to bf16 by one instruction and widened again.
typedef __bf16 v2bf16 __attribute__((ext_vector_type(2)));
typedef float v2f __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void round_pair_bf16(float a, float b, float &ra, float &rb) {
  const uint32_t p = __builtin_bit_cast(uint32_t, __builtin_convertvector((v2f{a, b}), v2bf16));
  ra = __uint_as_float(p << 16);
  rb = __uint_as_float(p & 0xffff0000u);
}

// act[i] = bf16(bf16(silu(bf16(g[i]))) * bf16(u[i])) as floats, with bf16(silu(g)) bit for bit what silu_mul<LO_BF16>
// computes: v_exp_f32 and v_rcp_f32 are good to an ulp of fp32, which is enough to round to bf16 correctly for every
// bf16 gate from kSiluHwMin up, given 1 + 2^-23 for the one in the denominator (silu(5.9375) lies three fp32 ulps below
// the middle between two bf16 numbers; the constant takes the quotient's error to the right side of it and moves no other
// gate).  Below, the reciprocal of 1 + exp(-g) is denormal and flushed: a wave that holds such a gate (or -inf) redoes those
// values the long way.  NaN gates give NaN.  A test drives every bf16 gate through it.
//
// 14 vector instructions per value, two of them transcendental, against about 36 for a table in LDS with its selects for
// the closed forms outside of it (gather, index arithmetic and conversions one by one): whole Qwen3-30B-A3B layer at 8192
// tokens 626 -> 607 us, at 2400: 264 -> 257; around 1 % on the DeepSeek-V3 share at 4096, within what two runs differ by.
constexpr float kSiluHwMin = -87.25f;
template <int N>
__device__ __forceinline__ void silu_mul_bf16(const float (&g)[N], const float (&u)[N], float (&act)[N]) {
  static_assert(N % 2 == 0, "values go in pairs");
  float gb[N], lowest = 0.0f;
#pragma unroll
  for (int i = 0; i < N; i += 2) {
    round_pair_bf16(g[i], g[i + 1], gb[i], gb[i + 1]);
    lowest = fminf(fminf(gb[i], gb[i + 1]), lowest);
    float s[2], ub[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const float e = __builtin_amdgcn_exp2f(gb[i + j] * -1.44269504088896341f);
      s[j] = gb[i + j] * __builtin_amdgcn_rcpf(1.00000011920928955078125f + e);
    }
    round_pair_bf16(s[0], s[1], s[0], s[1]);
    round_pair_bf16(u[i], u[i + 1], ub[0], ub[1]);
    round_pair_bf16(s[0] * ub[0], s[1] * ub[1], act[i], act[i + 1]);
  }
  if (__builtin_expect(__builtin_amdgcn_ballot_w64(lowest < kSiluHwMin) != 0, 0)) {
#pragma unroll
    for (int i = 0; i < N; ++i)
      if (gb[i] < kSiluHwMin) act[i] = bf16_to_f32(silu_mul<LO_BF16>(f32_to_bf16(gb[i]), f32_to_bf16(u[i])));
  }
}

// q = (int8) trunc(clamp(v / s, -128, 127))
__device__ __forceinline__ int quant_one(float v, float s) {
  float t = v / s;
  t = fmaxf(t, -128.0f);
  t = fminf(t, 127.0f);
  return static_cast<int>(t);
}

// The same value as quant_one(v, s) from y = 1.0f / s (one IEEE division per row instead of
// one per element): q = RN(v*y) is within an ulp of v/s, the remainder v - q*s is exact in
// a fused multiply-add, and RN(q + rem*y) is then the correctly rounded quotient (Markstein's
// theorem, valid for a correctly rounded reciprocal and no under/overflow).  Quotients
// of denormal magnitude may differ in the last bit; they truncate to 0 either way.  Not
// valid for s = inf (a row that holds an infinity) nor for a tiny s: callers take quant_one then.
__device__ __forceinline__ int quant_one_rcp(float v, float s, float y) {
  const float q = v * y;
  const float rem = __builtin_fmaf(-q, s, v);
  // one instruction for the two ends; a NaN quotient becomes -128 as in quant_one (v_med3_f32 of a NaN is the minimum)
  return static_cast<int>(__builtin_amdgcn_fmed3f(__builtin_fmaf(rem, y, q), -128.0f, 127.0f));
}

// The per-token rule's rounding: to nearest, ties to even.
__device__ __forceinline__ int rne_i8(float v) {
  v = fminf(fmaxf(v, -128.0f), 127.0f);
  return static_cast<int>(__builtin_rintf(v)); // v_rndne_f32
}

__device__ __forceinline__ uint32_t pack4_i8(int a, int b, int c, int d) {
  // byte 0 of each: v_perm_b32 selects 0-3 from its second operand, 4-7 from its first, 0x0c is zero
  return __builtin_amdgcn_perm(static_cast<uint32_t>(b), static_cast<uint32_t>(a), 0x0c0c0400u) |
         __builtin_amdgcn_perm(static_cast<uint32_t>(d), static_cast<uint32_t>(c), 0x04000c0cu);
}

__device__ __forceinline__ uint32_t quant4_rcp(const float *v, float s, float y) {
  return pack4_i8(quant_one_rcp(v[0], s, y), quant_one_rcp(v[1], s, y), quant_one_rcp(v[2], s, y), quant_one_rcp(v[3], s, y));
}
__device__ __forceinline__ uint32_t quant4_div(const float *v, float s) {
  return pack4_i8(quant_one(v[0], s), quant_one(v[1], s), quant_one(v[2], s), quant_one(v[3], s));
}
// four elements of one row -> four packed int8; y = 1.0f / s.  A small scale (a floor of zero lets it be one) is divided by: its
// reciprocal overflows below 2^-128, and the remainders lose bits before that.
__device__ __forceinline__ uint32_t quant4(const float *v, float s, float y) {
  return s >= 0x1p-100f && s < __builtin_inff() ? quant4_rcp(v, s, y) : quant4_div(v, s);
}

// The same for a group of 16-bit values, whose quotients are one multiplication: trunc(v * y) is trunc(v / s) for every value of
// the group if y is 1 / s to a few ulps, on the right side of it.  With the group's maximum b and a value a as integers (11 bits
// at most), v / s is 127 a / b times a power of two and the rounding of s; a quotient that is no integer is further than
// 1 / (127 a) of itself from one, which is more than 2^-18.  It is an integer n other than 0 where a = b, n = 127 (127 being
// prime), or where b is a multiple of 127 and s exact.  So only which side of 127 the maximum's own quotient rounds to has to be
// met, and an exact quotient is on the upper side.  floor: the least scale is floor / 127.  False where this does not hold - an
// infinity (a group's or the floor), a maximum so small that the floor, which is no 16-bit value, replaces it, or one whose scale
// a floor below 1e-10 lets become tiny - and the caller divides (group_quant8, quant4_div).
// 15 instead of 27 vector instructions for four values, and half of a row's: first GEMM of the Qwen3-30B-A3B layer at 8192 tokens
// 345.7 -> 334.0 us, whole layer with its router 566.5 -> 561.3; at 1531 tokens 180.1 -> 178.1, one token 18.16 -> 17.90.
__device__ __forceinline__ bool group_scale16(float amax, float floor, float &s, float &y) {
  const float top = fmaxf(amax, floor), r = 1.0f / 127.0f;
  const float q = top * r;
  s = __builtin_fmaf(__builtin_fmaf(-127.0f, q, top), r, q); // top / 127 correctly rounded (Markstein)
  const bool up = __builtin_fmaf(0x1p-18f, s, __builtin_fmaf(-127.0f, s, top)) >= 0.0f; // top / s rounds to 127 or above
  y = __builtin_amdgcn_rcpf(s) * (up ? 1.0f + 0x1p-21f : 1.0f - 0x1p-21f);
  // (with the default floor three comparisons: more of them cost the one-token kernels up to 4 %)
  return (floor >= 1e-10f && floor < __builtin_inff() && amax == 0.0f) ||
         (amax >= fmaxf(floor, 1e-10f) && amax < __builtin_inff());
}
// (a NaN becomes -128 as in quant_one)
__device__ __forceinline__ uint32_t quant4_mul(const float *v, float y) {
  int t[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) t[i] = static_cast<int>(__builtin_amdgcn_fmed3f(v[i] * y, -128.0f, 127.0f));
  return pack4_i8(t[0], t[1], t[2], t[3]);
}

// Eight values of a group of 16-bit values whose maximum is amax, and the group's scale.  A group that the multiplication does not
// hold for is quantised by one reciprocal where that holds: 8192 rows of 7168 with a floor above their maxima 30.5 us, with a
// division a value 38.5, without the attempt at the multiplication 29.1.  ONLY_DIV: at the default floor, below which next to no
// group's maximum lies, the division alone, which is less code (one token of the Qwen3-30B-A3B layer 18.06 -> 17.56 us).
template <bool ONLY_DIV = false>
__device__ __forceinline__ v2i group_quant8(const float (&v)[8], float amax, float floor, float &s) {
  float y;
  if (__builtin_expect(group_scale16(amax, floor, s, y), 1))
    return v2i{static_cast<int>(quant4_mul(&v[0], y)), static_cast<int>(quant4_mul(&v[4], y))};
  if (!ONLY_DIV && s >= 0x1p-100f) { // a finite maximum: s is what the division gives
    y = 1.0f / s;
    return v2i{static_cast<int>(quant4_rcp(&v[0], s, y)), static_cast<int>(quant4_rcp(&v[4], s, y))};
  }
  s = fmaxf(amax, floor) / 127.0f;
  return v2i{static_cast<int>(quant4_div(&v[0], s)), static_cast<int>(quant4_div(&v[4], s))};
}

// per_token_group_quant_int8 for the groups g = first + i * stride (reference:
// python/lightop/_lmslim_native/layers/gemm/int8_utils.py:74-122).  16 lanes own one group of
// 128 values (8 each); amax is reduced across those 16 lanes; the integers are those of IEEE quotients (group_quant8).
template <int DT>
__device__ __forceinline__ void group_quant_body(const uint16_t *__restrict__ x, int64_t groups, float eps,
                                                 int8_t *__restrict__ q, float *__restrict__ s, int64_t first,
                                                 int64_t stride, int sub) {
  for (int64_t g = first; g < groups; g += stride) {
    const v8u16 raw = *reinterpret_cast<const v8u16 *>(x + g * kGroup + sub * 8);
    float v[8];
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      v[i] = to_f32<DT>(raw[i]);
      amax = fmaxf(amax, fabsf(v[i]));
    }
#pragma unroll
    for (int d = 1; d < 16; d <<= 1) amax = fmaxf(amax, __shfl_xor(amax, d));
    float sc;
    const v2i packed = group_quant8(v, amax, eps, sc);
    *reinterpret_cast<v2i *>(q + g * kGroup + sub * 8) = packed;
    if (sub == 0) s[g] = sc;
  }
}

// per_token_quant_int8 (int8_utils.py:20-44: amax floored at 1e-10, s = amax / 127, q = rne(x * (127 / amax))): four
// wavefronts per row, blockDim.x / 256 rows per workgroup and pass, pieces of up to 8192 values kept in registers between
// the two steps.  Every wave of the workgroup makes the same number of passes.  red: 2 * 16 floats of LDS.
template <int DT>
__device__ __forceinline__ void row_quant_body(const uint16_t *__restrict__ x, int64_t rows, int64_t C,
                                               int8_t *__restrict__ q, float *__restrict__ s, int64_t block,
                                               int64_t nblocks, float *red) {
  constexpr int CH = 4;
  const int tid = threadIdx.x & 255, team = threadIdx.x >> 8, teams = blockDim.x >> 8;
  const int pieces = static_cast<int>(C / 8);
  int odd = 0; // two halves of `red` in turn: one barrier per pass
  for (int64_t base = block * teams; base < rows; base += nblocks * teams, odd ^= 1) {
    const int64_t row = base + team;
    const uint16_t *xr = x + (row < rows ? row : base) * C;
    v8u16 keep[CH];
    float amax = 1e-10f;
    auto widest = [&](const v8u16 raw) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < 8; ++i) amax = fmaxf(amax, fabsf(to_f32<DT>(raw[i])));
    };
#pragma unroll
    for (int j = 0; j < CH; ++j) // (a thread past the row re-reads its start: the same maximum)
      keep[j] = *reinterpret_cast<const v8u16 *>(xr + (tid + 256 * j < pieces ? tid + 256 * j : 0) * 8);
#pragma unroll
    for (int j = 0; j < CH; ++j) widest(keep[j]);
    for (int p = tid + 256 * CH; p < pieces; p += 256) widest(*reinterpret_cast<const v8u16 *>(xr + p * 8));
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) amax = fmaxf(amax, __shfl_xor(amax, d));
    if ((threadIdx.x & 63) == 0) red[odd * 16 + (threadIdx.x >> 6)] = amax;
    __syncthreads();
    const float *const r4 = red + odd * 16 + team * 4;
    amax = fmaxf(fmaxf(r4[0], r4[1]), fmaxf(r4[2], r4[3]));
    if (row >= rows) continue;
    const float inv = 127.0f / amax;
    if (tid == 0) s[row] = amax / 127.0f;
    auto emit = [&](int p, const v8u16 raw) __attribute__((always_inline)) {
      int b[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) b[i] = rne_i8(to_f32<DT>(raw[i]) * inv);
      *reinterpret_cast<v2i *>(q + row * C + p * 8) = v2i{static_cast<int>(pack4_i8(b[0], b[1], b[2], b[3])),
                                                         static_cast<int>(pack4_i8(b[4], b[5], b[6], b[7]))};
    };
#pragma unroll
    for (int j = 0; j < CH; ++j)
      if (tid + 256 * j < pieces) emit(tid + 256 * j, keep[j]);
    for (int p = tid + 256 * CH; p < pieces; p += 256) emit(p, *reinterpret_cast<const v8u16 *>(xr + p * 8));
  }
}

// The quantisation of the activations that rides in an alignment launch.
struct QuantJob {
  const uint16_t *x; // [M, H] bf16, or fp16
  int64_t M, H;
  float eps;         // floor of a group's maximum (rows: 1e-10)
  int8_t *q;
  float *s;          // [M, H/128], or [M] per row
};
// Workgroup `block` of `nblocks` that share the job (blockDim.x a multiple of 256).
template <bool PER_ROW, int DT>
__device__ __forceinline__ void quant_job(const QuantJob &j, int64_t block, int64_t nblocks) {
  if constexpr (PER_ROW) {
    __shared__ float red[32];
    row_quant_body<DT>(j.x, j.M, j.H, j.q, j.s, block, nblocks, red);
  } else {
    const int per_block = blockDim.x >> 4; // groups a workgroup handles per pass
    group_quant_body<DT>(j.x, j.M * (j.H / kGroup), j.eps, j.q, j.s, block * per_block + (threadIdx.x >> 4),
                         nblocks * per_block, threadIdx.x & 15);
  }
}

// The quantisation of x [M, H] (per group, or per row) and the routing alignment with the quantisation riding in the
// alignment's (second) launch: they are independent, and at decode sizes a launch costs as much
// as either.  scratch: the counters of the form with a launch for them (lo_moe_align_scratch_bytes);
// returns LO_ENOTSUP when that form is the one to take and they are missing - the caller then launches
// the two stages separately.
int launch_quant_align(const void *x, int dtype, bool per_row, int64_t M, int64_t H, float eps, int8_t *q, float *s,
                       const void *topk_ids, int ids_dtype, int64_t numel, int32_t num_experts,
                       int32_t block_size, const int32_t *expert_map, int32_t *sorted_ids, int64_t sorted_cap,
                       int32_t *expert_ids, int64_t expert_ids_cap, int32_t *num_tokens_post_pad,
                       uint8_t *slot_mask, void *scratch, int64_t scratch_bytes, hipStream_t stream);

} // namespace lo
