// Argument block and launchers shared by the grouped block-INT8 GEMM kernels.
#pragma once
#include "common.h"

namespace lo {

struct GemmArgs {
  const int8_t *A;       // [a_rows, K]
  const float *As;       // [a_rows, K/128]
  const int8_t *W;       // [E, N, K]
  const float *Ws;       // [E, NB, K/128]
  uint16_t *C;           // plain: [num_valid, N]
  int8_t *A2q;           // fused: [num_valid, I]
  float *A2s;            // fused: [num_valid, I/128]
  const float *topk_w;   // [num_valid]
  const int32_t *sorted; // [>= m_blocks*BM]
  const int32_t *expert_ids;
  const int32_t *ntpp;
  int64_t num_valid;
  int64_t a_rows;        // rows of A / As
  int64_t N;             // weight rows per expert (2I for the fused first GEMM)
  int64_t K;
  int32_t top_k;
  uint32_t row_mul;      // slot -> token row without a division: __umulhi(2 * slot, row_mul) >> row_shift (set_top_k)
  int32_t row_shift;
  int32_t n_tiles;       // workgroups along N
  int32_t E;             // experts held by W
  int32_t experts_routed; // experts the routing spreads the slots over (estimate, for tile order)
  int32_t mul_routed;
  int32_t w_shuffled;    // W is in the pre-shuffled layout (shuffle.hip)
  int32_t skip_nonlocal; // blocks of expert -1: leave the output rows untouched
  int32_t w4;            // W is packed int4 (load-time layout), Ws is [E, K/128, N]
  int32_t per_channel;   // As is [a_rows], Ws is [E, N]: scales applied once, after the whole-K int32 sum
  int32_t stream;        // 64- and 128-token tiles: experts have about one token block
  int32_t coarse_fill;   // 160-token tiles: round the token fragments in use up to 8
  int32_t out_f16;       // C holds IEEE half instead of bf16; fused: the values between the stages are rounded to half
  int32_t out_f32;       // C holds the fp32 sums themselves (block form, weight-streaming kernel only)
  int32_t fused;         // the fused epilogue's activation: kActSiluBf16 or kActTable (plain: 0)
  const uint16_t *act_table; // kActTable: T(act(g)) of every 16-bit pattern g
};

// Gated activations of a fused first stage; the kernels' FUSED_ACT parameter, 0 being a plain GEMM.  SiLU of bf16 rows is
// computed and comes in all three scale orders.  The others are looked up, 128 KB in L2: GELU, and SiLU of fp16 gates, which
// the short forms of exp and reciprocal do not round right (the long way costs the epilogue more than the lookup: Qwen3-30B-A3B
// layer at 8000 tokens 627 us against 618).  They exist in the default order, and in the kernels for 64 and 128 tokens and
// for row-major weights; otherwise the first stage is a plain GEMM and an activation launch, which with the weight-streaming
// kernel is as fast, its plain workgroups being finer (24 tokens: 100.0 plain, 101.1 fused).  Plain / fused, us:
// Qwen3-30B-A3B layer, fp16 333 tokens 133.8 / 124.7, 4000: 399 / 375, 8000: 684 / 618; GELU 100: 117.6 / 114.3, 8001: 639 /
// 598; DeepSeek-V3 share, fp16 2000: 326 / 314; Qwen3-235B-A22B-shaped layer, fp16 300: 434 / 409, row-major 492 / 468.
constexpr int kActSiluBf16 = 1, kActTable = 2;
// act[i] = T(T(act(T(g[i]))) * T(u[i])) as floats.
template <int FUSED_ACT, int N>
__device__ __forceinline__ void gated_act(const GemmArgs &a, const float (&g)[N], const float (&u)[N], float (&act)[N]) {
  if constexpr (FUSED_ACT == kActSiluBf16) {
    silu_mul_bf16<N>(g, u, act);
  } else {
    if (a.out_f16) {
#pragma unroll
      for (int i = 0; i < N; ++i) act[i] = f16_to_f32(act_mul_tab<LO_F16>(a.act_table, f32_to_f16(g[i]), f32_to_f16(u[i])));
    } else {
#pragma unroll
      for (int i = 0; i < N; ++i) act[i] = bf16_to_f32(act_mul_tab<LO_BF16>(a.act_table, f32_to_bf16(g[i]), f32_to_bf16(u[i])));
    }
  }
}
// (K <= 16384: what the kernels with such an epilogue hold scales for)
inline bool fused_table_supports(int64_t K, int block_size_m, int flags) {
  if (flags & (LO_GEMM_SEPARATE_ORDER | LO_GEMM_FUSED_SCALE | LO_GEMM_FORCE_STREAMING)) return false;
  if (K > 128 * kGroup) return false;
  const bool rows = !(flags & (LO_GEMM_W_PRESHUFFLED | LO_GEMM_W4));
  return block_size_m == 64 || block_size_m == 128 || (rows && (block_size_m == 16 || block_size_m == 32));
}
// Per-channel scales: a first stage that ends with the gated activation in 16 bits, C [num_valid, I], instead of gate and up
// (the row's quantisation follows in its own launch either way).  From 64 tokens on, where the kernels are not the
// weight-streaming one.  Plain / gated, whole path, us: Qwen3-30B-A3B-shaped layer at 300 tokens 127.7 / 124.0, at 700:
// 147.6 / 141.0, at 8000: 555 / 525, fp16 608 / 572; int4 at 300 tokens of the Qwen3-235B-A22B-shaped layer 252 / 245, at 6000:
// 1100 / 1061.
inline bool gated_channel_supports(int64_t K, int block_size_m, int flags) {
  if (flags & LO_GEMM_FORCE_STREAMING) return false;
  if (flags & LO_GEMM_W4) return block_size_m >= 128 && K <= 128 * kGroup;
  return block_size_m >= 64;
}
// Launcher macro MACRO(FUSED_ACT) of a per-channel GEMM.
#define LO_GATED_DISPATCH(a, fused_act, MACRO)                        \
  do {                                                                \
    if (!(fused_act)) MACRO(0);                                       \
    else if ((a).fused == ::lo::kActTable) MACRO(::lo::kActTable);    \
    else MACRO(::lo::kActSiluBf16);                                   \
  } while (0)
// Launcher macro MACRO(scale order, FUSED_ACT) for a fused first stage.
#define LO_FUSED_DISPATCH(a, ord, MACRO)                                                \
  do {                                                                                  \
    if ((a).fused == ::lo::kActTable) MACRO(::lo::kOrdContract, ::lo::kActTable);  \
    else LO_ORD_DISPATCH(ord, MACRO, ::lo::kActSiluBf16);                               \
  } while (0)

// A workgroup's start is a chain of memory round trips in front of its first operand: the arguments (a kernel's argument
// block is read field by field where the fields are used, behind the branches), the blocks in use, the block's expert, the slot
// ids.  start_args() has every argument that a start needs asked for in one go (a.E goes through it, to order it first);
// block_unused() takes what is loaded by the block index alone in one condition, which keeps those loads above the branch.
// Two round trips are left (24 tokens of the Qwen3-30B-A3B layer 100.5 -> 99.7 us, 700 per-channel ones 141.0 -> 139.8).
__device__ __forceinline__ int start_args(const GemmArgs &a) {
  int E;
  asm("" : "=s"(E) : "0"(a.E), "s"(a.A), "s"(a.As), "s"(a.W), "s"(a.Ws), "s"(a.sorted), "s"(a.expert_ids), "s"(a.ntpp),
      "s"(a.num_valid), "s"(a.a_rows), "s"(a.N), "s"(a.K), "s"(a.row_mul));
  return E;
}
// Whether the block starting at `first` is past the list.  (The second half is never true: no slot id is INT_MIN.)
__device__ __forceinline__ bool block_unused(int32_t first, int32_t blocks_end, int expert, int slots) {
  constexpr int kNever = -2147483647 - 1;
  __builtin_amdgcn_sched_barrier(0); // all of the loads before the first wait
  return (first >= blocks_end) | ((expert == kNever) & (__builtin_amdgcn_readfirstlane(slots) == kNever));
}

// Shape of the plain (not fused) weight-streaming workgroup: waves, and 16-row fragments per wave (gemm_ws.hip; the tile
// query reports the same numbers).  Two fragments rather than four: what a stage cannot fill with whole rounds of resident
// workgroups it loses, and a workgroup of half the bytes halves that.  us with four / two, one pass of the layer: per-channel
// Qwen3-30B-A3B layer at 20 tokens 96.6 / 90.7, per-channel DeepSeek-V3 share at 40: 180 / 169.5, int4 per-channel at 38: 190.5 /
// 185, block form, Qwen3-30B-A3B layer at 32 tokens 101.6 / 99.0 (one fragment with three or four K blocks in flight: 3 to
// 14 % slower).  Four for the block form's long outputs, which have tiles enough (DeepSeek-V3, 28 per expert), and for int4
// weights with K-group scales, whose workgroups fill their scale table first (60 tokens 231.6 with four, 234.7 with two).
constexpr int kWsPlainWaves = 4;
inline int ws_plain_fragments(const GemmArgs &a, int token_fragments) {
  if (token_fragments > 2) return token_fragments == 4 ? 2 : 1;
  if (a.per_channel) return 2;
  return a.w4 || a.N > 4096 ? 4 : 2;
}

// Division of a slot id below 2^31 by top_k as a multiplication: with L = ceil(log2 d) and m = floor(2^(31+L) / d) + 1,
// floor(n * m / 2^(31+L)) is the quotient for every n < 2^31 (m overshoots 2^(31+L) / d by less than 2^-31 of it), and m
// fits 32 bits.  A 32-bit division is some twenty dependent instructions in front of a tile's first copies.
inline void set_top_k(GemmArgs &a, int32_t d) {
  int L = 0;
  while ((1ll << L) < d) ++L;
  a.top_k = d;
  a.row_mul = static_cast<uint32_t>((1ull << (31 + L)) / static_cast<uint64_t>(d) + 1);
  a.row_shift = L;
}
// Token row of a slot id of the sorted list (padding and ids out of range: row 0, whose values are never used).
__device__ __forceinline__ int token_row(const GemmArgs &a, int64_t slot) {
  const uint32_t row = __umulhi(2u * static_cast<uint32_t>(slot), a.row_mul) >> a.row_shift;
  return slot < a.num_valid ? static_cast<int>(row) : 0;
}

// Routed weight of a slot, 1 where it is not wanted: asked for at a kernel's start, in front of the K loop's loads.  In the
// epilogue it is a round trip to memory for every token fragment, each in a branch of its own.  Weight-streaming kernel,
// Qwen3-30B-A3B layer at 24 / 60 tokens 96.1 -> 95.6, 110.0 -> 109.6 us, DeepSeek-V3 share at 160 234.7 -> 234.3; 64-token int4
// tiles, 400 tokens 282.0 -> 281.1.  (The 64-token int8 kernels gain nothing: 333 tokens 121.1 / 121.3, 500: 124.7 / 125.4.)
__device__ __forceinline__ float slot_weight(const GemmArgs &a, int64_t slot) {
  return a.mul_routed ? a.topk_w[slot < a.num_valid ? slot : 0] : 1.0f;
}

// The 16-bit form a plain epilogue stores: bf16, or IEEE half when the caller's activations are fp16.
// `body(cvt)` is run with the conversion of the output type; the choice is one wave-uniform branch
// around the caller's loops, so the bf16 path pays nothing per value (a per-value select cost the
// activation-stationary second GEMM 10 %).
template <typename Body>
__device__ __forceinline__ void with_out16(int f16, Body body) {
  if (__builtin_expect(f16 != 0, 0)) body([](float v) { return f32_to_f16(v); });
  else body([](float v) { return f32_to_bf16(v); });
}

// Order of the scale arithmetic per 128-wide K block (d = the block's exact int32 sum):
//   kOrdContract   acc = fma(f32(d) * a_s, b_s, acc)    the default: what the reference's Triton line
//                  `accumulator += tl.dot(a, b) * a_scale * b_scale` (int8.py:499-508) compiles to with
//                  the AMD backend's default enable_fp_fusion; three vector instructions per element,
//                  two in the kernels that fold without a conversion (fold_biased)
//   kOrdSeparate   acc = acc + (f32(d) * a_s) * b_s     the same line without fp fusion; four instructions
//                  (LO_GEMM_SEPARATE_ORDER)
//   kOrdFusedScale acc = fma(f32(d), a_s * b_s, acc)    two instructions, last-ulp differences in fp32
//                  (LO_GEMM_FUSED_SCALE)
// The CPU checker restates the first two bit for bit.
constexpr int kOrdSeparate = 0, kOrdFusedScale = 1, kOrdContract = 2;
inline int scale_order(int flags) {
  if (flags & LO_GEMM_SEPARATE_ORDER) return kOrdSeparate;
  return (flags & LO_GEMM_FUSED_SCALE) ? kOrdFusedScale : kOrdContract;
}
// One accumulator element.  sc = a_s * b_s is read by kOrdFusedScale only, as and bs by the other two.
template <int ORD>
__device__ __forceinline__ float fold_elem(int d, float sc, float as, float bs, float acc) {
  if constexpr (ORD == kOrdFusedScale) {
    return __builtin_fmaf(static_cast<float>(d), sc, acc);
  } else if constexpr (ORD == kOrdContract) {
    return __builtin_fmaf(static_cast<float>(d) * as, bs, acc);
  } else {
    float t = static_cast<float>(d) * as;
    t = t * bs;
    return acc + t;
  }
}
// The contracted fold without a conversion: two vector instructions per element, and bit for bit the three of fold_elem.
// The MFMA chain starts from the integer 2^23 instead of 0, so that the K block's sum d leaves it as the integer 2^23 + d.
// Read as a float, an integer of up to 24 bits is that integer times 2^-149: below 2^23 it is a denormal, from there on a
// normal number of the first binade, and both have the same spacing.  So with A = a_s * 2^85
//     fma(m, A, -2^-126 * A)  =  round(((2^23 + d) - 2^23) * a_s * 2^-64)  =  round(d * a_s) * 2^-64,
// the subtraction being exact inside the fused operation because 2^-126 * A is, and
//     fma(that, b_s * 2^64, acc)
// is the second step of the contracted order.  (A bias that is no power of two, as the usual 1.5 * 2^23, has a rounded product
// with a_s.)  |d| < 2^23 for any K block of int8 operands: 128 * 2^14 = 2^21.  v_fma_f32 takes denormals at full rate.
// It holds while nothing on the way leaves the normal range: |a_s| zero or in [2^-62, 2^43), |b_s| below 2^64.  The
// quantisation's scales lie between 2^-41 and the largest 16-bit value / 127, so that only rows of more than 10^15, weight
// scales of 10^19, or a caller's own scales ever leave it; kernels fold a tile that holds such a scale the long way.
constexpr int kFoldBias = 0x00800000;
__device__ __forceinline__ float fold_token_scale(float as) { return as * 0x1p85f; }
__device__ __forceinline__ float fold_weight_scale(float bs) { return bs * 0x1p64f; }
__device__ __forceinline__ bool fold_token_scale_ok(float as) {
  const float v = fabsf(as);
  return v == 0.0f || (v >= 0x1p-62f && v < 0x1p43f); // (a NaN is refused)
}
__device__ __forceinline__ bool fold_weight_scale_ok(float bs) { return fabsf(bs) < 0x1p64f; }
// m: the biased sum; as, bs: scales that went through the two functions above; as_bias = fold_bias(as).
__device__ __forceinline__ float fold_bias(float as) { return as * -0x1p-126f; }
__device__ __forceinline__ float fold_biased(int m, float as, float as_bias, float bs, float acc) {
  return __builtin_fmaf(__builtin_fmaf(__builtin_bit_cast(float, m), as, as_bias), bs, acc);
}
// Three-way dispatch of a launcher macro on the order: LO_ORD_DISPATCH(ord, MACRO, args...) expands to
// MACRO(order constant, args...).
#define LO_ORD_DISPATCH(ord, MACRO, ...)                                   \
  do {                                                                     \
    if ((ord) == ::lo::kOrdContract) MACRO(::lo::kOrdContract, __VA_ARGS__);      \
    else if ((ord) == ::lo::kOrdSeparate) MACRO(::lo::kOrdSeparate, __VA_ARGS__); \
    else MACRO(::lo::kOrdFusedScale, __VA_ARGS__);                         \
  } while (0)

// Buffer addressing: a wave-uniform 128-bit resource (base, extent) + one 32-bit lane
// offset + one scalar offset.  The K loop then advances a scalar only, no per-lane 64-bit
// address arithmetic, and a read past the extent returns zero instead of faulting.
typedef __amdgpu_buffer_rsrc_t brsrc;
__device__ __forceinline__ brsrc make_rsrc(const void *base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, static_cast<int>(bytes), 0x00020000);
}
constexpr int kCacheDefault = 0;
constexpr int kCacheStream = 2; // "nt": data that is read once (weights in the streaming regime)
template <int AUX = kCacheDefault>
__device__ __forceinline__ v4i bld16(brsrc r, int voff, int soff) {
  return __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, AUX);
}
__device__ __forceinline__ float bld_f32(brsrc r, int voff, int soff) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
}
__device__ __forceinline__ void bst16(brsrc r, v4i v, uint32_t voff, int soff) { // nothing past the extent
  __builtin_amdgcn_raw_buffer_store_b128(v, r, static_cast<int>(voff), soff, 0);
}

// Consecutive workgroup ids are dealt round-robin to the 8 XCDs, each with its own L2.
// The logical tile list is cut into chunks of (G token blocks x all weight tiles): the
// tiles of a chunk share token rows, and neighbouring token blocks mostly share an
// expert's weights; G is about one expert's worth of token blocks, so that an expert's
// weights are fetched into one L2 only.  Chunks are dealt round-robin to the XCDs, and the workgroups that
// an XCD receives one after the other walk through one chunk, so what is shared is
// fetched into that XCD's L2 once; blocks of experts that are not on this rank (which
// cluster by expert id) still spread evenly over all XCDs.
__device__ __forceinline__ bool tile_of(int bid, int n_tiles, int m_blocks, int G, int &mb, int &nt) {
  constexpr int XCD = 8;
  const int xcd = bid % XCD, slot = bid / XCD;
  const int span = G * n_tiles;                      // tiles per chunk
  const int chunk = (slot / span) * XCD + xcd, in = slot % span;
  const int first = chunk * G;
  if (first >= m_blocks) return false;
  const int gsz = (m_blocks - first < G) ? (m_blocks - first) : G;
  nt = in / G;
  const int off = in - nt * G;
  if (off >= gsz) return false;
  mb = first + off;
  return true;
}

// Output of the 32x32-MFMA kernels.  In the accumulator layout a lane (r = lane & 31, c = lane >> 5)
// holds, of one 32-token x 64-column piece, token r and columns rb*32 + 8q + 4c + i: four
// consecutive bf16 per (rb, q).  Stored directly that is 8 bytes to each of 64 different token
// rows per instruction, and the texture path, which also carries the operand loads these
// kernels are bound by, spends a cycle per row touched.  Each wave therefore turns its piece
// around in LDS (LDS operations of one wave execute in order: no barrier) and stores whole
// 128-byte row segments, eight rows per instruction.
//   stg   32 * kStgPitch bytes of LDS owned by this wave
//   o     the lane's 2 x 4 packed column quadruples
//   slot  output row of token r, or -1 (lanes r and r + 32 agree)
//   C     + slot * N + col0: first of the piece's 64 columns; 16-byte aligned
constexpr int kStgPitch = 64 * 2 + 16; // bytes per staged token row: 16 mod 128 keeps both passes conflict-free
__device__ __forceinline__ void wave_store_32x64_bf16(int8_t *stg, const v4u16 (&o)[2][4], int slot, uint16_t *C,
                                                      int64_t N, int64_t col0, int lane) {
  const int r = lane & 31, c = lane >> 5;
#pragma unroll
  for (int rb = 0; rb < 2; ++rb)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      *reinterpret_cast<v4u16 *>(stg + r * kStgPitch + (rb * 32 + 8 * q + 4 * c) * 2) = o[rb][q];
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int tok = (lane >> 3) + 8 * j;
    const v4i v = *reinterpret_cast<const v4i *>(stg + tok * kStgPitch + (lane & 7) * 16);
    const int ft = __shfl(slot, tok);
    if (ft >= 0) *reinterpret_cast<v4i *>(C + static_cast<int64_t>(ft) * N + col0 + (lane & 7) * 8) = v;
  }
  __builtin_amdgcn_wave_barrier();
}

// Kernel a stage is served by, and its workgroup shape (gemm_api.hip).
int pick_gemm_kernel(const GemmArgs &a, bool fused_act, int block_size_m, int flags);
void describe_gemm_kernel(int kernel, bool fused_act, int block_size_m, bool rows, const GemmArgs &a, lo_moe_tile *t);

// Decode-size whole path in two launches (gemm_dec.hip): weights in the load-time layout, bf16 or fp16 rows.
struct DecProblem {
  const void *x;
  int dtype;
  int64_t M, H, I;
  int32_t E, num_experts, top_k;
  const int8_t *w1;
  const float *w1s;
  const int8_t *w2;
  const float *w2s; // block scales, K-group scales [E, K/128, N] (LO_GEMM_W4) or, with `channel`, one scale per row
  const float *topk_w;
  const void *topk_ids;
  int ids_dtype;
  const int32_t *expert_map;
  int mul_on_input;
  float factor;
  const void *shared_output;
  void *act; // room for [M * top_k, I] 16-bit activations: the front of the caller's cache13
  void *out;
  bool channel;
};
// Whether the path is taken: by sizes, element type and flags alone, so that the tile query asks with the pointers null.
bool decode_path_applies(const DecProblem &d, int flags);
void decode_path_waves(int32_t top_k, int64_t H, int *gemm1_waves, int *gemm2_waves);
int launch_decode_path(const DecProblem &d, int flags, hipStream_t stream); // LO_ENOTSUP if it is not

// lo_moe_gemm_w8a8, and with `fused` its gated form (N = 2I, C [num_valid, I]).
int launch_gemm_w8a8(const int8_t *A, const float *As, const int8_t *W, const float *Ws, void *C, int c_dtype, int fused,
                     const uint16_t *act_table, const float *topk_w, const int32_t *sorted_ids, const int32_t *expert_ids,
                     const int32_t *num_tokens_post_pad, int64_t sorted_cap, int64_t num_valid, int64_t a_rows, int32_t E,
                     int32_t num_experts, int64_t N, int64_t K, int32_t top_k, int32_t block_size_m, int mul_routed,
                     int flags, hipStream_t stream);
// The fused first stage with a given activation (lo_moe_gemm1_silu_quant_block_int8 is this with kActSiluBf16).
int launch_gemm1_act_quant(const int8_t *A, const float *As, const int8_t *W, const float *Ws, int8_t *A2q, float *A2s,
                           int fused, bool f16, const uint16_t *act_table, const float *topk_w, const int32_t *sorted_ids,
                           const int32_t *expert_ids, const int32_t *num_tokens_post_pad, int64_t sorted_cap,
                           int64_t num_valid, int64_t a_rows, int32_t E, int32_t num_experts, int64_t I, int64_t K,
                           int32_t top_k, int32_t block_size_m, int mul_routed, int flags, hipStream_t stream);
// Weight-streaming kernels (gemm_ws.hip): block_size_m in {16, 32, 64, 128}.
int launch_gemm_ws(const GemmArgs &a, bool fused_act, int block_size_m, int flags, int64_t m_blocks,
                   hipStream_t s);
// LDS-tiled kernels (gemm_tile.hip): block_size_m 64 or 128, compute-bound regime.
int launch_gemm_tile(const GemmArgs &a, bool fused_act, int block_size_m, int flags, int64_t m_blocks,
                     hipStream_t s);
bool gemm_tile_supports(const GemmArgs &a, bool fused_act, int block_size_m);
// Activation-stationary kernel (gemm_as.hip): plain epilogue, block_size_m 64 or 128, short K.
int launch_gemm_as(const GemmArgs &a, int flags, int block_size_m, int64_t m_blocks, hipStream_t s);
bool gemm_as_supports(const GemmArgs &a, bool fused_act, int block_size_m);

// 128-token kernel, two four-wave workgroups per compute unit (gemm_t128.hip): pre-shuffled int8 weights.
int launch_gemm_t128(const GemmArgs &a, bool fused_act, int block_size_m, int flags, int64_t m_blocks, hipStream_t s);
bool gemm_t128_supports(const GemmArgs &a, bool fused_act, int block_size_m);
// Row-major int8 weights, block or per-channel scales (gemm_t128.hip): block_size_m 16, 32, 64 or 128.
bool gemm_rows_supports(const GemmArgs &a, bool fused_act, int block_size_m);
int launch_gemm_rows(const GemmArgs &a, bool fused_act, int block_size_m, int flags, int64_t m_blocks, hipStream_t s);
// W4A8 LDS-tiled kernel (gemm_w4.hip): block_size_m 64.
int launch_gemm_w4_tile(const GemmArgs &a, bool fused_act, int flags, int64_t m_blocks, hipStream_t s);
bool gemm_w4_tile_supports(const GemmArgs &a, bool fused_act, int block_size_m);
// Per-channel LDS-tiled kernel (gemm_pc.hip): block_size_m 64 or 128.
int launch_gemm_pc(const GemmArgs &a, bool fused_act, int block_size_m, int64_t m_blocks, hipStream_t s);
bool gemm_pc_supports(const GemmArgs &a, int block_size_m);

} // namespace lo
