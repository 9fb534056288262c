// Grouped block-INT8 GEMM for gfx950, activation-stationary form for a short K (the
// second GEMM of a layer with a small intermediate size).
//
// With K of a few hundred bytes the 64 gathered token rows of a token block fit in LDS
// whole (64 x K bytes plus their group scales).  A workgroup loads them once and then
// walks several 256-row weight tiles with them: the K loop needs no barrier, no LDS
// write and no token reload, the weight prefetch (two K blocks deep) runs on across tile boundaries, and the
// gather of sorted_token_ids is paid once per token block instead of once per tile.
// Each wave owns 64 rows x 64 tokens as 4 x 4 fragments of v_mfma_i32_16x16x64_i8 (weights as the A operand);
// reference: Triton fused_moe_kernel, python/lightop/_lmslim_native/layers/fused_moe/int8.py:485-541.
#include <type_traits>

#include "gemm.h"

namespace lo {

constexpr uint32_t kAsMaxOut = 0xfff00000u; // bytes of an output that a descriptor addresses; an offset that none of them has

// KBT: K / 128 as a compile-time constant (a multiple of three, so that a tile starts on ring buffer 0),
// or 0 for any K.  With it a tile's steps and its stores are straight-line code: the compiler then
// knows how many memory operations follow each weight load and waits for exactly those; in the
// general form the stores sit in a branch, the wait counts assume they did not happen, and after
// every tile the wave waits for loads it has only just issued.  (Instantiated for the Qwen3-30B-A3B layer's K = 768; other K were not
// measured with straight-line stores.)  Straight-line stores go through a descriptor of the output
// (< 4 GiB), padding tokens past its end.
template <int ORD, int KBT = 0>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
void moe_gemm_as_kernel(const GemmArgs a, int m_blocks, int group_m,
                                                          int n_groups, int n_cnt, int sub_shift) {
  extern __shared__ __attribute__((aligned(16))) int8_t smem[];
  constexpr int kTileM = 64;
  const int K = static_cast<int>(a.K);
  const int KB = K / kGroup;
  // Tokens in operand order: K half kh of K block kb of token fragment tb is the 1 KB at ((2 kb + kh) * 4 + tb) * 1024, lane after
  // lane.  A read of 64 consecutive pieces has no bank conflict (SQ_LDS_BANK_CONFLICT of the Qwen3-30B-A3B layer's second stage at
  // 8192 tokens 1.08e7 -> 3.3e6, the output staging's) and the rows need no registers on their way here.
  int8_t *const sA = smem;
  float *const sS = reinterpret_cast<float *>(smem + kTileM * K); // [KB][64]
  // per-wave staging of 16 output rows x 64 columns (bf16), for row-contiguous stores
  int8_t *const sStage = smem + kTileM * K + KB * kTileM * 4;
  int32_t *const sFlag = reinterpret_cast<int32_t *>(sStage + 4 * 16 * kStgPitch); // [wave]: a scale that the biased fold does not take
  float *const sB = reinterpret_cast<float *>(sFlag + 4);                          // weight-block scales of the workgroup's tiles
  // The contracted order folds without a conversion (fold_biased), or with one where the scales do not allow that.  In 16x16
  // fragments, whose bias is four registers: sixteen, beside 64 accumulators, 96 registers of weights and two fragments of 32x32,
  // spill.  With the weight-block scales in LDS, not in the ring of weights: second stage of the Qwen3-30B-A3B layer at 8192
  // tokens 223 -> 219 us, whole layer with its router 561 -> 553.
  constexpr bool kBiased = ORD == kOrdContract;

  int mb, ng;
  if (!tile_of(blockIdx.x, n_groups, m_blocks, group_m, mb, ng)) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wr = __builtin_amdgcn_readfirstlane(tid >> 6); // which 64 weight rows of a tile
  const int r = lane & 15, q = lane >> 4;
  // The start is two round trips: the ids and the block's expert, all of them, then everything that depends on them.  One after the
  // other they were seven.  With the tokens in operand order and the straight-line stores: Qwen3-30B-A3B layer with its router
  // at 8192 tokens 545.4 -> 540.9 us, 12000: 740.2 -> 736.4, 24000: 1491 -> 1487 (on a slower card 583.5, 578.9 with order and
  // stores alone, 575.4).
  const int32_t *const ids = a.sorted + static_cast<int64_t>(mb) * kTileM;
  const int32_t blocks_end = a.ntpp[0];
  const int e_raw = a.expert_ids[mb >> sub_shift];
  int32_t f[4]; // slots of the tokens this lane holds in the accumulator layout
#pragma unroll
  for (int tb = 0; tb < 4; ++tb) f[tb] = ids[tb * 16 + r];
  const int32_t f_lane = ids[lane], f_row = ids[wr * 16 + r];
  if (static_cast<int64_t>(mb) * kTileM >= blocks_end) return;
  // mb counts 64-token pieces; an alignment block of 128 tokens is two of them (sub_shift = 1), and
  // a piece that holds padding only is skipped
  // An expert_map entry outside the weight tensor is treated like an expert of another rank, but its
  // rows are always zero-filled: the slot mask of the alignment counts such a slot as local.
  const bool e_oob = e_raw >= a.E;
  const int e = e_oob ? -1 : e_raw;
  if (sub_shift && __builtin_amdgcn_ballot_w64(f_lane < a.num_valid) == 0) return;
  const int64_t N = a.N;
  const int n_tiles = static_cast<int>((N + 255) / 256);
  const int nt0 = ng * n_cnt;
  int nt_end = nt0 + n_cnt < n_tiles ? nt0 + n_cnt : n_tiles;
  // N % 64 == 0 is checked on the host; in the last tile the waves past N have no rows
  if (static_cast<int64_t>(nt_end - 1) * 256 + wr * 64 >= N) --nt_end;

  if (e < 0) {
    if ((!a.skip_nonlocal || e_oob)) {
      for (int nt = nt0; nt < nt_end; ++nt)
#pragma unroll
        for (int tb = 0; tb < 4; ++tb)
          if (f[tb] < a.num_valid)
#pragma unroll
            for (int rb = 0; rb < 4; ++rb)
              *reinterpret_cast<v2i *>(a.C + f[tb] * N + static_cast<int64_t>(nt) * 256 + wr * 64 + rb * 16 + 4 * q) =
                  v2i{0, 0};
    }
    return;
  }

  // Their routed weights as well, asked for here: fetched by each tile's stores, a weight waited, operations retiring in order,
  // for the rows stored and the fragments requested before it.
  float wgt[4];
#pragma unroll
  for (int tb = 0; tb < 4; ++tb) {
    wgt[tb] = 1.0f;
    if (a.mul_routed) wgt[tb] = a.topk_w[f[tb] < a.num_valid ? f[tb] : 0];
  }

  // KBT: where the lane's two pieces of a token fragment's rows go, in bytes of the output, or past its end
  const brsrc rC = make_rsrc(a.C, static_cast<uint32_t>(a.num_valid * N * 2));
  uint32_t coff[4][2];
  if constexpr (KBT > 0) {
#pragma unroll
    for (int tb = 0; tb < 4; ++tb)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int fs = __shfl(f[tb] < a.num_valid ? f[tb] : -1, (lane >> 3) + 8 * j);
        coff[tb][j] = fs >= 0 ? fs * static_cast<uint32_t>(N) * 2 + (lane & 7) * 16 : kAsMaxOut;
      }
  }

  const brsrc rW = make_rsrc(a.W + static_cast<int64_t>(e) * N * K, static_cast<uint32_t>(N * K));
  // The wave's 64 rows are four 2 KB blocks, in lane order; tile, K block and k-half go into the scalar offset.
  const int wkstride = shuf_kb_stride(static_cast<int>(N / 16));
  const int wtstride = 16 * shuf_nb_stride(KB); // 256 rows further
  const int woff = (nt0 * 16 + wr * 4) * shuf_nb_stride(KB) + lane * 16;

  // ---- the token block and every scale the workgroup needs, once ----------------------
  {
    const brsrc rA = make_rsrc(a.A, static_cast<uint32_t>(a.a_rows * K));
    const int aoff = token_row(a, f_row) * K + q * 16;
    int8_t *const dst = sA + wr * 1024;
#pragma unroll
    for (int p = 0; p < (KBT ? 2 * KBT : K / 64); ++p)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rA, dst + p * 4096, 16, aoff, p * 64, 0, 0);
  }
  const int NB = static_cast<int>((N + kGroup - 1) / kGroup);
  const int b_cnt = (n_cnt * 2 < NB - nt0 * 2 ? n_cnt * 2 : NB - nt0 * 2) * KB; // [tile][half][K block]
  const brsrc rAs = make_rsrc(a.As, static_cast<uint32_t>(a.a_rows * KB * 4));
  const brsrc rWs = make_rsrc(a.Ws + (static_cast<int64_t>(e) * NB + nt0 * 2) * KB, static_cast<uint32_t>(b_cnt > 0 ? b_cnt * 4 : 0));
  // (a padding token's is zero: row 0, which it is computed on, may be one that nobody wrote)
  const int asoff = f_lane < a.num_valid ? token_row(a, f_lane) * KB * 4 : 0x40000000;
  float as_mine[2]; // of token `lane`, K blocks wr and wr + 4: K <= 1024 (gemm_as_supports)
#pragma unroll
  for (int i = 0; i < 2; ++i) as_mine[i] = bld_f32(rAs, asoff, (wr + 4 * i < KB ? wr + 4 * i : KB - 1) * 4);
  const float ws_mine = bld_f32(rWs, tid * 4, 0);
  // `fit`: for the biased fold, noting one that it does not take
  auto fill_scales = [&](auto FIT) __attribute__((always_inline)) {
    constexpr bool fit = decltype(FIT)::value;
    bool bad = false;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int kb = wr + 4 * i;
      const float v = as_mine[i];
      bad |= !fold_token_scale_ok(v);
      if (kb < KB) sS[kb * kTileM + lane] = fit ? fold_token_scale(v) : v;
    }
    for (int i = tid; i < b_cnt; i += 256) {
      const float v = i < 256 ? ws_mine : bld_f32(rWs, i * 4, 0);
      bad |= !fold_weight_scale_ok(v);
      sB[i] = fit ? fold_weight_scale(v) : v;
    }
    if constexpr (fit) sFlag[wr] = __builtin_amdgcn_ballot_w64(bad) ? 1 : 0; // one value for the wave
  };

  using B0 = std::integral_constant<int, 0>;
  using B1 = std::integral_constant<int, 1>;
  using B2 = std::integral_constant<int, 2>;
  float acc[4][4][4]; // [token fragment][row fragment][element]
  // Ring of three weight buffers: a K block is short work (32 MFMAs per wave), an L2 round trip
  // under load is not, so fragments are requested two K blocks ahead.
  v4i wreg[3][4][2];   // [buffer][row fragment][k-half]

  auto load_w = [&](auto BUF, int nt, int kb) __attribute__((always_inline)) {
    constexpr int b = decltype(BUF)::value;
    const int so = (nt - nt0) * wtstride + kb * wkstride;
#pragma unroll
    for (int rb = 0; rb < 4; ++rb)
#pragma unroll
      for (int kh = 0; kh < 2; ++kh) wreg[b][rb][kh] = bld16(rW, woff, so + rb * shuf_nb_stride(KB) + kh * 1024);
  };
  auto fold = [&](auto BIASED, const v4i &d, float as, float as_bias, float bs, float *dst) __attribute__((always_inline)) {
    const float sc = ORD == kOrdFusedScale ? as * bs : 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if constexpr (decltype(BIASED)::value) dst[i] = fold_biased(d[i], as, as_bias, bs, dst[i]);
      else dst[i] = fold_elem<ORD>(d[i], sc, as, bs, dst[i]);
    // The accumulators must be final here: an empty asm that "modifies" them stops the
    // optimiser from postponing the fold (and keeping the int32 fragment alive instead).
#pragma unroll
    for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(dst[i]));
  };
  auto compute = [&](auto BIASED, auto BUF, int nt, int kb, bool live) __attribute__((always_inline)) {
    constexpr int b = decltype(BUF)::value;
    constexpr int c0 = decltype(BIASED)::value ? kFoldBias : 0;
    const v4i cinit = {c0, c0, c0, c0};
    // the wave's 64 rows lie in one 128-row block
    const float bs = sB[live ? ((nt - nt0) * 2 + (wr >> 1)) * KB + kb : 0];
    // Software pipeline over half token fragments: the MFMAs of two row fragments are issued, then the previous two are folded
    // into the fp32 accumulators while the matrix pipe works; the next token fragment is read under the first half.
    const int8_t *src = sA + kb * 8192 + lane * 16;
    const float *ts = sS + kb * kTileM + r;
    v4i bf[2][2], dprev[2];
    float as_t[2], as_prev = 0.0f, as_bias = 0.0f;
#pragma unroll
    for (int kh = 0; kh < 2; ++kh) bf[0][kh] = *reinterpret_cast<const v4i *>(src + kh * 4096);
    as_t[0] = live ? ts[0] : 0.0f; // a step past the end adds 0
    auto fold_pair = [&](int st) __attribute__((always_inline)) {
      const int tb = st >> 1, h = st & 1;
      if (h == 0) as_bias = fold_bias(as_prev);
      fold(BIASED, dprev[0], as_prev, as_bias, bs, acc[tb][2 * h]);
      fold(BIASED, dprev[1], as_prev, as_bias, bs, acc[tb][2 * h + 1]);
    };
#pragma unroll
    for (int st = 0; st < 8; ++st) {
      const int tb = st >> 1, h = st & 1;
      if (h == 0 && tb < 3) {
#pragma unroll
        for (int kh = 0; kh < 2; ++kh)
          bf[(tb + 1) & 1][kh] = *reinterpret_cast<const v4i *>(src + (tb + 1) * 1024 + kh * 4096);
        as_t[(tb + 1) & 1] = live ? ts[(tb + 1) * 16] : 0.0f;
      }
      v4i d[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) d[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wreg[b][2 * h + j][0], bf[tb & 1][0], cinit, 0, 0, 0);
#pragma unroll
      for (int j = 0; j < 2; ++j) d[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wreg[b][2 * h + j][1], bf[tb & 1][1], d[j], 0, 0, 0);
      if (st > 0) fold_pair(st - 1);
      __builtin_amdgcn_sched_barrier(0);
      dprev[0] = d[0];
      dprev[1] = d[1];
      as_prev = as_t[tb & 1];
    }
    fold_pair(7);
    __builtin_amdgcn_sched_barrier(0);
  };

  // The (tile, K block) pairs form one flat sequence of steps; step s uses buffer s % 3.
  // Positions in that sequence are kept as (tile, K block) counters: a division by KB per step
  // is a long scalar dependency chain in front of the loads.
  const int total = (nt_end - nt0) * KB;
  int l_nt = nt0, l_kb = 0; // the next step to load
  int c_nt = nt0, c_kb = 0; // the next step to compute
  auto load_step = [&](auto BUF) __attribute__((always_inline)) { // a step past the end re-reads the last one
    const bool past = l_nt >= nt_end;
    load_w(BUF, past ? nt_end - 1 : l_nt, past ? KB - 1 : l_kb);
    if (++l_kb == KB) {
      l_kb = 0;
      ++l_nt;
    }
  };
  auto zero_acc = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int tb = 0; tb < 4; ++tb)
#pragma unroll
      for (int rb = 0; rb < 4; ++rb)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[tb][rb][i] = 0.0f;
  };
  auto store_tile = [&](int nt) __attribute__((always_inline)) {
    const int nrow0 = nt * 256 + wr * 64;
    int8_t *stg = sStage + wr * (16 * kStgPitch);
#pragma unroll
    for (int tb = 0; tb < 4; ++tb) {
      with_out16(a.out_f16, [&](auto cvt) __attribute__((always_inline)) {
#pragma unroll
        for (int rb = 0; rb < 4; ++rb) {
          v4u16 o;
#pragma unroll
          for (int i = 0; i < 4; ++i) o[i] = cvt(acc[tb][rb][i] * wgt[tb]); // 1 leaves every value as it is
          *reinterpret_cast<v4u16 *>(stg + r * kStgPitch + (rb * 16 + 4 * q) * 2) = o;
        }
      });
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int j = 0; j < 2; ++j) { // 128-byte row segments, eight rows an instruction
        const int tok = (lane >> 3) + 8 * j;
        const v4i v = *reinterpret_cast<const v4i *>(stg + tok * kStgPitch + (lane & 7) * 16);
        if constexpr (KBT > 0) {
          bst16(rC, v, coff[tb][j], nrow0 * 2);
        } else {
          const int fs = __shfl(f[tb] < a.num_valid ? f[tb] : -1, tok);
          if (fs >= 0) *reinterpret_cast<v4i *>(a.C + static_cast<int64_t>(fs) * N + nrow0 + (lane & 7) * 8) = v;
        }
      }
      __builtin_amdgcn_wave_barrier();
    }
  };
  auto step = [&](auto BIASED, auto BUF, auto NEXT) __attribute__((always_inline)) {
    load_step(NEXT);
    __builtin_amdgcn_sched_barrier(0); // keep the prefetch ahead of the MFMAs
    const bool live = c_nt < nt_end;
    compute(BIASED, BUF, c_nt, c_kb, live);
    if (live && c_kb == KB - 1) { // a tile is complete
      store_tile(c_nt);
      zero_acc();
    }
    if (++c_kb == KB) {
      c_kb = 0;
      ++c_nt;
    }
  };

  if (total > 0) { // before the barrier: in flight while the tokens land
    load_step(B0{});
    load_step(B1{});
  }
  fill_scales(std::integral_constant<bool, kBiased>{});
  __builtin_amdgcn_s_waitcnt(0x0f70); // vmcnt(0): the copies into LDS have landed
  __syncthreads(); // the only barrier: the token block is complete
  zero_acc();
  constexpr std::integral_constant<bool, kBiased> biased{};
  if constexpr (kBiased) {
    const v4i met = *reinterpret_cast<const v4i *>(sFlag);
    if (__builtin_expect(__builtin_amdgcn_readfirstlane(met[0] | met[1] | met[2] | met[3]) != 0, 0)) {
      __syncthreads();
      fill_scales(std::false_type{});
      __syncthreads();
#pragma unroll 1
      for (int nt = nt0; nt < nt_end; ++nt) { // rare: one K block at a time
#pragma unroll 1
        for (int kb = 0; kb < KB; ++kb) {
          load_w(B0{}, nt, kb);
          compute(std::false_type{}, B0{}, nt, kb, true);
        }
        store_tile(nt);
        zero_acc();
      }
      return;
    }
  }
  if constexpr (KBT > 0) {
    static_assert(KBT % 3 == 0, "a tile must start on ring buffer 0");
    for (int nt = nt0; nt < nt_end; ++nt) {
#pragma unroll
      for (int kb = 0; kb < KBT; ++kb) {
        // the step two ahead: this tile's, or the next tile's first two (the last tile re-reads its end)
        const bool wrap = kb + 2 >= KBT;
        const bool past = wrap && nt + 1 >= nt_end;
        const int lnt = past ? nt : (wrap ? nt + 1 : nt), lkb = past ? KBT - 1 : (wrap ? kb + 2 - KBT : kb + 2);
        if (kb % 3 == 0) load_w(B2{}, lnt, lkb);
        else if (kb % 3 == 1) load_w(B0{}, lnt, lkb);
        else load_w(B1{}, lnt, lkb);
        __builtin_amdgcn_sched_barrier(0); // keep the prefetch ahead of the MFMAs
        if (kb % 3 == 0) compute(biased, B0{}, nt, kb, true);
        else if (kb % 3 == 1) compute(biased, B1{}, nt, kb, true);
        else compute(biased, B2{}, nt, kb, true);
      }
      store_tile(nt);
      zero_acc();
    }
  } else {
    for (int s = 0; s < total; s += 3) {
      step(biased, B0{}, B2{});
      step(biased, B1{}, B0{});
      step(biased, B2{}, B1{});
    }
  }
}

// weight tiles of a workgroup
static int as_tiles(int64_t N) {
  const int n_tiles = static_cast<int>((N + 255) / 256);
  return (n_tiles + 1) / 2;
}
static int64_t as_lds_bytes(int64_t N, int64_t K) {
  return 64 * K + (K / kGroup) * 64 * 4 + 4 * 16 * kStgPitch + as_tiles(N) * 2 * (K / kGroup) * 4 + 16;
}

bool gemm_as_supports(const GemmArgs &a, bool fused_act, int block_size_m) {
  if (fused_act || !a.w_shuffled || (block_size_m != 64 && block_size_m != 128)) return false;
  if (a.N % 64 != 0 || (reinterpret_cast<uintptr_t>(a.C) & 15) != 0) return false;
  if (a.K > 8 * kGroup || as_lds_bytes(a.N, a.K) > 80 * 1024) return false; // two workgroups per CU
  // Pays off only when the launch is several rounds of workgroups deep even with half a
  // token block's weight tiles per workgroup; below that the per-tile kernel balances better.
  return a.num_valid / 64 + (a.experts_routed + 1) / 2 >= 1024;
}

int launch_gemm_as(const GemmArgs &a0, int flags, int block_size_m, int64_t m_blocks_bs, hipStream_t s) {
  const int sub_shift = block_size_m == 128 ? 1 : 0;
  const int64_t m_blocks = m_blocks_bs << sub_shift; // in 64-token pieces
  GemmArgs a = a0;
  const int n_tiles = static_cast<int>((a.N + 255) / 256);
  // Weight tiles per workgroup: half of them.  Fewer workgroups than that leave the
  // launch unbalanced, more pay the token gather more often (measured on 128 experts,
  // N = 2048, K = 768: 250 us with two groups, 269 with one, 296 with eight at 8192 tokens).
  const int n_cnt = as_tiles(a.N);
  const int n_groups = (n_tiles + n_cnt - 1) / n_cnt;
  a.n_tiles = n_groups;
  int64_t G = a.num_valid / (static_cast<int64_t>(a.experts_routed > 0 ? a.experts_routed : 1) * 64);
  G = G < 2 ? 2 : (G > 16 ? 16 : G);
  const int64_t chunks = (m_blocks + G - 1) / G;
  const int64_t grid = (chunks + 7) / 8 * (G * n_groups) * 8;
  LO_REQUIRE(grid < (1ll << 31), LO_EINVAL, "moe_gemm: grid too large");
  const int ord = scale_order(flags);
  const size_t lds = static_cast<size_t>(as_lds_bytes(a.N, a.K));
  const dim3 g(static_cast<unsigned>(grid)), b(256);
  const int mbi = static_cast<int>(m_blocks), Gi = static_cast<int>(G);
#define LO_AS_LAUNCH(FS, KBT)                                                                         \
  do {                                                                                                \
    auto kern = moe_gemm_as_kernel<FS, KBT>;                                                          \
    static unsigned long long lds_done = 0; /* per instantiation: one bit per device */               \
    const int rc_lds = reserve_lds_once(reinterpret_cast<const void *>(kern), 80 * 1024, &lds_done);  \
    if (rc_lds) return rc_lds;                                                                        \
    hipLaunchKernelGGL(kern, g, b, lds, s, a, mbi, Gi, n_groups, n_cnt, sub_shift);                   \
  } while (0)
  if (a.K == 6 * kGroup && a.num_valid * a.N * 2 <= kAsMaxOut) LO_ORD_DISPATCH(ord, LO_AS_LAUNCH, 6);
  else LO_ORD_DISPATCH(ord, LO_AS_LAUNCH, 0);
#undef LO_AS_LAUNCH
  return check_launch("moe_gemm(activation-stationary)");
}

} // namespace lo
