// Grouped block-INT8 GEMM for gfx950, 128-token form with two independent workgroups per
// compute unit.
//
// The LDS-tiled kernels are bound by the rate at which compute units pull operands out of L2:
// bytes requested per multiply-add are 1/tokens + 1/rows of the workgroup tile.  A 128-token
// tile needs 128 fp32 accumulators per lane when four waves share 256 weight rows, which leaves
// no room for weight fragments double-buffered in registers (gemm_tile.hip) at two waves per
// SIMD, and a single eight-wave workgroup per compute unit (gemm_dma.hip) runs phase-locked.
// Here every operand byte enters the compute unit once by direct global -> LDS loads
// (buffer_load ... lds) and costs no staging registers, so four waves hold 128 tokens x 256
// rows in 72 KB of LDS and two such workgroups share a compute unit:
//   weights  each wave copies its own rows: per 128-wide K block four pre-shuffled 2 KB blocks
//            into a private 8 KB stage.  The wave reads the stage into registers at the start of
//            a K block and refills it at once with the next K block, so the stage needs no
//            barrier and no second copy, and is requested a whole K block ahead;
//   tokens   128 rows x 128 bytes per K block into a two-stage ring shared by the workgroup
//            (16-byte pieces XOR-swizzled by row, conflict-free operand reads), requested one K
//            block ahead; one barrier per K block.  Every wave reads each token fragment once per
//            K block and uses it against all 64 of its rows: LDS bandwidth is what this kernel
//            runs out of first;
//   scales   the tokens' group scales, through registers, one K block ahead; the weight-block
//            scales of the tile's rows (two per K block) go to LDS once, before the K loop, so
//            that the loop issues no vector-memory operation whose result it has to wait for
//            (the wait would also drain the copies in flight).
// A wave owns 64 rows x 128 tokens as 4 x 8 fragments of v_mfma_i32_16x16x64_i8 (weights as
// the A operand) and folds each fragment's exact int32 sum over a K block into fp32 as the
// 64-token kernel does (reference arithmetic: Triton fused_moe_kernel,
// python/lightop/_lmslim_native/layers/fused_moe/int8.py:485-519; fused epilogue :811-823).
#include <type_traits>

#include "gemm.h"

namespace lo {

constexpr int kT = 128;                       // tokens per workgroup
constexpr int kTWStage = 8192;                // one wave's weights for one K block
constexpr int kTW = 4 * kTWStage;             // [wave]
constexpr int kTAStage = kT * kGroup;         // token rows of one K block
constexpr int kTA = 2 * kTAStage;
constexpr int kTS = 2 * kT * 4;               // [stage][token] scales
constexpr int kTRed = 4 * kT * 4;             // [wave][token] amax exchange of the fused epilogue
constexpr int kTMaxKB = 128;                  // K blocks whose weight-block scales fit the table below
constexpr int kTBs = 2 * kTMaxKB * 4;         // [fragment][K block] weight-block scales of the tile
constexpr int kTIds = kT * 4;                  // the tile's sorted ids, for the epilogues
constexpr int kTFlag = 16;                    // [wave]: it met a scale that the biased fold does not take
constexpr int kTWgt = kT * 4;                  // routed weights of the tile's slots
constexpr int kTLds = kTW + kTA + kTS + kTRed + kTBs + kTIds + kTWgt + kTFlag;
// NTB = 10: 160 tokens per workgroup, for layers whose experts see a few tokens more than 128: a remainder block is a second
// pass over the expert's weights, and at that size the weights are what the stage streams.
constexpr int kT160 = 160;
constexpr int kTLds160 = kTW + 2 * kT160 * kGroup + 2 * kT160 * 4 + 4 * kT160 * 4 + kTBs + 2 * kT160 * 4 + kTFlag;
constexpr int kTPitch = 144;                  // staging pitch of the epilogues: 128 + 16

// Wait until all but the newest `N` vector-memory operations of this wave are complete and its
// LDS operations have landed.  (__syncthreads() would drain every copy in flight: the compiler
// treats a direct-to-LDS load as an LDS write that a workgroup fence must make visible.)
template <int N>
__device__ __forceinline__ void wait_copies() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
}
// 16 or 4 bytes a lane to LDS; once: with the streaming hint (a constant at each call)
__device__ __forceinline__ void copy_weights(brsrc r, int8_t *lds, int voff, int soff, bool once) {
  if (once) __builtin_amdgcn_raw_ptr_buffer_load_lds(r, lds, 16, voff, soff, 0, kCacheStream);
  else __builtin_amdgcn_raw_ptr_buffer_load_lds(r, lds, 16, voff, soff, 0, kCacheDefault);
}
__device__ __forceinline__ void copy_row_scales(brsrc r, int8_t *lds, int voff, int soff, bool once) {
  if (once) __builtin_amdgcn_raw_ptr_buffer_load_lds(r, lds, 4, voff, soff, 0, kCacheStream);
  else __builtin_amdgcn_raw_ptr_buffer_load_lds(r, lds, 4, voff, soff, 0, kCacheDefault);
}
template <int N>
__device__ __forceinline__ void wait_copies_barrier() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

//
// PC (with W4): the reference's own int4 form (fused_moe_kernel_int4_w4a8,
// python/lightop/_lmslim_native/layers/fused_moe/w4a8.py:341-395): one scale per token row and one
// per weight row, both applied in the epilogue, so the int32 sums run over the whole K inside the
// MFMA accumulators and the K loop has no scale arithmetic at all.
template <int FUSED_ACT, int ORD, bool STREAM, bool W4, bool PC = false, int NTB = 8, bool ROWS = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(NTB == 1 ? 4 : NTB <= 4 ? 3 : 2, NTB == 1 ? 4 : NTB <= 4 ? 3 : 2)))
void moe_gemm_t128_kernel(const GemmArgs a, int m_blocks, int group_m) {
  static_assert(!PC || (ORD == kOrdSeparate && (W4 || NTB == 10 || ROWS)),
                "per-channel scales: int4 weights, 160-token tiles of int8 weights or row-major ones");
  static_assert(NTB == 8 || NTB == 10 || ((NTB == 1 || NTB == 2 || NTB == 4) && ROWS),
                "16, 32 and 64 tokens: row-major weights");
  static_assert(!ROWS || (!W4 && NTB <= 8), "row-major weights: int8, up to 128 tokens");
  constexpr int T = 16 * NTB;        // tokens per workgroup
  constexpr int AST = T * kGroup;    // token rows of one K block
  constexpr int APW = NTB == 1 ? 1 : NTB / 2;       // 1 KB pieces (eight token rows) of a token stage that a wave copies
  constexpr int RED = 4 * T * 4;
  extern __shared__ __attribute__((aligned(16))) int8_t smem[];
  int8_t *const sA = smem + kTW;
  float *const sS = reinterpret_cast<float *>(smem + kTW + 2 * AST);
  float *const sRed = reinterpret_cast<float *>(smem + kTW + 2 * AST + 2 * T * 4); // [wave][token] amax of its 32 columns
  float *const sBs = reinterpret_cast<float *>(smem + kTW + 2 * AST + 2 * T * 4 + RED);
  int32_t *const sIds = reinterpret_cast<int32_t *>(smem + kTW + 2 * AST + 2 * T * 4 + RED + kTBs);

  float *const sWgt = reinterpret_cast<float *>(sIds + T);
  int32_t *const sFlag = sIds + 2 * T;
  // The contracted order folds without a conversion (fold_biased): 2 vector instructions an element and K block instead of 3,
  // where they were issued in 83 % of a SIMD's cycles.  Layer with its router, us, before / after: full DeepSeek-V3 layer, 8192
  // tokens 4828 / 4531, Qwen3-30B-A3B layer, 8192: 603.8 / 578.9, DeepSeek-V3 share, 4096: 539 / 525, int4 with K-group scales,
  // 2048: 629 / 594.  A tile that meets a scale outside of its range is done again with the conversion.
  constexpr bool kBiased = ORD == kOrdContract && !PC;
  // 160 tokens of int4 weights with K-group scales: 160 accumulators, unpacked weights and their row scales are more registers
  // than there are.  The wave takes its 64 rows in two halves, one after the other, with every token fragment: half of the
  // unpacked weights and, but for one stage, of the row scales at a time, and each token fragment read from LDS twice.  The
  // second half is read from LDS in mid K block, so the weights have two stages, in the room that 8-bit ones take; the row
  // scales' are in the amax exchange of the epilogue.  Qwen3-235B-A22B-shaped layer, 2048 tokens: 592 us in 128-token blocks, 516.
  constexpr bool kHalves = W4 && !PC && NTB == 10;
  // So the waves have to meet between the K loop and that epilogue: until then a slower one reads its row scales, and copies of
  // scales past the last K block land.  (The default order meets before it looks at the flags.)
  constexpr bool kMeet = kHalves && FUSED_ACT;

  int mb, nt;
  // (int8: every argument that the start needs asked for in one go, Qwen3-30B-A3B layer at 1000 tokens 159.2 -> 158.2 us, 1531: 171.6 ->
  // 171.2, DeepSeek-V3 share at 700 252.9 -> 252.5; int4 with K-group scales 529 / 531)
  const int E = W4 ? a.E : start_args(a);
  if (!tile_of(blockIdx.x, a.n_tiles, m_blocks, group_m, mb, nt)) return;
  int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6); // which 64 weight rows of the tile
  int r = lane & 15, q = lane >> 4;
  // Lane indexes derived afresh, so that nothing computed from them is kept through the K loop.
  auto derive = [&]() __attribute__((always_inline)) {
    if constexpr (kHalves) {
      asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(lane));
      tid = wave * 64 + lane;
    } else {
      asm volatile("" : "+v"(tid));
      lane = tid & 63;
    }
    r = lane & 15;
    q = lane >> 4;
  };
  const int32_t *const sorted = a.sorted + static_cast<int64_t>(mb) * T;
  // Everything the tile's start-up reads from memory by its block index alone is requested here, in one go:
  // the number of blocks in use, the block's expert and the sorted ids this thread needs (token rows it
  // copies, the last valid token, the token whose scales it carries).  Asked for one after the other, each
  // behind the branch on the one before, they were three round trips in front of the first operand copy.
  // (Not for the fused 160-token form: the values alive across the branches cost it registers it does not have.)
  constexpr bool kEarlyIds = !(FUSED_ACT && NTB == 10);
  const int32_t blocks_end = a.ntpp[0];
  const int e_raw = a.expert_ids[mb];
  // whether no other token block reads this one's weights (copy policy, below)
  constexpr bool kPolicy = !W4 && !ROWS && NTB == 8;
  const bool alone = kPolicy && (mb == 0 || a.expert_ids[mb - 1] != e_raw) &&
                     (mb + 1 >= m_blocks || a.expert_ids[mb + 1] != e_raw);
  const int cw = NTB == 1 ? wave & 1 : wave; // 16 tokens are two pieces: the first two waves copy them
  int32_t lf_copy[APW];
  int32_t lf_v0 = 0, lf_v1 = 0, lf_v2 = 0, lf_scale = 0;
  auto load_ids = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < APW; ++j) lf_copy[j] = sorted[(cw * APW + j) * 8 + (lane >> 3)];
    lf_v0 = sorted[lane & (T - 1 < 63 ? T - 1 : 63)];
    if constexpr (NTB >= 8) lf_v1 = sorted[lane + 64];
    if constexpr (NTB == 10) lf_v2 = sorted[128 + (lane & 31)];
    lf_scale = sorted[NTB <= 8 ? (tid & (T - 1)) : (tid < T ? tid : tid - T)];
  };
  if constexpr (kEarlyIds) load_ids();
  if (static_cast<int64_t>(mb) * T >= blocks_end) return;
  // An expert_map entry outside the weight tensor is treated like an expert of another rank, but its
  // rows are always zero-filled: the slot mask of the alignment counts such a slot as local.
  const bool e_oob = e_raw >= E;
  const int e = e_oob ? -1 : e_raw;
  const int64_t K = a.K, N = a.N;
  const int KB = static_cast<int>(K / kGroup);
  const int64_t I = N / 2;

  // first row of the wave's 64 (plain) or of its 32 gate rows (fused)
  const int64_t nrow0 = FUSED_ACT ? static_cast<int64_t>(nt) * kGroup + wave * 32
                                  : static_cast<int64_t>(nt) * 256 + wave * 64;
  const bool wave_active = FUSED_ACT || nrow0 < N; // N % 64 == 0 is checked on the host

  if (e < 0) {
    if constexpr (!FUSED_ACT) {
      if (wave_active && (!a.skip_nonlocal || e_oob)) {
        if constexpr (kHalves) derive(); // (the compiler moves this branch to the end)
#pragma unroll
        for (int tb = 0; tb < NTB; ++tb) {
          const int64_t ft = sorted[tb * 16 + r];
          if (ft < a.num_valid)
#pragma unroll
            for (int j = 0; j < 4; ++j)
              *reinterpret_cast<v2i *>(a.C + ft * N + nrow0 + j * 16 + 4 * q) = v2i{0, 0};
        }
      }
    }
    return;
  }

  // ---- what this wave copies -----------------------------------------------------------------------
  const int NBLK = static_cast<int>(N / 16);
  // W4: packed int4 weights in their load-time layout (1 KB per 16 rows x 128 K, the lane's two
  // k-steps in one 16-byte piece) and one scale per weight row and K block, [E, K/128, N]
  const int64_t wbytes = W4 ? N * K / 2 : N * K; // one expert
  const brsrc rW = make_rsrc(a.W + static_cast<int64_t>(e) * wbytes, static_cast<uint32_t>(wbytes));
  const brsrc rWs = make_rsrc(a.Ws + static_cast<int64_t>(e) * N * (PC ? 1 : KB), static_cast<uint32_t>(N * (PC ? 1 : KB) * 4));
  const brsrc rA = make_rsrc(a.A, static_cast<uint32_t>(a.a_rows * K));
  const brsrc rAs = make_rsrc(a.As, static_cast<uint32_t>(a.a_rows * (PC ? 1 : KB) * 4));
  const int wkstride = ROWS ? kGroup : W4 ? shuf_kb_stride(NBLK) / 2 : shuf_kb_stride(NBLK);
  const int wpstride = ROWS ? static_cast<int>(8 * K) : 1024; // second half of a 16-row block
  int wsoff[2][2]; // [step half][fragment]: the 2 KB block of 16 rows x 128 K (wave-uniform)
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int rf = 0; rf < 2; ++rf) {
      int64_t nb;
      if constexpr (FUSED_ACT) nb = (rf ? I / 16 : 0) + static_cast<int64_t>(nt) * 8 + wave * 2 + h;
      else nb = static_cast<int64_t>(nt) * 16 + wave * 4 + h * 2 + rf;
      if (nb >= NBLK) nb = 0; // rows past N: computed on block 0, never stored
      if constexpr (ROWS) wsoff[h][rf] = static_cast<int>(nb * 16 * K);
      else wsoff[h][rf] = static_cast<int>(nb) * (W4 ? shuf_nb_stride(KB) / 2 : shuf_nb_stride(KB));
    }
  // the lane's part of it: in lane order, or, row-major, a 1 KB piece is 128 bytes of eight rows, whole lines; slot lane & 7
  // of row lane >> 3 takes the row's 16-byte piece slot ^ row (as in the token stage)
  const int wvoff = ROWS ? static_cast<int>((lane >> 3) * K) + (((lane & 7) ^ (lane >> 3)) * 16) : lane * 16;
  // W4: lane l copies the scale of row l of the wave's 64 (fused: 32 gate rows, then the 32 up rows)
  int wsvoff = 0;
  if constexpr (W4) {
    int64_t row;
    if constexpr (FUSED_ACT) row = (lane < 32 ? 0 : I - 32) + static_cast<int64_t>(nt) * kGroup + wave * 32 + lane;
    else row = static_cast<int64_t>(nt) * 256 + wave * 64 + lane;
    if (row >= N) row = 0;
    wsvoff = static_cast<int>(row * 4);
  }
  // Copy policy of the weights.  A byte that one workgroup uses is requested with the streaming hint (it does not displace the
  // token rows and scales in L2) while experts have half a block on average, and past that by blocks of at most 64 tokens;
  // blocks of one expert share its weights through L2.  128-token int8 blocks look at their neighbours: by the layer's average
  // alone (STREAM: the other forms go by it, see the launches) skewed routing loses.
  constexpr std::integral_constant<bool, true> once{};
  constexpr std::integral_constant<bool, STREAM> by_launch{};
  // The first K block's weights depend on the expert only: they are requested before the token
  // ids are read, so that the two dependent round trips of the tile's start-up overlap.
  int8_t *const sWw = smem + wave * kTWStage; // int8: [row half][fragment][k half] x 1 KB; W4: [row half][fragment] x 1 KB, row scales
  // W4: the scales of the wave's 64 rows beside the weights of K block kb
  auto row_scales = [&](int kb) __attribute__((always_inline)) {
    return kHalves ? reinterpret_cast<int8_t *>(sRed) + ((kb & 1) * 4 + wave) * 256 : sWw + 4096;
  };
  auto copy_w0 = [&](bool once) __attribute__((always_inline)) {
    if constexpr (W4) {
#pragma unroll
      for (int p = 0; p < 4; ++p)
        copy_weights(rW, sWw + p * 1024, wvoff, wsoff[p >> 1][p & 1], once);
      if constexpr (!PC) copy_row_scales(rWs, row_scales(0), wsvoff, 0, once);
    } else {
#pragma unroll
      for (int p = 0; p < 8; ++p)
        copy_weights(rW, sWw + p * 1024, wvoff, wsoff[p >> 2][(p >> 1) & 1] + (p & 1) * wpstride, once);
    }
  };
  // (a block's tokens are not known yet: by the layer's average)
  if (kPolicy && a.stream) copy_w0(true);
  else copy_w0(STREAM);
  int avoff[5]; // 1 KB pieces wave*APW + j of a token stage, j < APW: eight token rows each
#pragma unroll
  for (int j = 0; j < APW; ++j) {
    const int t = (cw * APW + j) * 8 + (lane >> 3);
    const int64_t lf = kEarlyIds ? lf_copy[j] : sorted[t];
    const int piece = (lane & 7) ^ (t & 7); // slot lane & 7 of row t holds piece slot ^ (t & 7)
    // (the move leaves one register: an offset that stays the lower half of a 64-bit multiply-add keeps two through the K loop)
    asm("v_mov_b32 %0, %1" : "=v"(avoff[j]) : "v"(token_row(a, lf) * static_cast<int>(K) + piece * 16));
  }
  // The alignment puts a block's valid tokens first, so a block of 128 is on average half a block
  // of padding per expert: token fragments past the last valid token are skipped (taken from the position of the last valid token, not from their number, so that
  // a caller's own sorted ids with gaps are still computed in full).
  int nst; // pipeline stages per K block: two per 16 tokens in use
  {
    if constexpr (!kEarlyIds) {
      lf_v0 = sorted[lane];
      lf_v1 = sorted[lane + 64];
      if constexpr (NTB == 10) lf_v2 = sorted[128 + (lane & 31)];
    }
    const uint64_t v0 = __builtin_amdgcn_ballot_w64(lf_v0 < a.num_valid);
    const uint64_t v1 = NTB >= 8 ? __builtin_amdgcn_ballot_w64(lf_v1 < a.num_valid) : 0;
    int last = v1 ? 127 - __builtin_clzll(v1) : (v0 ? 63 - __builtin_clzll(v0) : 0);
    if constexpr (NTB == 10) {
      const uint64_t v2 = __builtin_amdgcn_ballot_w64(lane < 32 && lf_v2 < a.num_valid);
      if (v2) last = 191 - __builtin_clzll(v2);
    }
    nst = __builtin_amdgcn_readfirstlane(2 * ((last >> 4) + 1)); // the K loop comes in variants by the number of fragments
    if (NTB == 10 && a.coarse_fill && nst > 8 && nst < 16) nst = 16;
  }
  float wgt_mine = 1.0f;
  int asoff; // thread t and thread t + T both carry the scale of token t
  {
    const int64_t lf = kEarlyIds ? lf_scale : sorted[NTB <= 8 ? (tid & (T - 1)) : (tid < T ? tid : tid - T)];
    // (A padding token's is read as zero, past the end of the scales: the row it is computed on, 0, may be one that nobody
    // wrote - a slot of another rank's expert - and what it holds must not send the tile to the long fold.)
    asoff = PC || lf < a.num_valid ? token_row(a, lf) * (PC ? 1 : KB) * 4 : 0x40000000;
    // The epilogues take the ids from LDS: a global load in each of their exec-masked blocks is a
    // full memory round trip that nothing overlaps.
    if (tid < T) sIds[tid] = static_cast<int32_t>(lf);
    // The routed weights too: fetched by the epilogue, each of them waited, operations retiring in order, for the rows stored
    // before it (int4 with K-group scales, 2048 tokens 588 -> 579 us; Qwen3-30B-A3B layer, 8192: 553 -> 549).
    if (a.mul_routed) wgt_mine = a.topk_w[lf < a.num_valid ? lf : 0];
  }
  // weight-block scales of the tile: table row 0 / 1 = gate / up block (fused), or the first / second
  // 128 rows of the tile (plain: waves 0, 1 / waves 2, 3).  Thread t fetches entry (t >> 7, t & 127).
  const int NB = static_cast<int>((N + kGroup - 1) / kGroup);
  auto load_bs = [&]() __attribute__((always_inline)) {
    const int which = tid >> 7, kbi = tid & (kTMaxKB - 1);
    int64_t nblk = FUSED_ACT ? (which ? I / kGroup : 0) + nt : static_cast<int64_t>(nt) * 2 + which;
    if (nblk >= NB) nblk = 0;
    return !W4 && !PC && kbi < KB ? a.Ws[(static_cast<int64_t>(e) * NB + nblk) * KB + kbi] : 0.0f;
  };
  float bs_mine = load_bs();
  const float *const sBs0 = sBs + (FUSED_ACT ? 0 : (wave >> 1) * kTMaxKB);
  const float *const sBs1 = sBs + (FUSED_ACT ? kTMaxKB : (wave >> 1) * kTMaxKB);

  // piece p of the 8 + APW copies a wave issues per K block: 0..7 its weights, then its token rows
  auto copy_piece = [&](bool once, int p, int kb) __attribute__((always_inline)) {
    const int kc = kb < KB ? kb : KB - 1;
    if (p < 8) {
      if constexpr (W4) { // four weight pieces, the row scales, three empty slots
        if (p < 4)
          copy_weights(rW, sWw + (kHalves ? (kb & 1) * 4096 : 0) + p * 1024, wvoff,
                       __builtin_amdgcn_readfirstlane(kc * wkstride) + wsoff[p >> 1][p & 1], once);
        else if (p == 4 && !PC)
          copy_row_scales(rWs, row_scales(kb), wsvoff, __builtin_amdgcn_readfirstlane(kc) * static_cast<int>(N) * 4, once);
      } else {
        const int h = p >> 2, rf = (p >> 1) & 1, kh = p & 1;
        copy_weights(rW, sWw + p * 1024, wvoff, __builtin_amdgcn_readfirstlane(kc * wkstride) + wsoff[h][rf] + kh * wpstride,
                     once);
      }
    } else if (p - 8 < APW && (NTB > 1 || wave < 2)) {
      const int j = p - 8;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rA, sA + (kb & 1) * AST + (cw * APW + j) * 1024, 16, avoff[j],
                                               __builtin_amdgcn_readfirstlane(kc) * kGroup, 0, 0);
    }
  };
  auto copy_a = [&](int kb) __attribute__((always_inline)) {
#pragma unroll
    for (int p = 8; p < 8 + APW; ++p) copy_piece(STREAM, p, kb);
  };
  auto load_scale = [&](int kb) __attribute__((always_inline)) {
    if constexpr (PC) return 0.0f; // one scale per token, read by the epilogue
    return bld_f32(rAs, asoff, (kb < KB ? kb : KB - 1) * 4);
  };

  // ---- operand read offsets -------------------------------------------------------------------------
  // token fragment tb, k-half kh: piece 4*kh + q of row tb*16 + r sits in slot piece ^ (r & 7)
  int alds[2];
#pragma unroll
  for (int kh = 0; kh < 2; ++kh) alds[kh] = r * kGroup + (((4 * kh + q) ^ (r & 7)) * 16);

  // weight fragment's k-half kh inside its 2 KB: lane order, or (row-major) rows of 128 bytes swizzled like the tokens
  int wlds[2];
#pragma unroll
  for (int kh = 0; kh < 2; ++kh) wlds[kh] = ROWS ? alds[kh] : kh * 1024 + lane * 16;

  float acc[2][NTB][2][4]; // [step half][token fragment][fragment of the half][element]
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int tb = 0; tb < NTB; ++tb)
#pragma unroll
      for (int rf = 0; rf < 2; ++rf)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[h][tb][rf][i] = 0.0f;
  v4i acci[2][NTB][2]; // PC: the whole-K int32 sums
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int tb = 0; tb < NTB; ++tb)
#pragma unroll
      for (int rf = 0; rf < 2; ++rf) acci[h][tb][rf] = v4i{0, 0, 0, 0};

  // W4: every product carries the factor 16 of the unpacked nibbles; it is taken out through the row
  // scale, which read_w() multiplies by 1/16 once per K block (a power of two: (f32(d) * a_s) * (b_s / 16)
  // is bit for bit (f32(d / 16) * a_s) * b_s unless b_s lies below 2^-122 or the product above 2^124).
  // One scale per weight row: bs4[i] for row 4q + i.
  auto fold4 = [&](auto BIASED, const v4i &d, float as, float as_bias, const v4f &bs4, float *dst) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 4; ++i) // bs4 already holds scale / 16
      if constexpr (decltype(BIASED)::value) dst[i] = fold_biased(d[i], as, as_bias, bs4[i], dst[i]);
      else dst[i] = fold_elem<ORD>(d[i], ORD == kOrdFusedScale ? as * bs4[i] : 0.0f, as, bs4[i], dst[i]);
#pragma unroll
    for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(dst[i])); // keep the fold here
  };
  auto fold = [&](auto BIASED, const v4i &d, float sc, float as, float as_bias, float bs, float *dst) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if constexpr (decltype(BIASED)::value) dst[i] = fold_biased(d[i], as, as_bias, bs, dst[i]);
      else dst[i] = fold_elem<ORD>(d[i], sc, as, bs, dst[i]);
#pragma unroll
    for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(dst[i])); // keep the fold here
  };

  auto uniform = [](float v) { return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v))); };
  // One K block: the wave's 64 rows (two halves h of two fragments) against all 128 tokens.
  v4i w[2][2][2]; // the wave's weights of the current K block
  v4f wsc[2][2];  // W4: the scales of the lane's rows 4q .. 4q+3 of each fragment
  float ws_max = 0.0f; // W4: largest |row scale| so far (of row `lane` of the wave's 64)
  auto unpack = [&](const v4i &pk, v4i (&to)[2]) __attribute__((always_inline)) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        const uint32_t word = static_cast<uint32_t>(pk[2 * ks + x]);
        to[ks][2 * x] = static_cast<int>((word << 4) & 0xf0f0f0f0u);
        to[ks][2 * x + 1] = static_cast<int>(word & 0xf0f0f0f0u);
      }
  };
  // scales of the lane's rows 4q .. 4q+3 of fragment (h, rf), whose rows among the wave's 64 are: fused 32*rf + 16*h, plain 32*h + 16*rf
  auto read_scales = [&](auto BIASED, int h, int rf, int kb) __attribute__((always_inline)) {
    const int row0 = (FUSED_ACT ? 32 * rf + 16 * h : 32 * h + 16 * rf) + 4 * q;
    wsc[h][rf] = *reinterpret_cast<const v4f *>(row_scales(kb) + row0 * 4) * (decltype(BIASED)::value ? fold_weight_scale(0.0625f) : 0.0625f);
  };
  // the weights of K block kb (kHalves: of its first half)
  auto read_w = [&](auto BIASED, int kb) __attribute__((always_inline)) {
    if constexpr (W4) {
      if constexpr (decltype(BIASED)::value)
        ws_max = fmaxf(ws_max, fabsf(*reinterpret_cast<const float *>(row_scales(kb) + lane * 4)));
#pragma unroll
      for (int h = 0; h < (kHalves ? 1 : 2); ++h)
#pragma unroll
        for (int rf = 0; rf < 2; ++rf) {
          unpack(*reinterpret_cast<const v4i *>(sWw + (kHalves ? (kb & 1) * 4096 : 0) + (h * 2 + rf) * 1024 + lane * 16), w[h][rf]);
          if constexpr (!PC) read_scales(BIASED, h, rf, kb);
        }
    } else {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int rf = 0; rf < 2; ++rf)
#pragma unroll
          for (int kh = 0; kh < 2; ++kh)
            w[h][rf][kh] = *reinterpret_cast<const v4i *>(sWw + (h * 2 + rf) * 2048 + wlds[kh]);
    }
  };
  // Full tiles meet at the barrier two stages before the end of a K block instead of at its start:
  // by then every copy for the next K block has had eight stages to land and nobody reads this K
  // block's token stage or scales any more, so the next block's first operands are read from LDS
  // under the last two stages and no wave stands waiting for LDS right after a barrier.
  // (From twelve stages on, that is; with ten fragments of accumulators only the full variant, the others would spill.)
  constexpr int kEarlyFrom = NTB == 10 && !PC ? 20 : 12; // (int4 weights: none)
  float s_pending;   // token scales on their way from global memory to sS
  v4i bf_first[2];   // first token fragment of the next K block
  float as_first = 0.0f;
  auto put_scale = [&](auto BIASED, int stage, float s) __attribute__((always_inline)) {
    if (tid < T) {
      if constexpr (decltype(BIASED)::value) {
        if (__builtin_amdgcn_ballot_w64(!fold_token_scale_ok(s))) sFlag[wave] = 1;
        s = fold_token_scale(s);
      }
      sS[stage * T + tid] = s;
    }
  };
  auto kblock_halves = [&](auto BIASED, auto NST, auto ONCE, int kb) __attribute__((always_inline)) {
    constexpr int nst_c = decltype(NST)::value, nf = nst_c / 2; // a stage: one token fragment, two row fragments
    constexpr int c0 = decltype(BIASED)::value ? kFoldBias : 0;
    constexpr int kCopies = 5 + APW, per = nst_c > 12 ? 1 : nst_c > 4 ? 2 : 3; // copies a stage: spread out, they stand in nobody's way
    const v4i cinit = {c0, c0, c0, c0};
    const int off0 = (kb & 1) * AST + alds[0];
    const int8_t *const ta[2] = {sA + off0, sA + (off0 ^ 64)}; // (the other k-half, computed here: a register less through the loop)
    const float *ts = sS + (kb & 1) * T;
    v4i bf[2][2], pk[2], dprev[2];
    float as_t[2], as_p = 0.0f;
#pragma unroll
    for (int kh = 0; kh < 2; ++kh) bf[0][kh] = *reinterpret_cast<const v4i *>(ta[kh]);
    as_t[0] = ts[r];
    auto fold_stage = [&](int st) __attribute__((always_inline)) {
      const int tb = st % nf, h = st / nf;
      const float as_bias = decltype(BIASED)::value ? fold_bias(as_p) : 0.0f;
      fold4(BIASED, dprev[0], as_p, as_bias, wsc[h][0], acc[h][tb][0]);
      fold4(BIASED, dprev[1], as_p, as_bias, wsc[h][1], acc[h][tb][1]);
    };
#pragma unroll
    for (int st = 0; st < nst_c; ++st) {
      const int cur = st & 1, nxt = cur ^ 1, tbn = (st + 1) % nf;
#pragma unroll
      for (int c = st * per; c < st * per + per; ++c)
        if (c < kCopies) copy_piece(decltype(ONCE)::value, c < 5 ? c : c + 3, kb + 1);
      if (st + 1 < nst_c) {
#pragma unroll
        for (int kh = 0; kh < 2; ++kh) bf[nxt][kh] = *reinterpret_cast<const v4i *>(ta[kh] + tbn * 16 * kGroup);
        as_t[nxt] = ts[tbn * 16 + r];
      }
      if (st == nf - 1) {
#pragma unroll
        for (int rf = 0; rf < 2; ++rf) {
          pk[rf] = *reinterpret_cast<const v4i *>(sWw + (kb & 1) * 4096 + (2 + rf) * 1024 + lane * 16);
          read_scales(BIASED, 1, rf, kb);
        }
      }
      if (st == nf) {
#pragma unroll
        for (int rf = 0; rf < 2; ++rf) unpack(pk[rf], w[0][rf]);
      }
      v4i d[2];
#pragma unroll
      for (int rf = 0; rf < 2; ++rf) d[rf] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w[0][rf][0], bf[cur][0], cinit, 0, 0, 0);
#pragma unroll
      for (int rf = 0; rf < 2; ++rf) d[rf] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w[0][rf][1], bf[cur][1], d[rf], 0, 0, 0);
      if (st > 0) fold_stage(st - 1);
      if (st != nf && st != nf - 1) {
        if (st + 1 < nst_c) __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          if (st * per + g < kCopies && g < per) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
          // The products close up and the folds stand behind them, as in 128-token tiles (below): four after each / this, 128 experts
          // of 4096 x 1536 at 1800 / 2048 tokens 492 / 484, 534 / 526 us.
          if (!decltype(BIASED)::value) __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);
          else if (g < 3) __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
          else __builtin_amdgcn_sched_group_barrier(0x002, 10, 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      dprev[0] = d[0];
      dprev[1] = d[1];
      as_p = as_t[cur];
    }
    fold_stage(nst_c - 1);
    __builtin_amdgcn_sched_barrier(0);
    wait_copies<0>();
    read_w(BIASED, kb + 1);
  };
  auto kblock = [&](auto BIASED, auto NST, auto ONCE, int kb) __attribute__((always_inline)) {
    if constexpr (kHalves) {
      kblock_halves(BIASED, NST, ONCE, kb);
      return;
    }
    constexpr int nst_c = decltype(NST)::value; // stages of this variant: 4, 8, 12, 16 (or 20)
    constexpr int kFull = 2 * NTB;              // stages of a full tile
    constexpr int kE0 = nst_c - 2, kE1 = nst_c - 1;
    constexpr bool kEarly = nst_c >= kEarlyFrom && !W4 && NTB >= 8;
    const int8_t *ta = sA + (kb & 1) * AST;
    const float *ts = sS + (kb & 1) * T;
    v4i bf[2][2];
    float as_t[2];
    if constexpr (kEarly) {
      // this wave's reads of the weight stage are complete before copies are aimed at it again
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      bf[0][0] = bf_first[0];
      bf[0][1] = bf_first[1];
      as_t[0] = as_first;
    } else {
#pragma unroll
      for (int kh = 0; kh < 2; ++kh) bf[0][kh] = *reinterpret_cast<const v4i *>(ta + alds[kh]);
      as_t[0] = ts[r];
    }
    const float bs0 = W4 ? 0.0f : uniform(sBs0[kb]), bs1 = W4 ? 0.0f : uniform(sBs1[kb]);

    // The weight stage was read into registers before the barrier, so it is free; it and the other
    // token stage are refilled with the next K block, two copies per pipeline stage so that the
    // texture path never sees a burst that this wave (or the other workgroup's) queues behind.
    constexpr int c0 = decltype(BIASED)::value ? kFoldBias : 0;
    const v4i cinit = {c0, c0, c0, c0};
    v4i dprev[2];
    float as_p = 0.0f;
    float as_bias = 0.0f;
    float sc0 = 0.0f, sc1 = 0.0f; // scale products of the token fragment being folded (both row halves)
    auto fold_stage = [&](int st) __attribute__((always_inline)) { // fold the fragments of stage st
      const int tb = st >> 1, h = st & 1;
      if constexpr (PC) return;
      if (decltype(BIASED)::value && h == 0) as_bias = fold_bias(as_p);
      if constexpr (W4) {
        fold4(BIASED, dprev[0], as_p, as_bias, wsc[h][0], acc[h][tb][0]);
        fold4(BIASED, dprev[1], as_p, as_bias, wsc[h][1], acc[h][tb][1]);
        return;
      }
      if (ORD == kOrdFusedScale && h == 0) {
        sc0 = as_p * bs0;
        sc1 = FUSED_ACT ? as_p * bs1 : sc0;
      }
      fold(BIASED, dprev[0], sc0, as_p, as_bias, bs0, acc[h][tb][0]);
      fold(BIASED, dprev[1], sc1, as_p, as_bias, FUSED_ACT ? bs1 : bs0, acc[h][tb][1]);
    };
    // pipeline stage (tb, h): its MFMAs are issued, then the previous stage's fragments are folded
    // while the matrix pipe works; the operands of token fragment tb + 1 are requested in (tb, 0)
#pragma unroll
    for (int st = 0; st < (kFull < 4 ? 4 : kFull); ++st) {
      const int tb = st >> 1, h = st & 1;
      const int cur = tb & 1, nxt = cur ^ 1;
      // int4 weights with K-group scales, full blocks: nine copies, one a stage (two a stage crowd the scale reads: 128-token blocks of
      // 128 experts of 4096 x 1536, us, two / one, at 100 slots per expert 451 / 441, at 169: 749 / 733, at 500: 1729 / 1690; DeepSeek-V3
      // share at 172: 478 / 466, at 250: 626 / 609; blocks of at most 96 tokens lose 1 %, per-channel scales and int8 gain nothing)
      if constexpr (W4 && !PC && nst_c >= 14) {
        if (st < 5 + APW) copy_piece(decltype(ONCE)::value, st < 5 ? st : st + 3, kb + 1);
      } else if (nst_c >= 8 && st < 6) {
        copy_piece(decltype(ONCE)::value, 2 * st, kb + 1);
        copy_piece(decltype(ONCE)::value, 2 * st + 1, kb + 1);
      }
      if (NTB == 10 && nst_c >= 8 && st == 6) copy_piece(decltype(ONCE)::value, 12, kb + 1); // the fifth token piece of a 160-token stage
      if (nst_c < 8 && st < 4) {
        copy_piece(decltype(ONCE)::value, 3 * st, kb + 1);
        copy_piece(decltype(ONCE)::value, 3 * st + 1, kb + 1);
        copy_piece(decltype(ONCE)::value, 3 * st + 2, kb + 1);
      }
      if (st < nst_c) {
        if (kEarly && st == kE0) {
          wait_copies_barrier<0>();
          put_scale(BIASED, kb & 1, kb + 2 < KB ? s_pending : 0.0f);
          s_pending = load_scale(kb + 3);
          __builtin_amdgcn_sched_barrier(0);
        }
        if (h == 0 && st + 2 < nst_c) {
#pragma unroll
          for (int kh = 0; kh < 2; ++kh)
            bf[nxt][kh] = *reinterpret_cast<const v4i *>(ta + (tb + 1) * 16 * kGroup + alds[kh]);
          as_t[nxt] = ts[(tb + 1) * 16 + r];
        }
        v4i d[2];
#pragma unroll
        for (int rf = 0; rf < 2; ++rf)
          d[rf] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w[h][rf][0], bf[cur][0], PC ? acci[h][tb][rf] : cinit, 0, 0, 0);
#pragma unroll
        for (int rf = 0; rf < 2; ++rf)
          d[rf] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w[h][rf][1], bf[cur][1], d[rf], 0, 0, 0);
        if constexpr (PC) {
          acci[h][tb][0] = d[0];
          acci[h][tb][1] = d[1];
        }
        if (kEarly && st >= kE0) { // the next K block's operands of this half, over the ones just used
#pragma unroll
          for (int rf = 0; rf < 2; ++rf)
#pragma unroll
            for (int kh = 0; kh < 2; ++kh)
              w[h][rf][kh] = *reinterpret_cast<const v4i *>(sWw + (h * 2 + rf) * 2048 + wlds[kh]);
          if (st == kE0) {
            const int8_t *tan = sA + ((kb + 1) & 1) * AST;
#pragma unroll
            for (int kh = 0; kh < 2; ++kh) bf_first[kh] = *reinterpret_cast<const v4i *>(tan + alds[kh]);
            as_first = sS[((kb + 1) & 1) * T + r];
          }
        }
        if (st > 0) fold_stage(st - 1);
        if (h == 0 && st + 2 < nst_c) __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          if (nst_c >= 8 ? ((g < 2 && st < 6) || (NTB == 10 && g == 0 && st == 6)) : (g < 3 && st < 4))
            __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
          // 128-token tiles close the stage's products up and fold behind them.  Four (int4: five) after each / this, whole layer,
          // us: all experts of DeepSeek-V3, skewed, 5500 tokens 3244 / 3222, 8192: 4457 / 4430, 12000: 6253 / 6204; share 7000:
          // 650 / 647; Qwen3-235B-A22B-shaped layer 3000: 832 / 823, 6500: 1500 / 1498; Qwen3-30B-A3B layer 3000 and 8192: equal; row-major
          // weights, Qwen3-235B-A22B-shaped 4096: 1062 / 1049, 8192: 1834 / 1802, Qwen3-30B-A3B 8192: 554 / 546 (with the other steps
          // that are in the layer since); int4 with K-group scales, 128 experts of 4096 x 1536, 1100: 375 / 366, 2800: 724 / 711, 6000: 1313 / 1291.  int8 tiles of 160
          // lose (1531 tokens 177 / 180).
          if constexpr (decltype(BIASED)::value && !PC && (W4 || NTB == 8)) {
            if (g < 3) __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
            else __builtin_amdgcn_sched_group_barrier(0x002, W4 ? 14 : 10, 0);
          } else {
            __builtin_amdgcn_sched_group_barrier(0x002, decltype(BIASED)::value ? 4 : W4 ? 7 : 5, 0);
          }
        }
        if (kEarly && st == kE0) __builtin_amdgcn_sched_group_barrier(0x100, 7, 0);
        if (kEarly && st == kE1) __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
        __builtin_amdgcn_sched_barrier(0);
        dprev[0] = d[0];
        dprev[1] = d[1];
        as_p = as_t[cur];
      }
    }
    fold_stage(nst_c - 1);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (!kEarly) {
      // the next K block's weights have had a whole K block to arrive; reading them here puts the
      // LDS latency under the barrier instead of in front of the first MFMA
      wait_copies<0>();
      read_w(BIASED, kb + 1);
    }
  };

  // ---- prologue ------------------------------------------------------------------------------------------
  auto start = [&](auto BIASED) __attribute__((always_inline)) {
    const float s_now = load_scale(0);
    s_pending = load_scale(1);
    __builtin_amdgcn_sched_barrier(0);
    copy_a(0);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (decltype(BIASED)::value) {
      sFlag[wave] = !W4 && __builtin_amdgcn_ballot_w64(!fold_weight_scale_ok(bs_mine)) ? 1 : 0; // one value for the wave
      bs_mine = fold_weight_scale(bs_mine);
    }
    put_scale(BIASED, 0, s_now);
    sBs[tid] = bs_mine;
    wait_copies<0>();
    read_w(BIASED, 0);
  };

  auto k_loop = [&](auto BIASED, auto NST, auto ONCE) __attribute__((always_inline)) {
    if constexpr (decltype(NST)::value >= kEarlyFrom && !W4 && NTB >= 8) {
      wait_copies_barrier<0>(); // K block 0 is complete in LDS
      put_scale(BIASED, 1, 1 < KB ? s_pending : 0.0f);
      s_pending = load_scale(2);
#pragma unroll
      for (int kh = 0; kh < 2; ++kh) bf_first[kh] = *reinterpret_cast<const v4i *>(sA + alds[kh]);
      as_first = sS[r];
      __builtin_amdgcn_sched_barrier(0);
      for (int kb = 0; kb < KB; ++kb) kblock(BIASED, NST, ONCE, kb);
      return;
    }
    for (int kb = 0; kb < KB; ++kb) {
      // every copy this wave requested a K block ago has landed; after the barrier so have everyone
      // else's token rows, and nobody still reads the token stage and the scales of K block kb-1,
      // which are refilled below
      wait_copies_barrier<0>();
      put_scale(BIASED, (kb + 1) & 1, kb + 1 < KB ? s_pending : 0.0f);
      s_pending = load_scale(kb + 2);
      __builtin_amdgcn_sched_barrier(0);
      kblock(BIASED, NST, ONCE, kb);
    }
  };
  constexpr std::integral_constant<bool, kBiased> biased{};
  start(biased);
  if (tid < T) sWgt[tid] = wgt_mine;
  // one K loop per number of token fragments that hold valid tokens (wave-uniform choice)
  // in steps of 16 tokens where the registers allow it: a 96-token block costs three quarters of a full one
  if (kPolicy && alone && (a.stream || nst <= 8)) {
    if constexpr (kPolicy) {
      if (nst > 14) k_loop(biased, std::integral_constant<int, 16>{}, once);
      else if (nst > 12) k_loop(biased, std::integral_constant<int, 14>{}, once);
      else if (nst > 10) k_loop(biased, std::integral_constant<int, 12>{}, once);
      else if (nst > 8) k_loop(biased, std::integral_constant<int, 10>{}, once);
      else if (nst > 6) k_loop(biased, std::integral_constant<int, 8>{}, once);
      else if (nst > 4) k_loop(biased, std::integral_constant<int, 6>{}, once);
      else k_loop(biased, std::integral_constant<int, 4>{}, once);
    }
  } else if constexpr (NTB == 10 && PC) {
    if (nst > 18) k_loop(biased, std::integral_constant<int, 20>{}, by_launch);
    else if (nst > 16) k_loop(biased, std::integral_constant<int, 18>{}, by_launch);
    else if (nst > 14) k_loop(biased, std::integral_constant<int, 16>{}, by_launch);
    else if (nst > 12) k_loop(biased, std::integral_constant<int, 14>{}, by_launch);
    else if (nst > 10) k_loop(biased, std::integral_constant<int, 12>{}, by_launch);
    else if (nst > 8) k_loop(biased, std::integral_constant<int, 10>{}, by_launch);
    else k_loop(biased, std::integral_constant<int, 8>{}, by_launch);
  } else if constexpr (NTB == 10) {
    if (nst > 16) k_loop(biased, std::integral_constant<int, 20>{}, by_launch);
    else if (nst > 12) k_loop(biased, std::integral_constant<int, 16>{}, by_launch);
    else if (nst > 8) k_loop(biased, std::integral_constant<int, 12>{}, by_launch);
    else if (!kHalves || nst > 4) k_loop(biased, std::integral_constant<int, 8>{}, by_launch);
    // int4: skewed routing leaves many experts with a handful of tokens (128 experts of 4096 x 1536, Zipf 1.2, us, without / with
    // this variant: 1800 tokens 601 / 589, 2048: 682 / 672; DeepSeek-V3 share, Zipf 0.6, 4096: 669 / 641)
    else if constexpr (kHalves) k_loop(biased, std::integral_constant<int, 4>{}, by_launch);
  } else if constexpr (NTB == 8 && W4 && !PC) {
    if (nst > 12) k_loop(biased, std::integral_constant<int, 16>{}, by_launch);
    else if (nst > 8) k_loop(biased, std::integral_constant<int, 12>{}, by_launch);
    else if (nst > 4) k_loop(biased, std::integral_constant<int, 8>{}, by_launch);
    else k_loop(biased, std::integral_constant<int, 4>{}, by_launch);
  } else if constexpr (NTB == 8) {
    if (nst > 14) k_loop(biased, std::integral_constant<int, 16>{}, by_launch);
    else if (nst > 12) k_loop(biased, std::integral_constant<int, 14>{}, by_launch);
    else if (nst > 10) k_loop(biased, std::integral_constant<int, 12>{}, by_launch);
    else if (nst > 8) k_loop(biased, std::integral_constant<int, 10>{}, by_launch);
    else if (nst > 6) k_loop(biased, std::integral_constant<int, 8>{}, by_launch);
    else if (nst > 4) k_loop(biased, std::integral_constant<int, 6>{}, by_launch);
    else k_loop(biased, std::integral_constant<int, 4>{}, by_launch);
  } else if constexpr (NTB == 4) {
    if (nst > 6) k_loop(biased, std::integral_constant<int, 8>{}, by_launch);
    else if (nst > 4) k_loop(biased, std::integral_constant<int, 6>{}, by_launch);
    else k_loop(biased, std::integral_constant<int, 4>{}, by_launch);
  } else {
    k_loop(biased, std::integral_constant<int, 2 * NTB>{}, by_launch);
  }
  wait_copies<0>(); // no copy may still be writing LDS when the epilogue reuses it or the wave ends
  derive();
  if constexpr (kMeet && !kBiased) __syncthreads();
  if constexpr (kBiased) {
    // (the flags of the last token scales were written a barrier of the K loop ago)
    if constexpr (W4) {
      if (__builtin_amdgcn_ballot_w64(!fold_weight_scale_ok(ws_max))) sFlag[wave] = 1;
      __syncthreads();
    }
    const v4i met = *reinterpret_cast<const v4i *>(sFlag);
    if (__builtin_expect(__builtin_amdgcn_readfirstlane(met[0] | met[1] | met[2] | met[3]) != 0, 0)) {
      constexpr std::false_type plain{};
      __syncthreads(); // every wave is done with the token stages and the tables
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int tb = 0; tb < NTB; ++tb)
#pragma unroll
          for (int rf = 0; rf < 2; ++rf)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[h][tb][rf][i] = 0.0f;
      copy_w0(STREAM);
      bs_mine = load_bs();
      start(plain);
      k_loop(plain, std::integral_constant<int, 2 * NTB>{}, by_launch);
      wait_copies<0>();
      derive();
      if constexpr (kMeet) __syncthreads();
    }
  }
  if constexpr (!FUSED_ACT) {
    if (!wave_active) return;
    // A lane holds 4 consecutive columns of one token per fragment.  Each wave turns a 16-token x
    // 64-column piece around in its own (now idle) weight ring and stores 128-byte row segments.
    int8_t *stg = sWw;
    // PC: the scales of the lane's rows and of its eight tokens, fetched in one batch up front
    v4f pbs[2][2];
    float pas[NTB];
    if constexpr (PC) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int rf = 0; rf < 2; ++rf)
          pbs[h][rf] = __builtin_bit_cast(v4f, bld16(rWs, static_cast<int>((nrow0 + h * 32 + rf * 16 + 4 * q) * 4), 0));
#pragma unroll
      for (int tb = 0; tb < NTB; ++tb) {
        const int64_t ft = sIds[tb * 16 + r];
        pas[tb] = bld_f32(rAs, static_cast<int>(token_row(a, ft) * 4), 0);
      }
    }
#pragma unroll
    for (int tb = 0; tb < NTB; ++tb) {
      if (2 * tb >= nst) continue;
      const int64_t ft = sIds[tb * 16 + r];
      const bool valid = ft < a.num_valid;
      const float wgt = sWgt[tb * 16 + r];
      with_out16(a.out_f16, [&](auto cvt) __attribute__((always_inline)) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int rf = 0; rf < 2; ++rf) {
            v4u16 o;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              float v;
              if constexpr (PC && W4) { // left to right: routed weight, token scale, channel scale (w4a8.py:386-395)
                v = static_cast<float>(acci[h][tb][rf][i]);
                if (a.mul_routed) v = v * wgt;
                v = v * pas[tb];
                v = v * pbs[h][rf][i];
              } else if constexpr (PC) { // int8 weights: (f32(d) * ts) * b_s, ts = w * a_s (moe_w8a8.cu:452, :466)
                const float ts = a.mul_routed ? wgt * pas[tb] : pas[tb];
                v = static_cast<float>(acci[h][tb][rf][i]) * ts;
                v = v * pbs[h][rf][i];
              } else {
                v = acc[h][tb][rf][i];
                if (a.mul_routed) v = v * wgt;
              }
              o[i] = cvt(v);
            }
            *reinterpret_cast<v4u16 *>(stg + r * kTPitch + (h * 32 + rf * 16 + 4 * q) * 2) = o;
          }
      });
      __builtin_amdgcn_wave_barrier();
      const int slot = valid ? static_cast<int>(ft) : -1;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int tok = (lane >> 3) + 8 * j;
        const v4i v = *reinterpret_cast<const v4i *>(stg + tok * kTPitch + (lane & 7) * 16);
        const int fs = __shfl(slot, tok);
        if (fs >= 0) *reinterpret_cast<v4i *>(a.C + static_cast<int64_t>(fs) * N + nrow0 + (lane & 7) * 8) = v;
      }
      __builtin_amdgcn_wave_barrier();
    }
  } else if constexpr (PC) {
    // The gated activation of a per-channel first stage, in 16 bits: its quantisation needs the whole row.  Gate and up meet
    // here, so that half as much is written and read back as with a plain first stage, and by a launch without the activation.
    int8_t *stg = sWw;
    v4f pbs[2][2];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int rf = 0; rf < 2; ++rf)
        pbs[h][rf] = __builtin_bit_cast(v4f, bld16(rWs, static_cast<int>(((rf ? I : 0) + nrow0 + h * 16 + 4 * q) * 4), 0));
    float pas[NTB];
#pragma unroll
    for (int tb = 0; tb < NTB; ++tb) pas[tb] = bld_f32(rAs, static_cast<int>(token_row(a, sIds[tb * 16 + r]) * 4), 0);
#pragma unroll
    for (int tb = 0; tb < NTB; ++tb) {
      if (2 * tb >= nst) continue;
      const int64_t ft = sIds[tb * 16 + r];
      const bool valid = ft < a.num_valid;
      const float wgt = sWgt[tb * 16 + r];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        float gu[2][4], act[4];
#pragma unroll
        for (int rf = 0; rf < 2; ++rf)
#pragma unroll
          for (int i = 0; i < 4; ++i) { // the orders of the plain epilogue above; a weight of one changes nothing
            float v = static_cast<float>(acci[h][tb][rf][i]);
            if constexpr (W4) v = (v * wgt) * pas[tb];
            else v = v * (wgt * pas[tb]);
            gu[rf][i] = v * pbs[h][rf][i];
          }
        gated_act<FUSED_ACT, 4>(a, gu[0], gu[1], act);
        v4u16 o;
        with_out16(a.out_f16, [&](auto cvt) __attribute__((always_inline)) {
#pragma unroll
          for (int i = 0; i < 4; ++i) o[i] = cvt(act[i]);
        });
        *reinterpret_cast<v4u16 *>(stg + r * kTPitch + (h * 16 + 4 * q) * 2) = o;
      }
      __builtin_amdgcn_wave_barrier();
      const int slot = valid ? static_cast<int>(ft) : -1, tok = lane >> 2;
      const v4i v = *reinterpret_cast<const v4i *>(stg + tok * kTPitch + (lane & 3) * 16);
      const int fs = __shfl(slot, tok);
      if (fs >= 0) *reinterpret_cast<v4i *>(a.C + static_cast<int64_t>(fs) * I + nrow0 + (lane & 3) * 8) = v;
      __builtin_amdgcn_wave_barrier();
    }
  } else {
    // acc[h][tb][0] = gate, acc[h][tb][1] = up for activation columns nt*128 + wave*32 + 16h + 4q + i
    float actf[NTB][2][4];
    if (a.mul_routed) { // router weight on the first GEMM's output: rare, kept out of the main pass
#pragma unroll
      for (int tb = 0; tb < NTB; ++tb) {
        const float wgt = sWgt[tb * 16 + r];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int rf = 0; rf < 2; ++rf)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[h][tb][rf][i] = acc[h][tb][rf][i] * wgt;
      }
    }
    // Token fragments go in pairs that share one wave-uniform branch (of the last pair's second one every value may be zero).
#pragma unroll
    for (int tb = 0; tb < NTB; ++tb) {
      if (2 * (tb & ~1) >= nst) continue; // the same condition for both fragments of a pair
#pragma unroll
      for (int h = 0; h < 2; ++h) gated_act<FUSED_ACT, 4>(a, acc[h][tb][0], acc[h][tb][1], actf[tb][h]);
      float amax = 0.0f;
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < 4; ++i) amax = fmaxf(amax, fabsf(actf[tb][h][i]));
      amax = fmaxf(amax, __shfl_xor(amax, 16));
      amax = fmaxf(amax, __shfl_xor(amax, 32));
      if (q == 0) sRed[wave * T + tb * 16 + r] = amax;
    }
    __syncthreads(); // also: every wave is done with the token stages
    const int64_t G = I / kGroup;
    // the quantised tile (128 tokens x 128 columns of int8) leaves through LDS as whole rows
    int8_t *qst = sA;
    // scales of all eight fragments first, outside the branches on nst: the reads are in bounds
    // either way, and one batch of LDS reads replaces eight dependent chains
    float sc_all[NTB], y_all[NTB];
    bool plain = true; // one wave-uniform branch for the tile's rows
    auto row_max = [&](int tb) __attribute__((always_inline)) {
      const int t = tb * 16 + r;
      return fmaxf(fmaxf(sRed[t], sRed[T + t]), fmaxf(sRed[2 * T + t], sRed[3 * T + t]));
    };
#pragma unroll
    for (int tb = 0; tb < NTB; ++tb) {
      const bool fits = group_scale16(row_max(tb), 1e-10f, sc_all[tb], y_all[tb]);
      plain &= fits || 2 * (tb & ~1) >= nst; // (of fragments that are not in use nothing was written)
    }
    plain = __builtin_amdgcn_ballot_w64(!plain) == 0;
    auto put = [&](auto PLAIN) __attribute__((always_inline)) {
#pragma unroll
      for (int tb = 0; tb < NTB; ++tb) {
        if (2 * (tb & ~1) >= nst) continue;
        const int t = tb * 16 + r;
        if constexpr (!decltype(PLAIN)::value) sc_all[tb] = fmaxf(row_max(tb), 1e-10f) / 127.0f;
#pragma unroll
        for (int h = 0; h < 2; ++h)
          *reinterpret_cast<uint32_t *>(qst + t * kTPitch + wave * 32 + h * 16 + 4 * q) =
              decltype(PLAIN)::value ? quant4_mul(actf[tb][h], y_all[tb]) : quant4_div(actf[tb][h], sc_all[tb]);
        if (wave == (tb & 3) && q == 0) { // every wave holds every token's scale: the stores are shared out
          const int64_t ft = sIds[t];
          if (ft < a.num_valid) a.A2s[ft * G + nt] = sc_all[tb];
        }
      }
    };
    if (__builtin_expect(plain, 1)) put(std::true_type{});
    else put(std::false_type{});
    __syncthreads();
#pragma unroll
    for (int j = 0; j < (T * 8 + 255) / 256; ++j) {
      const int id = tid + 256 * j, tok = id >> 3, piece = id & 7;
      if (NTB == 1 && tok >= T) break;
      const int64_t ft = sIds[tok];
      if (ft < a.num_valid)
        *reinterpret_cast<v4i *>(a.A2q + ft * I + static_cast<int64_t>(nt) * kGroup + piece * 16) =
            *reinterpret_cast<const v4i *>(qst + tok * kTPitch + piece * 16);
    }
  }
}

bool gemm_t128_supports(const GemmArgs &a, bool fused_act, int block_size_m) {
  if (block_size_m == kT160) {
    if (!a.w_shuffled || a.K / kGroup > kTMaxKB) return false;
    return fused_act || a.N % 64 == 0;
  }
  if (block_size_m != 128 || !a.w_shuffled) return false;
  if (a.per_channel && !a.w4) return false; // int8 per-channel weights have gemm_pc.hip
  if (!fused_act && a.N % 64 != 0) return false;
  return a.K / kGroup <= kTMaxKB;
}

// ---- row-major weights -----------------------------------------------------------------------------------
// Weights as a checkpoint holds them, [E, N, K].  Loading an MFMA operand straight from global memory asks for 64 bytes
// of each of 16 rows per instruction (32 of 32 rows with the 32x32 form): every 128-byte line is requested two to four
// times over, and what of it is still in L1 by then is luck, the rows being a power of two apart.  Copied into LDS
// instead, a request is eight whole lines, each once, and the operand reads then find their 16-byte pieces swizzled by
// row as the tokens' are.  The data movement is otherwise that of the pre-shuffled form.  Measured (whole layer with its
// router, us, register-fed kernels / this one): Qwen3-30B-A3B layer at 24 tokens 146 / 105, at 250: 211 / 131, at 8192: 857 /
// 630; Qwen3-235B-A22B-shaped layer at 200 tokens 676 / 457; DeepSeek-V3 share at 64 tokens 302 / 213 - within a few
// percent of the load-time layout.
//
// Tiles: 16, 32, 64 or 128 tokens as the alignment blocks are, with four, three, three and two workgroups per compute unit
// (64 tokens at 167 registers: three instead of two take the layer at 8192 tokens from 706 to 653 us, the DeepSeek-V3 share
// at 4096 from 543 to 505).
bool gemm_rows_supports(const GemmArgs &a, bool fused_act, int block_size_m) {
  if (a.w_shuffled || a.w4 || a.out_f32) return false;
  if (block_size_m != 16 && block_size_m != 32 && block_size_m != 64 && block_size_m != 128) return false;
  return (fused_act || a.N % 64 == 0) && (a.per_channel || a.K / kGroup <= kTMaxKB);
}

template <int NTB>
static int launch_rows(const GemmArgs &a, bool fused_act, int ord, bool stream, dim3 g, int mbi, int gi, hipStream_t s) {
  constexpr int T = 16 * NTB;
  constexpr int kLds = kTW + 2 * T * kGroup + 2 * T * 4 + 4 * T * 4 + kTBs + 2 * T * 4 + kTFlag;
#define LO_ROWS_LAUNCH2(ORD, FA, ST, PCV)                                                                       \
  do {                                                                                                          \
    static unsigned long long lds_done = 0; /* per instantiation: one bit per device */                         \
    const auto kern = &moe_gemm_t128_kernel<FA, ORD, ST, false, PCV, NTB, true>;                                \
    const int rc_lds = reserve_lds_once(reinterpret_cast<const void *>(kern), kLds, &lds_done);                 \
    if (rc_lds) return rc_lds;                                                                                  \
    hipLaunchKernelGGL(kern, g, dim3(256), kLds, s, a, mbi, gi);                                                \
  } while (0)
#define LO_ROWS_LAUNCH(ORD, FA)                                                                                 \
  do {                                                                                                          \
    if (stream) LO_ROWS_LAUNCH2(ORD, FA, true, false);                                                          \
    else LO_ROWS_LAUNCH2(ORD, FA, false, false);                                                                \
  } while (0)
  if (a.per_channel) { // one order only: the scales meet in the epilogue
#define LO_ROWS_LAUNCH_PC(FA)                                           \
  do {                                                                  \
    if (stream) LO_ROWS_LAUNCH2(kOrdSeparate, FA, true, true);          \
    else LO_ROWS_LAUNCH2(kOrdSeparate, FA, false, true);                \
  } while (0)
    LO_GATED_DISPATCH(a, fused_act, LO_ROWS_LAUNCH_PC);
#undef LO_ROWS_LAUNCH_PC
  } else if (fused_act) {
    LO_FUSED_DISPATCH(a, ord, LO_ROWS_LAUNCH);
  } else {
    LO_ORD_DISPATCH(ord, LO_ROWS_LAUNCH, 0);
  }
#undef LO_ROWS_LAUNCH
#undef LO_ROWS_LAUNCH2
  return check_launch(a.per_channel ? "moe_gemm_w8a8(rows)" : fused_act ? "moe_gemm1_silu_quant(rows)" : "moe_gemm(rows)");
}

int launch_gemm_rows(const GemmArgs &a0, bool fused_act, int block_size_m, int flags, int64_t m_blocks, hipStream_t s) {
  GemmArgs a = a0;
  a.n_tiles = fused_act ? static_cast<int32_t>(a.N / 2 / kGroup) : static_cast<int32_t>((a.N + 255) / 256);
  const int64_t experts = a.experts_routed > 0 ? a.experts_routed : 1;
  // one token block per expert, by and large: the weights have one reader (as in gemm_tile.hip)
  const bool stream = a.num_valid <= experts * 48;
  int64_t G = a.num_valid / (experts * block_size_m);
  G = G < 2 ? 2 : (G > 16 ? 16 : G);
  const int64_t chunks = (m_blocks + G - 1) / G;
  const int64_t grid = (chunks + 7) / 8 * (G * a.n_tiles) * 8;
  LO_REQUIRE(grid < (1ll << 31), LO_EINVAL, "moe_gemm: grid too large");
  const int ord = scale_order(flags);
  const dim3 g(static_cast<unsigned>(grid));
  const int mbi = static_cast<int>(m_blocks), gi = static_cast<int>(G);
  switch (block_size_m) {
  case 16: return launch_rows<1>(a, fused_act, ord, stream, g, mbi, gi, s);
  case 32: return launch_rows<2>(a, fused_act, ord, stream, g, mbi, gi, s);
  case 64: return launch_rows<4>(a, fused_act, ord, stream, g, mbi, gi, s);
  default: return launch_rows<8>(a, fused_act, ord, stream, g, mbi, gi, s);
  }
}

int launch_gemm_t128(const GemmArgs &a0, bool fused_act, int block_size_m, int flags, int64_t m_blocks,
                     hipStream_t s) {
  GemmArgs a = a0;
  a.n_tiles = fused_act ? static_cast<int32_t>(a.N / 2 / kGroup) : static_cast<int32_t>((a.N + 255) / 256);
  const int64_t experts = a.experts_routed > 0 ? a.experts_routed : 1;
  // token blocks of a chunk: about an expert's
  int64_t G = (a.num_valid + (block_size_m == kT160 ? experts * 64 : 0)) / (experts * block_size_m);
  // (One block of 160 an expert, and not many experts: a chunk is one block.  What spills into a second block is a handful of
  // workgroups after the first round, and in chunks of two they meet on a few dies.  DeepSeek-V3 share, chunks of two / of one, us:
  // 4000 tokens 490 / 465, 4200: 492 / 469, 3500, where nothing spills: 363 / 364; second stage with 5 of 32 experts past 160:
  // 166 / 148.  Two blocks an expert share its weights and stay together (Qwen3-30B-A3B layer, 4096 tokens 332 / 363), and 256
  // experts of skewed routing, some with many, lose as well: 4000 tokens 2988 / 3013.)
  const int64_t least = block_size_m == kT160 && a.E <= 128 ? 1 : 2;
  G = G < least ? least : (G > 16 ? 16 : G);
  const int64_t chunks = (m_blocks + G - 1) / G;
  const int64_t grid = (chunks + 7) / 8 * (G * a.n_tiles) * 8;
  LO_REQUIRE(grid < (1ll << 31), LO_EINVAL, "moe_gemm: grid too large");
  const int ord = scale_order(flags);
  const dim3 g(static_cast<unsigned>(grid)), b(256);
  const int mbi = static_cast<int>(m_blocks), gi = static_cast<int>(G);
#define LO_T128_LAUNCH(FA, FS, ST, W)                                                                           \
  do {                                                                                                          \
    static unsigned long long lds_done = 0; /* per instantiation: one bit per device */                         \
    const int rc_lds = reserve_lds_once(reinterpret_cast<const void *>(&moe_gemm_t128_kernel<FA, FS, ST, W>),    \
                                        kTLds, &lds_done);                                                      \
    if (rc_lds) return rc_lds;                                                                                  \
    hipLaunchKernelGGL((moe_gemm_t128_kernel<FA, FS, ST, W>), g, b, kTLds, s, a, mbi, gi);                      \
  } while (0)
#define LO_T128_LAUNCH_PC2(FA, ST, W, NTB, LDS)                                                                 \
  do {                                                                                                          \
    static unsigned long long lds_done = 0;                                                                     \
    const auto kern = &moe_gemm_t128_kernel<FA, kOrdSeparate, ST, W, true, NTB>;                                \
    const int rc_lds = reserve_lds_once(reinterpret_cast<const void *>(kern), LDS, &lds_done);                  \
    if (rc_lds) return rc_lds;                                                                                  \
    hipLaunchKernelGGL(kern, g, b, LDS, s, a, mbi, gi);                                                         \
  } while (0)
#define LO_T128_LAUNCH_PC(FA)                                                                                   \
  do {                                                                                                          \
    if (a.stream) LO_T128_LAUNCH_PC2(FA, true, true, 8, kTLds);                                                 \
    else LO_T128_LAUNCH_PC2(FA, false, true, 8, kTLds);                                                         \
  } while (0)
#define LO_T160_LAUNCH_PC(FA)                                                                                   \
  do {                                                                                                          \
    if (a.w4 && a.stream) LO_T128_LAUNCH_PC2(FA, true, true, 10, kTLds160);                                     \
    else if (a.w4) LO_T128_LAUNCH_PC2(FA, false, true, 10, kTLds160);                                           \
    else if (a.stream) LO_T128_LAUNCH_PC2(FA, true, false, 10, kTLds160);                                       \
    else LO_T128_LAUNCH_PC2(FA, false, false, 10, kTLds160);                                                    \
  } while (0)
#define LO_T128_PICK(FS, FA)                                                                                    \
  do {                                                                                                          \
    if (a.w4) LO_T128_LAUNCH(FA, FS, false, true);                                                              \
    else LO_T128_LAUNCH(FA, FS, false, false);                                                                  \
  } while (0)
  if (block_size_m == kT160) {
    // Tiles for one or two rounds of the 512 resident workgroups and almost half a round more: if they take different
    // times, the compute units that finish first take both workgroups of the half round and the rest none.  Kept alike they
    // finish together, and the half round is one workgroup to a compute unit.  Whole layer, us, fragments as they are / rounded
    // up to 8: Qwen3-30B-A3B layer (1.5 rounds of first-stage tiles) at 75 slots per expert 181 / 186, at 84: 191 / 185, at
    // 92: 197 / 184, at 108: 205 / 195, at 118: 203 / 203; 62 experts of 4096 x 1536 (1.45) at 72: 279 / 289, at 84: 290 / 282, at
    // 92: 302 / 283.  It costs time where the last round is fuller (130 experts of 2048 x 768, 1.52 rounds, at 92: 209 / 215)
    // or shorter (128 of 2048 x 640, 1.25, at 88: 172 / 183), with a longer K (48 of 7168 x 2048, 1.5, at 88: 453 / 469) and with
    // per-channel scales (the first layer at 92: 196 / 198).
    const double slots = static_cast<double>(a.num_valid) / (a.experts_routed > 0 ? a.experts_routed : 1);
    const double rounds = static_cast<double>(a.E) * a.n_tiles / 512.0, part = rounds - static_cast<int>(rounds); // (a block an expert)
    a.coarse_fill = !a.per_channel && a.K <= 4096 && slots >= 84.0 && rounds >= 1.0 && rounds < 3.0 && part >= 0.4 && part <= 0.5;
    // Copy policy.  int8 weights: the streaming hint while an expert has one block, with large experts while it is far from full,
    // and not where skewed routing gives some of many experts several blocks.  With it / without, whole call with its router, us:
    // Qwen3-30B-A3B layer at 96 slots 180 / 185, at 128: 199 / 205, per-channel 201 / 205; 128 experts of 4096 x 1536 at 94 to 128: equal;
    // DeepSeek-V3 share at 94: 361 / 366, at 125: 502 / 481, per-channel 462 / 447; the full layer with Zipf routing at 128: 3096 / 2571;
    // two blocks an expert, Qwen3-30B-A3B layer at 262: 338 / 301.  (The number of experts says nothing about skew: it parts the
    // layers measured.)  int4 weights, half the bytes, with one scale per row: with it where an expert has one block, 128 experts of
    // 4096 x 1536 at 2048 tokens 422 / 435, at 4300: 745 / 710.  int4 weights with K-group scales: in the first stage only, whose
    // weights are twice the second's; there it costs skewed routing, whose busy experts' blocks share them, and gains uniform routing
    // nothing.  With it in both / the first / neither: the same layer at 1800 / 2048 / 2300 tokens 483 / 484 / 484, 522 / 518 / 540, 586 /
    // 594 / 600, Zipf 1.2 585 / 573 / 547, 674 / 656 / 627, 683 / 668 / 638; 128 experts of 2048 x 768 at 1800: 192 / 184 / 188, Zipf 1.2
    // 226 / 216 / 208; DeepSeek-V3 share at 4096: 338 / 342 / 345, Zipf 0.6 635 / 623 / 594.
    a.stream = a.w4 ? slots <= 160.0 : a.E <= 128 && slots < (a.N * a.K <= (8 << 20) ? 160.0 : 112.0);
#define LO_T160_LAUNCH2(FS, FA, ST, W)                                                                          \
  do {                                                                                                          \
    static unsigned long long lds_done = 0;                                                                     \
    const auto kern = &moe_gemm_t128_kernel<FA, FS, ST, W, false, 10>;                                          \
    const int rc_lds = reserve_lds_once(reinterpret_cast<const void *>(kern), kTLds160, &lds_done);             \
    if (rc_lds) return rc_lds;                                                                                  \
    hipLaunchKernelGGL(kern, g, b, kTLds160, s, a, mbi, gi);                                                    \
  } while (0)
#define LO_T160_LAUNCH(FS, FA)                                                                                  \
  do {                                                                                                          \
    if (a.w4) LO_T160_LAUNCH2(FS, FA, (FA) != 0, true);                                                         \
    else if (a.stream) LO_T160_LAUNCH2(FS, FA, true, false);                                                    \
    else LO_T160_LAUNCH2(FS, FA, false, false);                                                                 \
  } while (0)
    if (a.per_channel) {
      LO_GATED_DISPATCH(a, fused_act, LO_T160_LAUNCH_PC);
    } else if (fused_act) {
      LO_ORD_DISPATCH(ord, LO_T160_LAUNCH, kActSiluBf16);
    } else {
      LO_ORD_DISPATCH(ord, LO_T160_LAUNCH, 0);
    }
#undef LO_T160_LAUNCH
#undef LO_T160_LAUNCH2
    return check_launch(fused_act ? "moe_gemm1_silu_quant(t160)" : "moe_gemm(t160)");
  }
  // Copy policy.  int8: a block that shares its weights runs without the hint, one alone with it up to this average (past it up to
  // 64 tokens).  With the hint / without at 40 / 50 / 62 / 80 slots per expert, us: DeepSeek-V3 share 288 / 298, 301 / 310, 311 / 313,
  // 325 / 327; the full layer's skewed routing, where the average misleads, at 500 / 1000 / 2000 tokens: 1022 / 992, 1475 / 1337,
  // 2006 / 1611.  int4 with one scale per row, by the average, 128 experts of 4096 x 1536 at 16 / 32 / 44 / 62 slots: 251 / 258, 270 /
  // 271, 285 / 283, 306 / 303.  int4 with K-group scales, here from 50 slots per expert on, without it: at 50 / 62 340 / 334, 361 / 357.
  a.stream = a.num_valid <= experts * (a.w4 ? 40 : kT / 2);
  if (a.per_channel) {
    LO_GATED_DISPATCH(a, fused_act, LO_T128_LAUNCH_PC);
  } else if (fused_act) {
    LO_FUSED_DISPATCH(a, ord, LO_T128_PICK);
  } else {
    LO_ORD_DISPATCH(ord, LO_T128_PICK, 0);
  }
#undef LO_T128_PICK
#undef LO_T160_LAUNCH_PC
#undef LO_T128_LAUNCH_PC
#undef LO_T128_LAUNCH_PC2
#undef LO_T128_LAUNCH
  return check_launch(fused_act ? "moe_gemm1_silu_quant(t128)" : "moe_gemm(t128)");
}

} // namespace lo
