// Decode-size whole path of the fused MoE in two launches.
//
// With a handful of tokens the path is a stream of weights (2 * tokens op/B against a ridge of
// 629) and every launch costs about as much as the bytes it moves, so the stages of the
// reference (quant, align, GEMM1, activation + quant, GEMM2, reduce:
// python/lightop/_lmslim_native/layers/fused_moe/int8.py:752-888, w4a8.py:560-640) are folded into two kernels
// that need no alignment buffers, no quantised copy of x and no per-slot output rows, and whose
// workgroups never wait for one another:
//
//   dec_gemm1_kernel   one workgroup per (expert hit, 16 activation columns).  Every wave reads topk_ids itself and
//                      finds the u-th distinct expert of this rank and the slots routed to it by ballots (u =
//                      blockIdx.y, blockIdx.y + gridDim.y, ...), so an expert's weights are read once and no workgroup
//                      is launched for a slot of another rank.  The waves split K: each streams its own K blocks of the
//                      16 gate rows and the matching 16 up rows from HBM, three or four of them in flight, quantises its K range
//                      of the token rows into LDS meanwhile, and leaves one product f32(d) * a_s per K block in LDS
//                      (1x128 groups, layers/gemm/int8_utils.py:74-122).  The sum over K runs in K order (acc =
//                      fma(product, b_s, acc), or acc + product * b_s with LO_GEMM_SEPARATE_ORDER), so after one barrier the
//                      last wave walks the products; it ends with the gated activation (int8.py:811-838) and writes
//                      the 16-bit activations [S, I].
//   dec_gemm2_kernel   one workgroup per (token, 16 to 128 output columns), its waves sharing out the token's slots on
//                      this rank and the 16-column pieces: a wave re-quantises its slot's activation row
//                      (int8.py:813-823) into LDS while its expert's 16 weight rows are on their way, multiplies
//                      (int8.py:857-880), and the workgroup then reduces the token's slots in slot order
//                      (csrc/kernels/moe_align_sum_kernels.cu:619-633, :886-909) and writes the output row.  No per-slot
//                      rows in HBM and no separate reduction launch.
//
// PC: per-channel scales (int8.py:771-855 with block_shape=None; with W4 the reference's own int4 form, w4a8.py:202-401).
// A token's scale needs its whole row, so the waves exchange row maxima before they quantise; the int32 sums of the waves'
// K ranges are added exactly and the scales meet in the epilogue.
//
// The second kernel reads an expert's weights once per slot routed to it, which is why the path
// is taken only while slots rarely share an expert.
#include <cstdlib>
#include <type_traits>

#include "gemm.h"

namespace lo {

constexpr int kDecTP = 4;     // token rows the first kernel multiplies per pass
constexpr int kDecMaxKBw = 7; // K blocks per wave of the first kernel
constexpr int kDecMaxSlots = 512;
constexpr int kDecMaxKB2 = 32;  // K blocks of the second kernel (I <= 4096): its activation row is held in registers

struct DecArgs {
  const uint16_t *x;         // [M, H] 16-bit
  const void *ids;           // [S] int32 / int64
  const int32_t *expert_map; // [Eg] or null
  const float *topk_w;       // [S]
  const int8_t *w1, *w2;     // load-time layout
  const float *w1s, *w2s;
  const uint16_t *shared;    // [M, H] or null
  const uint16_t *table;     // T(act(g)) of the gated activation, or null: SiLU, computed
  uint16_t *act;             // [S, I]: activation(gate) * up of every local slot
  uint16_t *out;             // [M, H]
  float factor;
  int32_t ids64, M, S, top_k, E, Eg, H, I, kbw, mul_on_input;
  int32_t ebits;             // bits of a local expert id
  int32_t nrb2;              // 16-column pieces per workgroup of the second kernel
  int32_t floor2;            // (PC) the second quantisation floors the row maximum (GELU)
  int32_t contract;          // acc = fma(f32(d) * a_s, b_s, acc) (the default order); 0: acc + (f32(d) * a_s) * b_s
};

// Local expert that serves flat slot s, or -1 (also for an id or a map entry out of range: served by nobody, adds zero).
__device__ __forceinline__ int dec_expert(const DecArgs &a, int s) {
  const int64_t g = a.ids64 ? static_cast<const int64_t *>(a.ids)[s] : static_cast<const int32_t *>(a.ids)[s];
  int le = -1;
  if (g >= 0 && g < a.Eg) le = a.expert_map ? a.expert_map[g] : static_cast<int>(g);
  return le >= a.E ? -1 : le;
}

// Eight values of a 16-bit row as floats and their largest magnitude.
template <int DT> __device__ __forceinline__ float dec_widen8(const v8u16 raw, float (&v)[8]) {
  float amax = 0.0f;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    v[i] = to_f32<DT>(raw[i]);
    amax = fmaxf(amax, fabsf(v[i]));
  }
  return amax;
}

// Quantise one 128-value group (8 values per lane of a 16-lane group) and return the packed bytes.  MUL: by one multiplication a
// value; not in the first kernel of int4 weights with K-group scales, where more registers spill with it (36 bytes instead of 20: one
// token of the Qwen3-235B-A22B-shaped layer 28.5 us instead of 27.5).
template <int DT, bool MUL = true> __device__ __forceinline__ v2i dec_quant8(const v8u16 raw, float &scale) {
  float v[8];
  float amax = dec_widen8<DT>(raw, v);
#pragma unroll
  for (int d = 1; d < 16; d <<= 1) amax = fmaxf(amax, __shfl_xor(amax, d));
  if constexpr (MUL) return group_quant8<true>(v, amax, 1e-10f, scale);
  const float s = fmaxf(amax, 1e-10f) / 127.0f, y = 1.0f / s;
  scale = s;
  if (s < __builtin_inff()) return v2i{static_cast<int>(quant4_rcp(&v[0], s, y)), static_cast<int>(quant4_rcp(&v[4], s, y))};
  return v2i{static_cast<int>(quant4_div(&v[0], s)), static_cast<int>(quant4_div(&v[4], s))};
}

// The per-token rule: round to nearest of v * (127 / amax).
template <int DT> __device__ __forceinline__ v2i dec_quant8_row(const v8u16 raw, float inv) {
  float v[8];
  (void)dec_widen8<DT>(raw, v);
  int q[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) q[i] = rne_i8(v[i] * inv);
  return v2i{static_cast<int>(pack4_i8(q[0], q[1], q[2], q[3])), static_cast<int>(pack4_i8(q[4], q[5], q[6], q[7]))};
}

__device__ __forceinline__ float wave_max64(float v) {
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) v = fmaxf(v, __shfl_xor(v, d));
  return v;
}

// The two MFMA operands (k-steps) of a K block from a lane's 16 bytes of packed int4 in the load-time
// layout: int8 values 16 times too large (reference nibble order: layers/fused_moe/w4a8.py:341, :375-377).
__device__ __forceinline__ void unpack_int4(const v4i pk, v4i &w0, v4i &w1) {
#pragma unroll
  for (int x = 0; x < 2; ++x) {
    const uint32_t a0 = static_cast<uint32_t>(pk[x]), a1 = static_cast<uint32_t>(pk[2 + x]);
    w0[2 * x] = static_cast<int>((a0 << 4) & 0xf0f0f0f0u);
    w0[2 * x + 1] = static_cast<int>(a0 & 0xf0f0f0f0u);
    w1[2 * x] = static_cast<int>((a1 << 4) & 0xf0f0f0f0u);
    w1[2 * x + 1] = static_cast<int>(a1 & 0xf0f0f0f0u);
  }
}

__device__ __forceinline__ float lane_value(float v, int l) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l));
}
__device__ __forceinline__ uint64_t lane_mask(uint64_t v, int l) {
  return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), l)) |
         static_cast<uint64_t>(static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v >> 32), l))) << 32;
}

// Both kernels are chains of dependent memory round trips (ids -> expert -> weights), each about as
// long as the streaming itself at these sizes, so everything whose address does not depend on the
// routing is requested before the routing is looked at, everything that depends on the expert only the moment the expert
// is known, and what is needed first is requested first: vector-memory operations return in order, so a small load
// behind the weights would be waited for as long as they are.
// KBW: K blocks per wave at most (4, or kDecMaxKBw; a wave's steps past its own count re-read its last block and meet
// zeros).  W4: packed int4 weights in their load-time layout (one 16-byte piece per lane holds both k-steps of a K
// block), block form: one scale per weight row and K block, [E, K/128, N]; the factor 16 of the unpacked nibbles leaves through
// the scales.
template <int KBW, bool W4, bool PC, int DT>
__device__ __forceinline__ void dec_gemm1_body(const DecArgs &a) {
  extern __shared__ __attribute__((aligned(16))) int8_t smem[];
  constexpr int RQ = (KBW + 3) / 4; // 16-byte pieces of a token row per lane: lane (gq, sub) holds piece sub of group gq + 4q
  constexpr bool GS = W4 && !PC;    // group scales of int4 weights, one per row and K block
  constexpr int RING = KBW > 4 && !(W4 && PC) ? 3 : 4; // K blocks of weights a wave has in flight: what 128 registers hold
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int W = blockDim.x >> 6;
  const int n = lane & 15, c = lane >> 4;
  const int sub = lane & 15, gq = lane >> 4;
  const int rb = blockIdx.x;
  const int KB = a.H / kGroup, KBw = a.kbw, kb0 = wave * KBw;
  const int I = a.I, N = 2 * I;
  const int pitch = KBw * kGroup + 16;

  // LDS: the products of every K block (PC: the waves' int32 sums) and the weight scales they meet, slot list (long batches
  // only), row maxima, per-wave token tiles
  constexpr int SB = GS ? 32 : 2; // weight scales per K block: one per row ([8 values][4 c]), else gate block, up block
  float *const sT = reinterpret_cast<float *>(smem);                            // [KB][8 values][4 c][TP tokens]; PC [W][...]
  int32_t *const sTi = reinterpret_cast<int32_t *>(smem);
  float *const sB = sT + (PC ? W : KB) * 128;                                   // [KB][SB]
  float *const sMax = sB + (PC ? 0 : KB * SB);                                  // [W][TP]
  int32_t *const sSlots = reinterpret_cast<int32_t *>(sMax + W * kDecTP);       // [S rounded up to 4], [4]
  const int list = a.S > 64 ? ((a.S + 3) & ~3) : 0;
  int32_t *const sMeta = sSlots + list;
  float *const sAs = reinterpret_cast<float *>(sMeta + 4) + wave * (kDecTP * KBW); // [TP][KBW] of this wave
  int8_t *const sA = reinterpret_cast<int8_t *>(reinterpret_cast<float *>(sMeta + 4) + W * (kDecTP * KBW)) + wave * (kDecTP * pitch);

  auto load_row = [&](int64_t t, v8u16 (&raw)[RQ]) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < RQ; ++q) {
      const int g = gq + 4 * q;
      raw[q] = *reinterpret_cast<const v8u16 *>(a.x + t * a.H + (kb0 + (g < KBw ? g : 0)) * kGroup + sub * 8);
    }
  };
  v8u16 raw[kDecTP][RQ];
  if (a.M == 1) load_row(0, raw[0]); // one token: its row does not wait for the routing

  const int64_t wbytes = W4 ? static_cast<int64_t>(N) * a.H / 2 : static_cast<int64_t>(N) * a.H;
  const int wkstride = W4 ? shuf_kb_stride(N / 16) / 2 : shuf_kb_stride(N / 16);
  const int wnstride = W4 ? shuf_nb_stride(KB) / 2 : shuf_nb_stride(KB);
  const int woff[2] = {rb * wnstride + lane * 16, (I / 16 + rb) * wnstride + lane * 16};
  const int wsoff[2] = {(rb * 16 + 4 * c) * 4, (I + rb * 16 + 4 * c) * 4}; // GS: the lane's four gate rows, its four up rows

  // ---- this rank's experts among the first 64 slots: lane = slot
  int le = -1;
  uint64_t peers = 0, uniq = 0;
  bool first = false;
  if (a.S <= 64) {
    if (lane < a.S) le = dec_expert(a, lane);
    const bool on = le >= 0;
    peers = __builtin_amdgcn_ballot_w64(on);
    for (int b = 0; b < a.ebits; ++b) {
      const uint64_t set = __builtin_amdgcn_ballot_w64(on && ((le >> b) & 1));
      peers &= ((le >> b) & 1) ? set : ~set;
    }
    first = on && (peers & ((1ull << lane) - 1)) == 0;
    uniq = __builtin_amdgcn_ballot_w64(first);
  }

  for (int u = blockIdx.y;; u += gridDim.y) {
    int e, cnt;
    uint64_t rest = 0; // the expert's slots not yet served (S <= 64)
    if (a.S <= 64) {
      if (u >= __builtin_popcountll(uniq)) return;
      const uint64_t at = __builtin_amdgcn_ballot_w64(first && __builtin_popcountll(uniq & ((1ull << lane) - 1)) == u);
      const int s0 = __builtin_ctzll(at);
      e = __builtin_amdgcn_readlane(le, s0);
      rest = lane_mask(peers, s0);
      cnt = __builtin_popcountll(rest);
    } else { // long batches (forced): slot u's workgroup serves the expert if it is the first slot routed to it
      if (u >= a.S) return;
      e = __builtin_amdgcn_readfirstlane(dec_expert(a, u));
      if (e < 0) continue;
      if (wave == 0) {
        int k = 0;
        for (int b = 0; b * 64 < a.S; ++b) {
          const int s = b * 64 + lane;
          const bool mine = s < a.S && dec_expert(a, s < a.S ? s : 0) == e;
          const uint64_t bal = __builtin_amdgcn_ballot_w64(mine);
          if (mine) sSlots[k + __builtin_popcountll(bal & ((1ull << lane) - 1))] = s;
          k += __builtin_popcountll(bal);
        }
        if (lane == 0) sMeta[0] = k;
      }
      __syncthreads();
      cnt = sMeta[0];
      if (sSlots[0] != u) {
        __syncthreads(); // nobody still reads the list when the next round writes it
        continue;
      }
    }

    const brsrc rW = make_rsrc(a.w1 + static_cast<int64_t>(e) * wbytes, static_cast<uint32_t>(wbytes));
    const brsrc rWs = make_rsrc(a.w1s + static_cast<int64_t>(e) * KB * N, static_cast<uint32_t>(GS ? static_cast<int64_t>(KB) * N * 4 : 0));
    v4i wbuf[RING][2][W4 ? 1 : 2];
    v4f wsc[GS ? RING : 1][2];
    auto issue = [&](int slot, int p) __attribute__((always_inline)) {
      const int kb = kb0 + (p < KBw ? p : KBw - 1);
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        if constexpr (W4) {
          wbuf[slot][g][0] = bld16<kCacheStream>(rW, woff[g], kb * wkstride);
          if constexpr (GS) // the weights' cache policy: mixed policies cost time
            wsc[slot][g] = __builtin_bit_cast(v4f, bld16<kCacheStream>(rWs, wsoff[g], kb * N * 4));
        } else {
#pragma unroll
          for (int ks = 0; ks < 2; ++ks)
            wbuf[slot][g][ks] = bld16<kCacheStream>(rW, woff[g], kb * wkstride + ks * 1024);
        }
      }
    };

    for (int chunk0 = 0; chunk0 < cnt; chunk0 += kDecTP) {
      const int nc = cnt - chunk0 < kDecTP ? cnt - chunk0 : kDecTP;
      int slot[kDecTP]; // of this pass; entries from nc on repeat the first
#pragma unroll
      for (int i = 0; i < kDecTP; ++i) {
        slot[i] = i == 0 ? 0 : slot[0];
        if (i < nc) {
          if (a.S <= 64) {
            slot[i] = __builtin_ctzll(rest);
            rest &= rest - 1;
          } else {
            slot[i] = __builtin_amdgcn_readfirstlane(sSlots[chunk0 + i]);
          }
        }
      }
      // ---- requests in the order of need: token rows, weight scales, the first weights ------------------
      if (a.M > 1) load_row(slot[0] / a.top_k, raw[0]);
#pragma unroll
      for (int i = 1; i < kDecTP; ++i) // (one token as well: several of its slots may be this expert's)
        if (i < nc) load_row(slot[i] / a.top_k, raw[i]);
      // block scales of the wave's K range: lanes 0..7 the gate rows', lanes 8..15 the up rows'; PC: the channel scales of
      // the last wave's columns, one gate and one up row per lane
      float bs_l = 0.0f, bs_u = 0.0f;
      if constexpr (PC) {
        const int64_t row = static_cast<int64_t>(e) * N + rb * 16 + ((lane >> 2) & 3) * 4 + (lane >> 4);
        bs_l = a.w1s[row];
        bs_u = a.w1s[row + I];
      } else if constexpr (!W4) {
        const int kb = (lane & 7) < KBw ? lane & 7 : 0;
        bs_l = a.w1s[(static_cast<int64_t>(e) * (N / kGroup) + ((lane >> 3) & 1) * (I / kGroup) + rb / 8) * KB + kb0 + kb];
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int p = 0; p < RING; ++p) issue(p, p);
      __builtin_amdgcn_sched_barrier(0);

      // ---- quantise this pass's token rows (the wave's K range only) into the wave's LDS tile -----
      if constexpr (PC) { // the rows' maxima over all waves first
#pragma unroll
        for (int i = 0; i < kDecTP; ++i)
          if (i < nc) {
            float amax = 0.0f, v[8];
#pragma unroll
            for (int q = 0; q < RQ; ++q) amax = fmaxf(amax, dec_widen8<DT>(raw[i][q], v)); // (a repeated group changes nothing)
            amax = wave_max64(amax);
            if (lane == 0) sMax[wave * kDecTP + i] = amax;
          }
        __syncthreads();
      }
#pragma unroll
      for (int i = 0; i < kDecTP; ++i)
        if (i < nc) {
          float row_inv = 0.0f;
          if constexpr (PC) {
            float amax = 1e-10f;
            for (int w = 0; w < W; ++w) amax = fmaxf(amax, sMax[w * kDecTP + i]);
            row_inv = 127.0f / amax;
            if (lane == 0) sAs[i * KBW] = amax / 127.0f;
          }
#pragma unroll
          for (int q = 0; q < RQ; ++q) {
            const int g = gq + 4 * q;
            if (g < KBw) {
              v2i packed;
              if constexpr (PC) {
                packed = dec_quant8_row<DT>(raw[i][q], row_inv);
              } else {
                float sc;
                packed = dec_quant8<DT, !GS>(raw[i][q], sc);
                if (sub == 0) sAs[i * KBW + g] = sc;
              }
              *reinterpret_cast<v2i *>(sA + i * pitch + g * kGroup + sub * 8) = packed;
            }
          }
        }
      __builtin_amdgcn_wave_barrier();

      // ---- one product f32(d) * a_s per K block: weights from registers, tokens from LDS; the products
      //      of the pass's tokens and the weight scales they meet go to LDS, K block by K block.  PC: the int32 sum of
      //      the wave's K range ------------------------------------------------------------------------------
      v4i dsum[2] = {v4i{0, 0, 0, 0}, v4i{0, 0, 0, 0}};
#pragma unroll
      for (int p = 0; p < KBW; ++p) {
        const int buf = p % RING;
        v4i b0 = v4i{0, 0, 0, 0}, b1 = v4i{0, 0, 0, 0};
        float as = 0.0f;
        if (n < nc && p < KBw) {
          b0 = *reinterpret_cast<const v4i *>(sA + n * pitch + p * kGroup + c * 16);
          b1 = *reinterpret_cast<const v4i *>(sA + n * pitch + p * kGroup + 64 + c * 16);
          if constexpr (!PC) as = sAs[n * KBW + p];
        }
        const float bs[2] = {lane_value(bs_l, p), lane_value(bs_l, 8 + p)};
#pragma unroll
        for (int g = 0; g < 2; ++g) {
          v4i w0, w1;
          if constexpr (W4) {
            unpack_int4(wbuf[buf][g][0], w0, w1);
          } else {
            w0 = wbuf[buf][g][0];
            w1 = wbuf[buf][g][W4 ? 0 : 1];
          }
          v4i d = PC ? dsum[g] : v4i{0, 0, 0, 0};
          d = __builtin_amdgcn_mfma_i32_16x16x64_i8(w0, b0, d, 0, 0, 0);
          d = __builtin_amdgcn_mfma_i32_16x16x64_i8(w1, b1, d, 0, 0, 0);
          if constexpr (PC) {
            dsum[g] = d;
          } else if (n < nc && p < KBw) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
              sT[((kb0 + p) * 8 + g * 4 + i) * 16 + c * kDecTP + n] = static_cast<float>(d[i]) * as;
            if constexpr (GS) { // the scales of the lane's four rows, as loaded ([c][i]; the factor 1/16 is applied by the reader)
              if (n == 0) *reinterpret_cast<v4f *>(sB + ((kb0 + p) * 2 + g) * 16 + c * 4) = wsc[GS ? buf : 0][g];
            } else {
              if (lane == 0) sB[(kb0 + p) * 2 + g] = bs[g];
            }
          }
        }
        if (p + RING < KBW) {
          __builtin_amdgcn_sched_barrier(0);
          issue(buf, p + RING);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      if constexpr (PC) {
        if (n < nc)
#pragma unroll
          for (int g = 0; g < 2; ++g)
#pragma unroll
            for (int i = 0; i < 4; ++i) sTi[(wave * 8 + g * 4 + i) * 16 + c * kDecTP + n] = dsum[g][i];
      }
      __syncthreads();

      // ---- the sum over K in K order, then the gated activation (SiLU of bf16 rows computed, not looked up: a table
      //      entry would be one more dependent round trip).  Lane (i, c, token) of the last wave adds the gate terms
      //      and the up terms of activation column 4c + i. ---------------------------------------------
      if (wave == W - 1) {
        float accg = 0.0f, accu = 0.0f;
        const int i = lane >> 4, cc = (lane >> 2) & 3, tok = lane & 3;
        const int64_t fslot = tok == 0 ? slot[0] : tok == 1 ? slot[1] : tok == 2 ? slot[2] : slot[3];
        const float wgt = a.mul_on_input ? a.topk_w[fslot] : 1.0f;
        if constexpr (PC) {
          int32_t dg = 0, du = 0;
          for (int w = 0; w < W; ++w) {
            dg += sTi[w * 128 + lane];
            du += sTi[w * 128 + 64 + lane];
          }
          // every wave knows the token's scale; int8: (f32(d) * ts) * b_s with ts = w * a_s (moe_w8a8.cu:452), packed int4 left
          // to right: routed weight, token scale, channel scale (w4a8.py:386-395).  A weight of one changes nothing.
          const float as = sAs[tok * KBW];
          accg = static_cast<float>(dg);
          accu = static_cast<float>(du);
          if constexpr (W4) {
            accg = ((accg * wgt) * as) * bs_l;
            accu = ((accu * wgt) * as) * bs_u;
          } else {
            const float ts = wgt * as;
            accg = (accg * ts) * bs_l;
            accu = (accu * ts) * bs_u;
          }
        } else {
          auto sum_k = [&](auto CONTRACT) __attribute__((always_inline)) {
            auto add = [](float acc, float t, float b) __attribute__((always_inline)) {
              if constexpr (W4) b = b * 0.0625f; // int4 nibbles are unpacked 16 times too large
              if constexpr (decltype(CONTRACT)::value) return __builtin_fmaf(t, b, acc);
              const float tb = t * b;
              return acc + tb;
            };
            // lane (i, c, token): row 4c + i of the fragment
            const int brow = cc * 4 + i;
            const float *const bg = sB + (W4 ? brow : 0), *const bu = sB + (W4 ? 16 + brow : 1);
            int kb = 0;
            for (; kb + 4 <= KB; kb += 4) {
              float tg[4], tu[4], sg[4], su[4];
#pragma unroll
              for (int j = 0; j < 4; ++j) {
                tg[j] = sT[(kb + j) * 128 + lane];
                tu[j] = sT[(kb + j) * 128 + 64 + lane];
                sg[j] = bg[(kb + j) * SB];
                su[j] = bu[(kb + j) * SB];
              }
#pragma unroll
              for (int j = 0; j < 4; ++j) {
                accg = add(accg, tg[j], sg[j]);
                accu = add(accu, tu[j], su[j]);
              }
            }
            for (; kb < KB; ++kb) {
              accg = add(accg, sT[kb * 128 + lane], bg[kb * SB]);
              accu = add(accu, sT[kb * 128 + 64 + lane], bu[kb * SB]);
            }
          };
          if (a.contract) sum_k(std::true_type{});
          else sum_k(std::false_type{});
          accg = accg * wgt;
          accu = accu * wgt;
        }
        if (tok < nc) {
          const uint16_t g16 = from_f32<DT>(accg), u16 = from_f32<DT>(accu);
          uint16_t o;
          if (a.table) o = act_mul_tab<DT>(a.table, g16, u16);
          else o = silu_mul<DT>(g16, u16);
          a.act[fslot * I + rb * 16 + 4 * cc + i] = o;
        }
      }
      __syncthreads(); // the products' LDS (and the slot list) is free again
    }
  }
}

// Four waves per SIMD (two workgroups of eight waves per compute unit, one streaming while the other starts or sums).
template <int KBW, bool W4, bool PC, int DT>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4, 4))) void dec_gemm1_kernel(const DecArgs a) {
  dec_gemm1_body<KBW, W4, PC, DT>(a);
}

template <int PD, int RAWN, bool W4, bool PC, int DT> // weight K blocks in flight per wave; 16-byte pieces of the activation row per lane
__global__ __launch_bounds__(512) void dec_gemm2_kernel(const DecArgs a) {
  extern __shared__ __attribute__((aligned(16))) int8_t smem[];
  constexpr bool GS = W4 && !PC;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int W = blockDim.x >> 6;
  const int n = lane & 15, c = lane >> 4;
  const int t = blockIdx.y, nrb = a.nrb2;
  const int H = a.H, I = a.I, KB = I / kGroup, k = a.top_k;

  uint16_t *const sC = reinterpret_cast<uint16_t *>(smem);                     // [nrb][k][16] per-slot output values
  const int head = (nrb * k * 16 * 2 + 15) & ~15;
  float *const sAs = reinterpret_cast<float *>(smem + head) + wave * KB;       // [KB] of this wave
  int8_t *const sA = smem + head + ((W * KB * 4 + 15) & ~15) + wave * I;       // [I] of this wave

  const int sub = lane & 15, gq = lane >> 4;
  v8u16 raw[RAWN];
  auto load_act = [&](int s) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < RAWN; ++q) {
      const int g = gq + 4 * q;
      raw[q] = *reinterpret_cast<const v8u16 *>(a.act + static_cast<int64_t>(s) * I + (g < KB ? g : 0) * kGroup + sub * 8);
    }
  };
  // Where every expert is on this rank, piece it of the workgroup's work is slot it % k: its activation row does not
  // wait for the routing.
  const bool all_here = a.expert_map == nullptr;
  float wgt = 1.0f;
  if (all_here) {
    load_act(t * k + wave % k);
    wgt = a.topk_w[t * k + wave % k];
  }
  // lane j: the expert of the token's slot j
  const int le = lane < k ? dec_expert(a, t * k + lane) : -1;
  const uint64_t here = __builtin_amdgcn_ballot_w64(le >= 0);
  const int nloc = all_here ? k : __builtin_popcountll(here);
  for (int it = wave; it < nloc * nrb; it += W) {
    const int rbi = it / nloc, jj = it - rbi * nloc;
    int j = jj;
    if (!all_here) { // the jj-th set bit
      const uint64_t at = __builtin_amdgcn_ballot_w64(le >= 0 && __builtin_popcountll(here & ((1ull << lane) - 1)) == jj);
      j = __builtin_ctzll(at);
    }
    const int rb = blockIdx.x * nrb + rbi;
    const int s = t * k + j;
    const int e = __builtin_amdgcn_readlane(le, j);
    if (e < 0) continue; // (its activation row was never written: nothing of it is used)
    if (!all_here || it != wave) {
      load_act(s);
      wgt = a.topk_w[s];
    }
    if (a.mul_on_input) wgt = 1.0f;

    const int64_t wbytes = W4 ? static_cast<int64_t>(H) * I / 2 : static_cast<int64_t>(H) * I;
    const brsrc rW = make_rsrc(a.w2 + static_cast<int64_t>(e) * wbytes, static_cast<uint32_t>(wbytes));
    const brsrc rWs = make_rsrc(a.w2s + static_cast<int64_t>(e) * KB * H, static_cast<uint32_t>(GS ? static_cast<int64_t>(KB) * H * 4 : 0));
    const int wkstride = W4 ? shuf_kb_stride(H / 16) / 2 : shuf_kb_stride(H / 16);
    const int woff = rb * (W4 ? shuf_nb_stride(KB) / 2 : shuf_nb_stride(KB)) + lane * 16;
    const int wsoff = (rb * 16 + 4 * c) * 4; // GS: the scales of the lane's four rows
    // what is needed last of the small loads goes out before the weights all the same (they return in order)
    float bs_l = 0.0f;  // lane l: the block scale of K block l
    v4f bs_pc = v4f{0.f, 0.f, 0.f, 0.f}; // PC: the channel scales of the lane's four rows
    if constexpr (PC) bs_pc = *reinterpret_cast<const v4f *>(a.w2s + static_cast<int64_t>(e) * H + rb * 16 + 4 * c);
    else if constexpr (!W4) bs_l = a.w2s[(static_cast<int64_t>(e) * (H / kGroup) + rb / 8) * KB + (lane < KB ? lane : 0)];
    v4i wbuf[PD][W4 ? 1 : 2];
    v4f wsc[GS ? PD : 1];
    auto issue = [&](int p, int kb) __attribute__((always_inline)) {
      kb = kb < KB ? kb : KB - 1;
      if constexpr (W4) {
        wbuf[p][0] = bld16<kCacheStream>(rW, woff, kb * wkstride);
        if constexpr (GS) wsc[p] = __builtin_bit_cast(v4f, bld16<kCacheStream>(rWs, wsoff, kb * H * 4));
      } else {
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) wbuf[p][ks] = bld16<kCacheStream>(rW, woff, kb * wkstride + ks * 1024);
      }
    };
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int p = 0; p < PD; ++p) issue(p, p);
    __builtin_amdgcn_sched_barrier(0);

    // the activation row, re-quantised, into the wave's LDS row
    float row_as = 0.0f;
    if constexpr (PC) {
      float amax = 0.0f, v[8];
#pragma unroll
      for (int q = 0; q < RAWN; ++q) amax = fmaxf(amax, dec_widen8<DT>(raw[q], v));
      amax = wave_max64(amax);
      if (a.floor2) amax = fmaxf(amax, 1e-10f);
      const float inv = amax == 0.0f ? 0.0f : 127.0f / amax;
      row_as = amax / 127.0f;
#pragma unroll
      for (int q = 0; q < RAWN; ++q) {
        const int gi = gq + 4 * q;
        if (gi < KB) *reinterpret_cast<v2i *>(sA + gi * kGroup + sub * 8) = dec_quant8_row<DT>(raw[q], inv);
      }
    } else {
#pragma unroll
      for (int q = 0; q < RAWN; ++q) {
        const int gi = gq + 4 * q;
        if (gi < KB) {
          float sc;
          const v2i packed = dec_quant8<DT>(raw[q], sc);
          *reinterpret_cast<v2i *>(sA + gi * kGroup + sub * 8) = packed;
          if (sub == 0) sAs[gi] = sc;
        }
      }
    }
    __builtin_amdgcn_wave_barrier();

    v4f acc = v4f{0.f, 0.f, 0.f, 0.f};
    v4i dsum = v4i{0, 0, 0, 0};
    auto step = [&](int p, int kb) __attribute__((always_inline)) {
      // every column of the token operand is the same row: all lanes end up with valid sums
      const v4i b0 = *reinterpret_cast<const v4i *>(sA + kb * kGroup + c * 16);
      const v4i b1 = *reinterpret_cast<const v4i *>(sA + kb * kGroup + 64 + c * 16);
      v4i w0, w1;
      if constexpr (W4) {
        unpack_int4(wbuf[p][0], w0, w1);
      } else {
        w0 = wbuf[p][0];
        w1 = wbuf[p][W4 ? 0 : 1];
      }
      v4i d = PC ? dsum : v4i{0, 0, 0, 0};
      d = __builtin_amdgcn_mfma_i32_16x16x64_i8(w0, b0, d, 0, 0, 0);
      d = __builtin_amdgcn_mfma_i32_16x16x64_i8(w1, b1, d, 0, 0, 0);
      if constexpr (PC) {
        dsum = d;
        return;
      }
      const float as = sAs[kb], bs = lane_value(bs_l, kb);
      v4f bs4 = v4f{0.f, 0.f, 0.f, 0.f};
      if constexpr (GS) bs4 = wsc[GS ? p : 0] * 0.0625f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float tt = static_cast<float>(d[i]) * as;
        if (a.contract) {
          acc[i] = __builtin_fmaf(tt, GS ? bs4[i] : bs, acc[i]);
        } else {
          tt = tt * (GS ? bs4[i] : bs);
          acc[i] = acc[i] + tt;
        }
      }
    };
    // (all but the last PD steps refill the ring: no branch around a load, so that each wait counts exactly what is behind it)
    int kb = 0;
    for (; kb + PD < KB; kb += PD) {
#pragma unroll
      for (int p = 0; p < PD; ++p) {
        step(p, kb + p);
        __builtin_amdgcn_sched_barrier(0);
        issue(p, kb + PD + p);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int p = 0; p < PD; ++p)
      if (kb + p < KB) step(p, kb + p);
    if (n == 0) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float v;
        if constexpr (PC) {
          v = static_cast<float>(dsum[i]);
          if constexpr (W4) v = ((v * wgt) * row_as) * bs_pc[i];
          else v = (v * (wgt * row_as)) * bs_pc[i];
        } else {
          v = acc[i] * wgt;
        }
        sC[(rbi * k + j) * 16 + 4 * c + i] = from_f32<DT>(v);
      }
    }
    __builtin_amdgcn_wave_barrier(); // the next piece of this wave reuses the LDS row
  }
  __syncthreads();

  // ---- the token's slots in slot order, the slots of other ranks left out ------------------------
  if (tid < 16 * nrb) {
    const int rbi = tid >> 4, col = tid & 15;
    float acc = 0.0f;
    for (int j = 0; j < k; ++j)
      if ((here >> j) & 1) acc = acc + to_f32<DT>(sC[(rbi * k + j) * 16 + col]);
    const int64_t o = static_cast<int64_t>(t) * H + (blockIdx.x * nrb + rbi) * 16 + col;
    uint16_t r;
    if (a.shared) {
      uint16_t xv = from_f32<DT>(acc);
      xv = from_f32<DT>(to_f32<DT>(xv) * a.factor);
      r = from_f32<DT>(to_f32<DT>(xv) + to_f32<DT>(a.shared[o]));
    } else {
      r = from_f32<DT>(acc * a.factor);
    }
    a.out[o] = r;
  }
}

// K split of the first kernel: waves per workgroup such that each holds at most kDecMaxKBw K
// blocks, preferring four or more blocks per wave.  0: no admissible split.
static int pick_waves(int KB) {
  int fallback = 0;
  for (int w = 8; w >= 1; w >>= 1) {
    if (KB % w || KB / w > kDecMaxKBw) continue;
    if (KB / w >= 4) return w;
    fallback = w; // fewer than four blocks per wave: take the smallest such split
  }
  return fallback;
}

// Largest number of routed slots the two-launch path is taken for.  Its second kernel reads an
// expert's weights once per slot, so it pays while slots rarely share an expert.
static int decode_max_slots() {
  static const int v = [] {
    const char *s = std::getenv("LIGHTOP_AMD_DECODE_MAX_SLOTS");
    if (!s || !*s) return -1;
    const long x = std::strtol(s, nullptr, 10);
    return static_cast<int>(x < 0 ? 0 : (x > kDecMaxSlots ? kDecMaxSlots : x));
  }();
  return v;
}

// Column pieces per workgroup of the second kernel, and the dynamic LDS of both kernels.
static int decode_path_nrb2(const DecProblem &d, int W2) {
  // A rank that holds a fraction of the experts serves that fraction of a token's slots: its workgroups of the second kernel
  // take as many more 16-column pieces, so that their waves have work, while the grid still covers the chip (one token of
  // a 32/256 rank, 7168 wide: 10.0 us with one piece, 15.7 with eight; four tokens: 27.1 with one, 19.8 with eight).
  int nrb2 = 1;
  while (nrb2 < 8 && static_cast<int64_t>(nrb2) * 2 * d.E <= d.num_experts && d.H / 16 * d.M / (2 * nrb2) >= 384) nrb2 *= 2;
  while (nrb2 * 16 > 64 * W2) nrb2 /= 2;
  return nrb2;
}
static void decode_path_lds(const DecProblem &d, bool w4, size_t *l1, size_t *l2) {
  const int64_t S = d.M * d.top_k;
  const size_t KB1 = static_cast<size_t>(d.H / kGroup), KB2 = static_cast<size_t>(d.I / kGroup);
  int w1, w2;
  decode_path_waves(d.top_k, d.H, &w1, &w2);
  const size_t W1 = static_cast<size_t>(w1), W2 = static_cast<size_t>(w2);
  const size_t list = S > 64 ? static_cast<size_t>((S + 3) & ~int64_t(3)) * 4 : 0;
  *l1 = (d.channel ? W1 * 512 : KB1 * (128 + (w4 ? 32 : 2)) * 4) + W1 * kDecTP * 4 + list + 16 +
        W1 * kDecTP * kDecMaxKBw * 4 + W1 * kDecTP * (KB1 / W1 * kGroup + 16);
  *l2 = ((static_cast<size_t>(decode_path_nrb2(d, w2)) * d.top_k * 32 + 15) & ~size_t(15)) +
        ((W2 * KB2 * 4 + 15) & ~size_t(15)) + W2 * static_cast<size_t>(d.I);
}

bool decode_path_applies(const DecProblem &d, int flags) {
  const bool w4 = (flags & LO_GEMM_W4) != 0;
  const int64_t S = d.M * d.top_k;
  if (d.dtype != LO_BF16 && d.dtype != LO_F16) return false;
  if (d.M < 1 || S > kDecMaxSlots || d.top_k > 64) return false;
  if (d.H % kGroup || d.I % kGroup || 2 * d.I * d.H >= (1ll << 31)) return false;
  // the activations [S, I] live in the caller's buffer: [S, max(2I, H)], or [S, H] for bf16 rows with SiLU in the block form
  if (!d.channel && !(flags & LO_FUSED_ACT_GELU) && d.dtype == LO_BF16 && d.I > d.H) return false;
  if (d.I / kGroup > kDecMaxKB2 || pick_waves(static_cast<int>(d.H / kGroup)) == 0) return false;
  size_t l1, l2;
  decode_path_lds(d, w4, &l1, &l2);
  if (l1 > 64 * 1024 || l2 > 64 * 1024) return false;
  if (flags & LO_FUSED_FORCE_DECODE_PATH) return true;
  const int forced = decode_max_slots();
  if (forced >= 0) return S <= forced;
  // Where the two launches and the staged path with its weight-streaming kernels cross (us, two launches / staged):
  // int8, at most four K blocks per wave: Qwen3 30B 57.6 / 69.5 and 235B 190 / 190 at 64 slots;
  // int8, longer K: DeepSeek-V3's 32-expert share 72 / 82 at 4 tokens and 96 / 90 at 8, all 256 experts 81 / 87 at 1 token and
  // 120 / 113 at 2, so what counts are the slots on this rank;
  // int4, per-channel scales: 70 / 72 at 32 slots and 122 / 108 at 64;
  // int4, K groups: experts of 2048 x 768 20 / 32 at 16 slots, 4096 x 768 28 / 39, 4096 x 1536 40 / 43 at 12 and 48 / 44 at 16,
  // 4096 x 3584 65 / 51 at 14; with fp16 rows or GELU, whose staged path has a launch more, 4096 x 1536 48 / 48 at 16.
  if (w4 && d.channel) return S <= 32;
  if (w4) {
    const bool large = d.H * d.I >= 4096ll * 1536, fused_stage = d.dtype == LO_BF16 && !(flags & LO_FUSED_ACT_GELU);
    return S <= (large && fused_stage ? 12 : 16);
  }
  const int KB = static_cast<int>(d.H / kGroup);
  if (KB / pick_waves(KB) <= 4) return S <= 64;
  return S <= 32 && S * d.E <= static_cast<int64_t>(8) * d.num_experts;
}

void decode_path_waves(int32_t top_k, int64_t H, int *gemm1_waves, int *gemm2_waves) {
  *gemm1_waves = pick_waves(static_cast<int>(H / kGroup));
  *gemm2_waves = top_k < 8 ? top_k : 8;
}

// Whole path in two launches; LO_ENOTSUP when the problem is not a decode-size one this file serves.
int launch_decode_path(const DecProblem &d, int flags, hipStream_t stream) {
  const bool w4 = (flags & LO_GEMM_W4) != 0, gelu = (flags & LO_FUSED_ACT_GELU) != 0;
  if (!decode_path_applies(d, flags)) return LO_ENOTSUP;
  const int64_t S = d.M * d.top_k;
  const int KB1 = static_cast<int>(d.H / kGroup), KB2 = static_cast<int>(d.I / kGroup);
  int W1, W2;
  decode_path_waves(d.top_k, d.H, &W1, &W2);

  DecArgs a{};
  a.x = static_cast<const uint16_t *>(d.x);
  a.ids = d.topk_ids; a.ids64 = d.ids_dtype == LO_I64; a.expert_map = d.expert_map; a.topk_w = d.topk_w;
  a.w1 = d.w1; a.w2 = d.w2; a.w1s = d.w1s; a.w2s = d.w2s;
  a.shared = static_cast<const uint16_t *>(d.shared_output);
  a.act = static_cast<uint16_t *>(d.act); a.out = static_cast<uint16_t *>(d.out);
  a.factor = d.factor;
  a.M = static_cast<int>(d.M); a.S = static_cast<int>(S); a.top_k = d.top_k; a.E = d.E; a.Eg = d.num_experts;
  a.H = static_cast<int>(d.H); a.I = static_cast<int>(d.I); a.kbw = KB1 / W1;
  a.mul_on_input = d.mul_on_input ? 1 : 0;
  a.floor2 = gelu ? 1 : 0;
  while ((1 << a.ebits) < d.E) ++a.ebits;
  // two orders only: LO_GEMM_FUSED_SCALE buys nothing at this size and gets the default order
  a.contract = scale_order(flags) == kOrdSeparate ? 0 : 1;
  if (gelu) {
    const int rc = act_table(stream, LO_ACT_GELU, d.dtype, &a.table);
    if (rc) return rc;
  }
  a.nrb2 = decode_path_nrb2(d, W2);
  // workgroups along the distinct experts: what the batch can hit here, some to spare; more are served in rounds
  int64_t hits = S;
  if (S <= 64) {
    const int64_t expect = (S * d.E + d.num_experts - 1) / d.num_experts;
    hits = expect + expect / 2 + 1;
    hits = hits < S ? hits : S;
    hits = hits < d.E ? hits : d.E;
  }

  size_t l1, l2;
  decode_path_lds(d, w4, &l1, &l2);
  const dim3 g1(static_cast<unsigned>(d.I / 16), static_cast<unsigned>(hits));
  const dim3 g2(static_cast<unsigned>(d.H / 16 / a.nrb2), static_cast<unsigned>(d.M));
#define LO_DEC_LAUNCH(W4V, PCV, DTV)                                                                             \
  do {                                                                                                           \
    if (a.kbw <= 4) hipLaunchKernelGGL((dec_gemm1_kernel<4, W4V, PCV, DTV>), g1, dim3(64 * W1), l1, stream, a);  \
    else hipLaunchKernelGGL((dec_gemm1_kernel<kDecMaxKBw, W4V, PCV, DTV>), g1, dim3(64 * W1), l1, stream, a);    \
    const int rc = check_launch("fused_experts(decode, gemm1)");                                                 \
    if (rc) return rc;                                                                                           \
    if (KB2 <= 6) hipLaunchKernelGGL((dec_gemm2_kernel<6, 2, W4V, PCV, DTV>), g2, dim3(64 * W2), l2, stream, a); \
    else if (KB2 <= 8) hipLaunchKernelGGL((dec_gemm2_kernel<8, 2, W4V, PCV, DTV>), g2, dim3(64 * W2), l2, stream, a); \
    else if (KB2 <= 16) hipLaunchKernelGGL((dec_gemm2_kernel<8, 4, W4V, PCV, DTV>), g2, dim3(64 * W2), l2, stream, a); \
    else hipLaunchKernelGGL((dec_gemm2_kernel<8, 8, W4V, PCV, DTV>), g2, dim3(64 * W2), l2, stream, a);          \
  } while (0)
#define LO_DEC_DTYPE(W4V, PCV)                                    \
  do {                                                            \
    if (d.dtype == LO_F16) LO_DEC_LAUNCH(W4V, PCV, LO_F16);       \
    else LO_DEC_LAUNCH(W4V, PCV, LO_BF16);                        \
  } while (0)
  if (d.channel) {
    if (w4) LO_DEC_DTYPE(true, true);
    else LO_DEC_DTYPE(false, true);
  } else if (w4) LO_DEC_DTYPE(true, false);
  else LO_DEC_DTYPE(false, false);
#undef LO_DEC_DTYPE
#undef LO_DEC_LAUNCH
  return check_launch("fused_experts(decode, gemm2)");
}

} // namespace lo
