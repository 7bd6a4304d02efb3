// The grouped GEMMs of DeepSeek's prefill MoE (dsk::moe_prefill, ds41f-4xgx10-switchless/engine/kernels/dsk.h:268-295;
// arithmetic engine/kernels/moe.cu:519-534, 974-981 and ref/inference/model.py:841-851): MXFP4 routed experts and the FP8
// shared expert against rows given as act_quant(x) (e4m3 with a ue8m0 scale per 32 values), on gfx950's block-scaled
// matrix instruction v_mfma_scale_f32_16x16x128_f8f6f4: a lane holds 32 k of one row of each operand and ONE E8M0 scale
// byte, the instruction scales every 32 consecutive k - exactly the formats' scale group - so weights (e2m1 or e4m3),
// activations and both scale tensors go to the instruction as stored - no conversion, no scaled adds on the vector unit -
// and the accumulators run through K inside the matrix unit.
//
// The tiling, the LDS staging by global_load_lds (lane-permuted sources so that the fragment reads are conflict-free),
// the hand-counted waits and the workgroup -> (tile, row group) map are those of pf_gemm_fp8.cuh; what differs:
//   * a weight row of a 128-k block is 64 bytes (e2m1) - four lanes a row, piece q of row r at slot q ^ sw4(r) -, or 128 of two blocks;
//   * the scales come in words of four blocks' bytes a weight row and a position, read back a word a lane;
//   * UP's epilogue is DeepSeek's: gate, up rounded to bf16, up clamped to +-limit and gate from above, silu(gate) * up
//     times the position's routing weight (none for the shared expert), rounded to bf16, then quantised per 32 channels
//     (ue8m0) for the down projection; DOWN rounds each position's outputs to bf16 (the reference's per-pick rounding).
#pragma once
#include "pf_gemm_fp8.cuh"

namespace dsgx {
namespace pfmx {

using pf8::dma16;
using pf8::dma4;
using pf8::kThreads;
using pf8::kWgRows;
using pf8::sw4;
using pf8::swz;
using pf8::v4f_t;
using pf8::v8i_t;
using pf8::wait_loads;

// A tile's shape by its positions (64, 128 or 256) and its weights' format. What a turn waits for is the way of its operands into
// LDS, and there the lines that a load instruction names count as much as its bytes (hidden 5120, intermediate 2304, 256
// experts of 32 rows each, gate/up 895 us before):
//   * a scale word of 4 bytes a row and block named 32 lines for 128 bytes; e2m1 experts' scale words therefore come for four
//     blocks at a time, 16 bytes a row, into two buffers of their own (with no scale loads at all 640 us, with those a
//     block 729 with coalesced stand-ins); e4m3 rows share a word by 32 and keep theirs with the block;
//   * half a line a weight row and block (e2m1: 64 bytes) named every line twice: tiles of up to 64 positions, whose weights are
//     most of their bytes, take two blocks a turn and whole lines (the larger shapes: 2% at 192 rows an expert, and LDS holds
//     three stages of one block only).
// Together 895 -> 693 us; the whole call at T = 3000 (Zipf) 1777 -> 1546, at T = 300 1115 -> 878. Four to eight stages instead of
// three return nothing, two cost 15%.
template <int POS, int WF>
struct Shape {
  static constexpr bool F4 = WF == DSGX_FMT_MXFP4_G32;
  static constexpr int WP = POS == 256 ? 2 : 1;     // position groups of waves
  static constexpr int kPos = POS, kSub = POS / 16, WR = 8 / WP, RA = 2 * WP;
  static constexpr int TB = F4 && POS <= 64 ? 2 : 1;  // 128-k blocks a turn
  static constexpr int kRowB = F4 ? 64 * TB : 128;  // bytes of a weight row in a turn
  static constexpr int kStageW = kWgRows * kRowB;
  static constexpr int kStageX = kPos * 128;        // one block's activations
  static constexpr int kStageBytes = kStageW + TB * kStageX;
  static constexpr int kWords = F4 ? 4 : 1;         // blocks whose scale words come together
  static constexpr int kGroupW = kWgRows * 4 * kWords, kGroupX = kPos * 4 * kWords;  // their scale words: the weight rows', the positions'
  static constexpr int kGroup = kGroupW + kGroupX, kGroups = F4 ? 2 : 3;  // (e4m3: a buffer a stage)
  static constexpr int kStages = 3 * kStageBytes + kGroups * kGroup <= 160 * 1024 ? 3 : 2;
  static constexpr int kLoadsW = kRowB == 64 ? 2 : 4;       // a wave's loads a turn: its two weight tiles ...
  static constexpr int kHalfX = kPos / 64;                  // ... and its half tiles of eight positions, a load a block
  static constexpr int kLoads = kLoadsW + TB * kHalfX + (F4 ? 0 : 2);  // (e4m3: and its two loads of scale words)
  static constexpr int kLds = kStages * kStageBytes + kGroups * kGroup;  // (the epilogues reuse it: UP kPos x 256 B, DOWN 8 x 2 WP KiB)
};

// The shared expert's side of a launch that holds its tiles too (k_gemm_mixed): the first `grid` workgroups are theirs
struct SharedRows {
  unsigned grid;
  const uint8_t *aq, *as, *wa, *sa, *wb, *sb;
  uint16_t* h;
  uint8_t *hq, *hs;
  uint16_t* d;
};
struct Args {
  const uint8_t* aq;   // activations, e4m3 [rows][K]
  const uint8_t* as;   // their ue8m0 scales [rows][K / 32]
  const int* gather;   // position -> activation row (null: the position itself)
  const int* tile_e;   // the tile list (null: the shared expert on rows [0, nrows))
  const int* tile_m0;
  const int* ntiles;
  const int* off;
  int nrows;
  int H, I;
  const uint8_t *wa, *sa, *wb, *sb;  // UP: gate (w1), up (w3); DOWN: w2 in wa / sa. Expert e at + e * wstride / sstride.
  size_t wstride, sstride;
  const float* posw;   // UP, routed: the positions' routing weights (null: the shared expert, no weight)
  float limit;
  uint16_t* h;         // UP: h bf16 [position][I] (before its quantisation)
  uint8_t* hq;         // UP: h as e4m3 [position][I]
  uint8_t* hs;         // UP: its ue8m0 scales [position][I / 32]
  uint16_t* d;         // DOWN: bf16 [position][H]
  SharedRows sh;       // (grid 0: the launch holds routed tiles only)
};

// 128-byte rows (activations, e4m3 weights) lie in LDS in pf_gemm_fp8.cuh's layout, whose fragment reads (a lane's two
// neighbouring slots 2 part, 2 part + 1, swizzled by row) run without bank conflicts; what differs is WHICH 16 bytes of the
// row a slot holds: the block-scaled instruction wants bytes 16 part ... and 64 + 16 part ... in a lane, so logical piece
// x holds the row's piece x / 2 + 4 (x % 2). (Reading pieces part and 4 + part of rows stored in natural order instead
// costs every second LDS cycle to bank conflicts - measured.)
__device__ __forceinline__ int pc8(int x) { return (x >> 1) + 4 * (x & 1); }

template <int CBSZ>
__device__ __forceinline__ v4f_t mfma_mx(v8i_t a, v8i_t b, v4f_t c, int sa, int sb) {
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, c, CBSZ, 0, 0, sa, 0, sb);
}

template <bool UP, int POS, int WF>
__device__ __forceinline__ void gemm_tile(const Args& g, uint8_t* smem, int e, int m0, int mend, int ns) {
  using S = Shape<POS, WF>;
  constexpr bool F4 = S::F4;
  constexpr int WP = S::WP, kPosWave = S::kPos / 8;
  constexpr int CBSZ = F4 ? 4 : 0;
  const int K = UP ? g.H : g.I, KB = K / 128, G = K / 32;
  if (mend > m0 + S::kPos) mend = m0 + S::kPos;
  const size_t eo = e < 0 ? 0 : (size_t)e;
  const uint8_t *wa = g.wa + eo * g.wstride, *sa = g.sa + eo * g.sstride;
  const uint8_t *wb = UP ? g.wb + eo * g.wstride : wa, *sb = UP ? g.sb + eo * g.sstride : sa;
  const int tid = threadIdx.x, lane = tid & 63, wave = uni(tid >> 6), r16 = lane & 15, part = lane >> 4;
  const int rg = wave % S::WR, pg = wave / S::WR;
  const int c0 = ns * (kWgRows / 2), r0 = ns * kWgRows;
  auto tile_row = [&](int i, const uint8_t*& wbase, const uint8_t*& sbase) {  // first weight row of 16-row tile i, its tensors
    if (UP) {
      wbase = (i & 1) ? wb : wa, sbase = (i & 1) ? sb : sa;
      return c0 + 16 * (i >> 1);
    }
    wbase = wa, sbase = sa;
    return r0 + 16 * i;
  };
  const int nmt = uni(min(S::kSub, (mend - m0 + 15) / 16));
  const int nj = uni(nmt > pg ? (nmt - pg + WP - 1) / WP : 0);
  // ---- what this lane fetches ----
  // weights: the wave brings tiles 2 wave, 2 wave + 1. 64-byte rows: one instruction a tile, lane -> row lane / 4, piece
  // (lane % 4) ^ sw4(row); 128-byte rows: two instructions a tile (rows 0-7, 8-15), lane -> row lane / 8, piece (lane % 8) ^
  // swz(row) (e4m3) or (lane % 8) ^ (row % 8) (two blocks of e2m1, whose lanes read pieces part and 4 + part)
  const uint8_t* pw[2][2];
  const uint8_t* pws;  // lanes 0-31: the scale words of row lane % 16 of tile 2 wave + lane / 16
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const uint8_t *wbase, *sbase;
    const int row = tile_row(2 * wave + t, wbase, sbase);
    if (S::kRowB == 64) {
      const int r = lane >> 2;
      pw[t][0] = wbase + (size_t)(row + r) * (K / 2) + 16 * ((lane & 3) ^ sw4(r));
      pw[t][1] = pw[t][0];
    } else {
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) {
        const int r = 8 * hh + (lane >> 3);
        pw[t][hh] = F4 ? wbase + (size_t)(row + r) * (K / 2) + 16 * ((lane & 7) ^ (r & 7)) : wbase + (size_t)(row + r) * K + 16 * pc8((lane & 7) ^ swz(r));
      }
    }
    if (((lane >> 4) & 1) == t) pws = sbase + (size_t)(F4 ? row + r16 : (row + r16) / 32) * G;
  }
  // activations: half tile kHalfX wave + i is positions 8 (kHalfX wave + i) ...; a wave whose half tiles hold no rows brings none
  const bool brings_x = POS > 64 || m0 + 8 * wave < mend;
  auto row_of = [&](int p) {  // the activation row of the tile's position p (a ragged tile re-reads its last row: never stored)
    const int pos = min(m0 + p, mend - 1);
    return (size_t)(g.gather ? g.gather[pos] : pos);
  };
  const uint8_t* px[S::kHalfX];
#pragma unroll
  for (int i = 0; i < S::kHalfX; ++i) {
    const int p = 8 * (S::kHalfX * wave + i) + (lane >> 3);
    px[i] = g.aq + row_of(p) * K + 16 * pc8((lane & 7) ^ swz(p & 15));
  }
  const uint8_t* pxs = g.as + row_of(kPosWave * wave + (lane & (kPosWave - 1))) * G;  // lanes 0 .. kPosWave - 1: the scale words of the wave's positions
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem;
  constexpr int kGroups0 = S::kStages * S::kStageBytes;  // the groups' scale words behind the stages
  // load number i (0 .. kLoads - 1) of turn t: the activations (L2 hits mostly), the weights last: a wave's loads return in
  // issue order, so a load that waits for HBM holds back every later one of its wave and the cache's miss slots with them
  // (weights first: 7% slower, measured). A turn issues them one at a time between its MFMAs (issue_some), so that the
  // texture unit works through a block's 50 KB while the matrix unit runs instead of in front of it: issued together after
  // the barrier they cost every wave the time the unit takes to accept them all (measured: a third of a turn).
  const int TN = KB / S::TB;
  constexpr int kFirst = F4 ? 0 : 2;  // (e4m3: the turn's scale words in front; 32 weight rows share a word, so they name few lines)
  auto issue_one = [&](int t, int i) {
    const int tc = t < TN ? t : TN - 1;  // (past the end: the last turn again, into a stage nobody reads)
    const uint32_t st = lds0 + (uint32_t)(t % S::kStages) * S::kStageBytes;
    const uint32_t wbase = st + (uint32_t)wave * (2 * 16 * S::kRowB), xbase = st + S::kStageW + (uint32_t)wave * (S::kHalfX * 1024);
    if (i < kFirst) {
      const uint32_t at = lds0 + kGroups0 + (uint32_t)(t % S::kStages) * S::kGroup;
      if (i == 0) {
        if (brings_x && lane < kPosWave) dma4(reinterpret_cast<const float*>(pxs + 4 * tc), uni(at + S::kGroupW + (uint32_t)wave * (4 * kPosWave)));
      } else {
        if (lane < 32) dma4(reinterpret_cast<const float*>(pws + 4 * tc), uni(at + (uint32_t)wave * 128));
      }
    } else if (i < kFirst + S::TB * S::kHalfX) {
      const int b = (i - kFirst) / S::kHalfX, q = (i - kFirst) % S::kHalfX;
      if (brings_x) dma16(px[q] + (size_t)tc * (128 * S::TB) + 128 * b, uni(xbase + b * S::kStageX + q * 1024));
    } else {
      const int q = i - kFirst - S::TB * S::kHalfX;
      if (S::kRowB == 64) dma16(pw[q][0] + (size_t)tc * 64, uni(wbase + q * 1024));
      else dma16(pw[q >> 1][q & 1] + (size_t)tc * 128, uni(wbase + (q >> 1) * 2048 + (q & 1) * 1024));
    }
  };
  // e2m1: the scale words of the group that turn t opens (blocks 4 q ... 4 q + 3; the last ones of a row from its end): two loads
  // a wave. Rows of fewer than four blocks have no 16 bytes: their words are put in place by hand.
  constexpr int kGroupTurns = 4 / S::TB;
  auto first_block = [&](int q) { return min(4 * q, KB - 4); };
  auto issue_scales = [&](int t) {
    const int q = t / kGroupTurns, kb = first_block(q);
    const uint32_t at = lds0 + kGroups0 + (uint32_t)(q & 1) * S::kGroup;
    if (lane < 32) dma16(pws + 4 * kb, uni(at + (uint32_t)wave * 512));
    if (brings_x && lane < kPosWave) dma16(pxs + 4 * kb, uni(at + S::kGroupW + (uint32_t)wave * (16 * kPosWave)));
  };
  if (F4 && KB >= 4) {
    issue_scales(0);
  } else if (F4) {
    for (int kb = 0; kb < KB; ++kb) {
      uint32_t* at = reinterpret_cast<uint32_t*>(smem + kGroups0) + kb;
      if (lane < 32) at[(32 * wave + lane) * 4] = ldg_u32(pws + 4 * kb);
      if (lane < kPosWave) at[S::kGroupW / 4 + (kPosWave * wave + lane) * 4] = ldg_u32(pxs + 4 * kb);
    }
  }
#pragma unroll
  for (int s = 0; s + 1 < S::kStages; ++s)
#pragma unroll
    for (int i = 0; i < S::kLoads; ++i) issue_one(s, i);

  // fragment reads. The instruction numbers an 8-bit operand's k as 64 h + 16 part + i (h: the lane's first or second four
  // registers, i: the byte) and a 4-bit operand's as 32 part + i, and takes the scale of k block g = k / 32 from the lanes
  // of part g (measured with one-hot operands): so activations and e4m3 weights give lane (row r16, part) the 16-byte
  // pieces part and 4 + part of its row's 128 bytes (LDS slots 2 part and 2 part + 1, see pc8), e2m1 weights piece part of
  // the row's 64, and every operand's scale byte `part` of the row's four goes to the lanes of that part.
  const int rd0 = (r16 >> 3) * 1024 + (r16 & 7) * 128 + ((2 * part) ^ swz(r16)) * 16;
  const int rd1 = (r16 >> 3) * 1024 + (r16 & 7) * 128 + ((2 * part + 1) ^ swz(r16)) * 16;
  const int rd4 = r16 * 64 + (part ^ sw4(r16)) * 16;
  const int rd4b[2] = {(r16 >> 3) * 1024 + (r16 & 7) * 128 + (part ^ (r16 & 7)) * 16, (r16 >> 3) * 1024 + (r16 & 7) * 128 + ((4 + part) ^ (r16 & 7)) * 16};
  auto frag8 = [&](const uint8_t* t) {
    const u32x4_t lo = *reinterpret_cast<const u32x4_t*>(t + rd0), hi = *reinterpret_cast<const u32x4_t*>(t + rd1);
    return v8i_t{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
  };
  auto frag4 = [&](const uint8_t* t, int b) {
    const u32x4_t lo = *reinterpret_cast<const u32x4_t*>(t + (S::TB == 2 ? rd4b[b] : rd4));
    return v8i_t{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, 0, 0, 0, 0};
  };
  constexpr int kScaleT = 64 * S::kWords;   // bytes of a 16-row (16-position) tile's scale words
  const int rds = r16 * (4 * S::kWords);    // the lane's row's among them; its byte: `part`
  const int rsh = 8 * part;

  v4f_t acc[S::RA][8];
#pragma unroll
  for (int t = 0; t < S::RA; ++t)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[t][j] = v4f_t{0.f, 0.f, 0.f, 0.f};

  auto run = [&](auto nj_c) {
    constexpr int NJ = decltype(nj_c)::value;
    for (int t = 0; t < TN; ++t) {
      // turn t's loads have landed; with three stages turn t + 1's may be in flight (the scale words of the group that it opens,
      // which come first, are waited for: a count of its own for those turns is a branch in every turn and 1% slower)
      if (S::kStages == 2) wait_loads<0>();
      else if (brings_x) wait_loads<S::kLoads>();
      else wait_loads<S::kLoadsW + kFirst / 2>();
      __syncthreads();
      const int tn = t + S::kStages - 1;
      // loads i with i * NJ / kLoads == j go out after the fragment reads of 16-position tile j, a group's scale words after the
      // first tile's (in front of the turn's first reads they cost the 256-position tiles 2%, at its end every shape 4%)
      auto issue_some = [&](int j) {
        if (F4 && j == 0 && tn % kGroupTurns == 0 && tn < TN) issue_scales(tn);
#pragma unroll
        for (int i = 0; i < S::kLoads; ++i)
          if (i * (NJ > 0 ? NJ : 1) / S::kLoads == j) issue_one(tn, i);
      };
      if (NJ == 0) issue_some(0);
      if (NJ == 0) continue;
      const uint8_t* st = smem + (size_t)(t % S::kStages) * S::kStageBytes;
      const uint8_t* W = st + S::RA * rg * (16 * S::kRowB);
      const uint8_t* X = st + S::kStageW + pg * 2048;
      const int q = t / kGroupTurns, word = S::TB * t - (KB >= 4 ? first_block(q) : 0);  // e2m1: the turn's first word of its group's
      const uint8_t* GS = smem + kGroups0 + (F4 ? (size_t)(q & 1) * S::kGroup + 4 * word : (size_t)(t % S::kStages) * S::kGroup);
      const uint8_t* WS = GS + S::RA * rg * kScaleT + rds;
      const uint8_t* XS = GS + S::kGroupW + pg * kScaleT + rds;
      v8i_t fa[S::TB][S::RA];
      int fs[S::TB][S::RA];
#pragma unroll
      for (int b = 0; b < S::TB; ++b)
#pragma unroll
        for (int i = 0; i < S::RA; ++i) {
          fa[b][i] = F4 ? frag4(W + i * (16 * S::kRowB), b) : frag8(W + i * 2048);
          fs[b][i] = (*reinterpret_cast<const uint32_t*>(WS + i * kScaleT + 4 * b) >> rsh) & 0xFFu;
        }
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        v8i_t fb[S::TB];
        int xsb[S::TB];
#pragma unroll
        for (int b = 0; b < S::TB; ++b) {
          fb[b] = frag8(X + b * S::kStageX + j * (2048 * WP));
          xsb[b] = (*reinterpret_cast<const uint32_t*>(XS + j * (kScaleT * WP) + 4 * b) >> rsh) & 0xFFu;
        }
        issue_some(j);
#pragma unroll
        for (int b = 0; b < S::TB; ++b)
#pragma unroll
          for (int i = 0; i < S::RA; ++i) acc[i][j] = mfma_mx<CBSZ>(fa[b][i], fb[b], acc[i][j], fs[b][i], xsb[b]);
      }
    }
  };
  constexpr int kMaxNJ = S::kSub / WP, kMinNJ = WP == 2 ? 0 : 1;
  auto run_nj = [&](auto self, auto n) {
    constexpr int N = decltype(n)::value;
    if (N == kMaxNJ || nj == N) run(n);
    else if constexpr (N < kMaxNJ) self(self, std::integral_constant<int, N + 1>{});
  };
  run_nj(run_nj, std::integral_constant<int, kMinNJ>{});
  wait_loads<0>();
  __syncthreads();

  // register q of lane l is weight row 4 (l / 16) + q of the 16-row tile, position l % 16 of the 16 positions
  if (UP) {
    const int I = g.I;
    const float lim = g.limit;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (j >= nj) break;
      const int p = 16 * (pg + WP * j) + r16;
      const float wv = (g.posw && m0 + p < mend) ? g.posw[m0 + p] : 1.f;
#pragma unroll
      for (int b = 0; b < S::RA / 2; ++b) {
        float gt[4], up[4], hv[4];
        bf16_round4(acc[2 * b][j], 1.f, gt), bf16_round4(acc[2 * b + 1][j], 1.f, up);
#pragma unroll
        for (int q = 0; q < 4; ++q) up[q] = fminf(fmaxf(up[q], -lim), lim), gt[q] = fminf(gt[q], lim);
        silu4(gt, hv);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          hv[q] = __fmul_rn(hv[q], up[q]);
          if (g.posw) hv[q] = __fmul_rn(wv, hv[q]);
        }
        const int ch = 16 * (S::RA / 2 * rg + b) + 4 * part;
        const int piece = (ch >> 3) ^ (p & 15);
        *reinterpret_cast<uint2*>(smem + p * 256 + piece * 16 + (ch & 4) * 2) = make_uint2(pack_bf16(hv[0], hv[1]), pack_bf16(hv[2], hv[3]));
      }
    }
    __syncthreads();
    // 16 lanes a position, 8 channels a lane: a scale group (32 channels) is 4 lanes. The scale byte is the exponent of
    // max(amax, 1e-4) / 448 rounded up to a power of two (ds41f engine/kernels/common.cuh:53-66); codes e4m3(h * 2^(127 - e)).
    const int l16 = tid & 15;
    for (int p = tid >> 4; p < 16 * nmt; p += kThreads / 16) {
      const int pos = m0 + p;
      const u32x4_t hv = *reinterpret_cast<const u32x4_t*>(smem + p * 256 + (l16 ^ (p & 15)) * 16);
      float v[8];
#pragma unroll
      for (int i = 0; i < 4; ++i) v[2 * i] = bf16_bits_to_f32(hv[i] & 0xFFFFu), v[2 * i + 1] = bf16_bits_to_f32(hv[i] >> 16);
      float amax = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) amax = fmaxf(amax, fabsf(v[i]));
      amax = dpp_max<0xB1>(amax);
      amax = dpp_max<0x4E>(amax);
      const uint32_t bb = __float_as_uint(__fmul_rn(fmaxf(amax, 1e-4f), 1.0f / 448.0f));
      const uint32_t eb = ((bb >> 23) & 0xFFu) + ((bb & 0x7FFFFFu) != 0 ? 1u : 0u);
      const float inv = __uint_as_float((254u - eb) << 23);
      float qv[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) qv[i] = fminf(448.f, fmaxf(-448.f, __fmul_rn(v[i], inv)));
      uint32_t o0 = __builtin_amdgcn_cvt_pk_fp8_f32(qv[0], qv[1], 0, false), o1 = __builtin_amdgcn_cvt_pk_fp8_f32(qv[4], qv[5], 0, false);
      o0 = __builtin_amdgcn_cvt_pk_fp8_f32(qv[2], qv[3], o0, true), o1 = __builtin_amdgcn_cvt_pk_fp8_f32(qv[6], qv[7], o1, true);
      if (pos < mend) {
        *reinterpret_cast<u32x4_t*>(g.h + (size_t)pos * I + c0 + 8 * l16) = hv;
        *reinterpret_cast<uint2*>(g.hq + (size_t)pos * I + c0 + 8 * l16) = make_uint2(o0, o1);
        if ((l16 & 3) == 0) g.hs[(size_t)pos * (I / 32) + c0 / 32 + (l16 >> 2)] = (uint8_t)eb;
      }
    }
  } else {
    // a 16-position tile of the wave at a time through its own piece of LDS: written as held (4 consecutive rows of one
    // position = 8 bytes of bf16), read back as whole rows (32 WP rows = 64 WP bytes a position), 4 WP lanes a position
    const int H = g.H;
    constexpr int RB = 64 * WP, PC = RB / 16;  // bytes and 16-byte pieces of a position's rows of this wave
    uint8_t* my = smem + wave * (1024 * WP);
    const int row0 = r0 + 16 * S::RA * rg;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (j >= nj) break;
#pragma unroll
      for (int t = 0; t < S::RA; ++t) {
        const uint32_t lo = pack_bf16(acc[t][j][0], acc[t][j][1]), hi = pack_bf16(acc[t][j][2], acc[t][j][3]);
        const int c = 2 * t + (part >> 1);  // the 16-byte piece: rows 16 t + 4 part ... are bytes 32 t + 8 part ...
        *reinterpret_cast<uint2*>(my + r16 * RB + ((c ^ r16) & (PC - 1)) * 16 + (part & 1) * 8) = make_uint2(lo, hi);
      }
#pragma unroll
      for (int i = 0; i < (16 * PC + 63) / 64; ++i) {
        const int idx = i * 64 + lane, p = idx / PC, c = idx % PC;
        const u32x4_t v = *reinterpret_cast<const u32x4_t*>(my + p * RB + ((c ^ p) & (PC - 1)) * 16);
        const int pos = m0 + 16 * (pg + WP * j) + p;
        if (pos < mend) *reinterpret_cast<u32x4_t*>(g.d + (size_t)pos * H + row0 + 8 * c) = v;
      }
    }
  }
}

// The tile of the shared expert's rows from m0 on (e4m3 weights), in the smallest shape that holds them
template <bool UP>
__device__ __forceinline__ void shared_tile(const Args& g, uint8_t* smem, int m0, int mend, int ns) {
  constexpr int F8 = DSGX_FMT_FP8_B32E;
  if (mend - m0 > 128) gemm_tile<UP, 256, F8>(g, smem, -1, m0, mend, ns);
  else if (mend - m0 > 64) gemm_tile<UP, 128, F8>(g, smem, -1, m0, mend, ns);
  else gemm_tile<UP, 64, F8>(g, smem, -1, m0, mend, ns);
}
// The shared expert (tile_e null: tiles of 256 rows over [0, nrows)).
template <bool UP>
__global__ void __launch_bounds__(kThreads) k_gemm(Args g) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const int NS = UP ? g.I / (kWgRows / 2) : g.H / kWgRows;
  int tile, ns;
  pf8::task_of<true>(NS, tile, ns);
  if (ns >= NS || tile * 256 >= g.nrows) return;
  shared_tile<UP>(g, smem, tile * 256, g.nrows, ns);
}
// The routed experts' list of both tile shapes (bit 30 of tile_e: a 256-position tile), an expert's tiles next to each other.
// A remainder of up to 64 rows runs two blocks a turn where K is pairs of blocks.
template <bool UP>
__global__ void __launch_bounds__(kThreads) k_gemm_mixed(Args g) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  constexpr int F4 = DSGX_FMT_MXFP4_G32;
  const int NS = UP ? g.I / (kWgRows / 2) : g.H / kWgRows;
  int tile, ns;
  if (blockIdx.x < g.sh.grid) {  // (the same for the whole workgroup)
    pf8::task_of<true>(NS, tile, ns);
    if (ns >= NS || tile * 256 >= g.nrows) return;
    Args q = g;
    q.aq = g.sh.aq, q.as = g.sh.as, q.gather = nullptr, q.posw = nullptr, q.wstride = q.sstride = 0;
    q.wa = g.sh.wa, q.sa = g.sh.sa, q.wb = g.sh.wb, q.sb = g.sh.sb, q.h = g.sh.h, q.hq = g.sh.hq, q.hs = g.sh.hs, q.d = g.sh.d;
    shared_tile<UP>(q, smem, tile * 256, g.nrows, ns);
    return;
  }
  pf8::task_of<false>(NS, tile, ns, blockIdx.x - g.sh.grid);
  if (ns >= NS || tile >= *g.ntiles) return;
  const int te = g.tile_e[tile], e = te & 0xFFFF;
  const int m0 = g.off[e] + g.tile_m0[tile], mend = g.off[e + 1];
  const bool pairs = (UP ? g.H : g.I) % 256 == 0;
  if (te >> 30) gemm_tile<UP, 256, F4>(g, smem, e, m0, mend, ns);
  else if (mend - m0 <= 64 && pairs) gemm_tile<UP, 64, F4>(g, smem, e, m0, mend, ns);
  else gemm_tile<UP, 128, F4>(g, smem, e, m0, mend, ns);
}

}  // namespace pfmx
}  // namespace dsgx
