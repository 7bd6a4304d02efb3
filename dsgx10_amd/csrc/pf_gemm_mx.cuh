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
using pf8::kMaxPos;
using pf8::kThreads4;
using pf8::kWaves;
using pf8::kWgRows;
using pf8::sc_half;
using pf8::static_for;
using pf8::sw4;
using pf8::swz;
using pf8::v4f_t;
using pf8::v8i_t;
using pf8::wait_loads;

// A tile's shape by its positions (32, 64 or 160; the shared expert's 64 or 128), its weights' format and the blocks of a turn.
// What bounds these launches is what L2 does not hold, at 5.5 TB/s (hidden 5120, intermediate 2304, 256 experts, top-6, T = 3000:
// gate/up 5.7 GB of missed lines in 1.02 ms, 3.2 of them weights and their scales once), and tiles of few rows:
//   * two workgroups of four waves a CU (pf_gemm_fp8.cuh): whole call T = 60 / 300 / 3000 474 / 882 / 1537 -> 435 / 830 / 1470 us;
//   * half a line a weight row and block (e2m1: 64 bytes) names every line twice: tiles of up to 64 positions take two blocks a
//     turn, whole lines;
//   * a line of scale words is a row's for 32 blocks and has left L2 when its next words are asked for: with four blocks' words a
//     load scale words were 1.25 of the 5.7 GB; eight a load (the weight rows' in ONE buffer, which the wave frees by reading it) 5.3
//     GB, gate/up 1022 -> 989 us (5.9 GB with the shared expert's tiles and the stores);
//   * an expert of many rows reads its weights once a tile: 160 positions instead of 128 (T = 2000 / 6000 1280 -> 1246, 2100 -> 2013).
// R > 0: the shared expert's shape for one workgroup a CU (k_few): weights and activations R turns ahead, and two buffers of the weight
// rows' scale words.
template <int POS, int WF, int TB_, int R = 0>
struct Shape {
  static constexpr bool F4 = WF == DSGX_FMT_MXFP4_G32;
  static constexpr int kPos = POS, kSub = POS / 16, RA = 4, TB = TB_;
  static constexpr int kRowB = F4 ? 64 * TB : 128;  // bytes of a weight row in a turn
  static constexpr int kTileB = 16 * kRowB, LT = kRowB / 64;  // a 16-row weight tile, its loads
  static constexpr int kRing = R ? 4 * R : F4 ? (POS == 32 ? 6 : 4) : POS == 128 ? 4 : 6;  // the wave's own ring of weight tiles
  static constexpr int kAhead = R ? R : 1, kStages = kAhead + 1;
  static constexpr int kStageX = POS * 128;         // one block's activations; a stage is TB blocks
  static constexpr int kHX = POS / 8 / kWaves;      // the 8-position half tiles that a wave brings
  static constexpr int kOffX = kWaves * kRing * kTileB, kOffS = kOffX + kStages * TB * kStageX;
  static constexpr int kScaleW = kWgRows * 32, kScaleX = POS * 32;  // eight blocks' scale words of the weight rows, and of the positions (two such buffers)
  static constexpr int kOffSX = kOffS + (R ? 2 : 1) * kScaleW, kLds = kOffSX + 2 * kScaleX;   // (the epilogues reuse it: UP kPos x 256 B, DOWN 4 x 2 KiB)
  static_assert(F4 || TB == 1, "pairs of blocks are for 64-byte rows");
  static_assert(R == 0 || TB == 1, "R blocks of weights");
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
  const int* tile_e;   // the list of tiles of kMaxPos positions (null: the shared expert on rows [0, nrows))
  pf8::Map map;
  const int* tile_m0;
  const int* ntiles;
  const int* off;
  int nrows;
  const int *tile_e_low, *tile_m0_low, *ntiles_low;  // the same rows as a list of tiles of kLowPos positions
  int slots;           // workgroups that the chip holds at once (lower_tiles)
  int stream;          // weights of experts of one small tile as streaming loads
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

template <bool UP, int POS, int WF, int TB, bool STREAM = false, int R = 0>
__device__ __forceinline__ void gemm_tile(const Args& g, uint8_t* smem, int e, int m0, int mend, int ns) {
  using S = Shape<POS, WF, TB, R>;
  constexpr bool F4 = S::F4;
  constexpr int CBSZ = F4 ? 4 : 0;
  const int K = UP ? g.H : g.I, KB = K / 128, G = K / 32;
  if (mend > m0 + S::kPos) mend = m0 + S::kPos;
  const size_t eo = e < 0 ? 0 : (size_t)e;
  const uint8_t *wa = g.wa + eo * g.wstride, *sa = g.sa + eo * g.sstride;
  const uint8_t *wb = UP ? g.wb + eo * g.wstride : wa, *sb = UP ? g.sb + eo * g.sstride : sa;
  const int tid = threadIdx.x, lane = tid & 63, wave = uni(tid >> 6), r16 = lane & 15, part = lane >> 4;
  const int c0 = ns * (kWgRows / 2), r0 = ns * kWgRows;
  // The workgroup's sixteen 16-row tiles, four a wave: first weight row of tile i. UP: tile 2 c is the gate rows, tile 2 c + 1 the
  // up rows of channels c0 + 16 c ...
  auto tile_row = [&](int i) { return UP ? c0 + 16 * (i >> 1) : r0 + 16 * i; };
  const int RB = F4 ? K / 2 : K;  // bytes of a weight row
  const uint8_t* wt[S::RA];
#pragma unroll
  for (int t = 0; t < S::RA; ++t) wt[t] = (UP && (t & 1) ? wb : wa) + (size_t)tile_row(S::RA * wave + t) * RB;
  const int nmt = uni(min(S::kSub, (mend - m0 + 15) / 16));
  // ---- what this lane fetches ----
  // weights: 64-byte rows: one instruction a tile, lane -> row lane / 4, piece (lane % 4) ^ sw4(row); 128-byte rows: two
  // instructions a tile (rows 0-7, 8-15), lane -> row lane / 8, piece (lane % 8) ^
  // swz(row) (e4m3) or (lane % 8) ^ (row % 8) (two blocks of e2m1, whose lanes read pieces part and 4 + part)
  uint32_t ow[2];
#pragma unroll
  for (int hh = 0; hh < 2; ++hh) {
    const int r = S::kRowB == 64 ? lane >> 2 : 8 * hh + (lane >> 3);
    const int piece = S::kRowB == 64 ? (lane & 3) ^ sw4(r) : F4 ? (lane & 7) ^ (r & 7) : pc8((lane & 7) ^ swz(r));
    ow[hh] = (uint32_t)r * RB + 16 * piece;
  }
  // the scale words of eight blocks of the wave's 64 rows: two loads, lane -> row 32 i + lane / 2 of them, half sc_half(row, lane)
  const uint8_t* pws[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = 32 * i + (lane >> 1), row = tile_row(S::RA * wave + (r >> 4)) + (r & 15);
    pws[i] = (UP && ((r >> 4) & 1) ? sb : sa) + (size_t)(F4 ? row : row / 32) * G + (KB >= 8 ? 16 * sc_half(r & 15, lane) : 0);
  }
  // activations: half tile kHX wave + i is positions 8 (kHX wave + i) ...; those past the tile's rows are not fetched (R: they are, so that
  // every wave has as many loads in flight as its waits count)
  const int nhx = R ? S::kHX : uni(min(S::kHX, max(0, (mend - m0 + 7) / 8 - S::kHX * wave)));
  auto row_of = [&](int p) {  // the activation row of the tile's position p (a ragged tile re-reads its last row: never stored)
    const int pos = min(m0 + p, mend - 1);
    return (uint32_t)(g.gather ? g.gather[pos] : pos);
  };
  uint32_t ox[S::kHX];
#pragma unroll
  for (int i = 0; i < S::kHX; ++i) {
    const int p = 8 * (S::kHX * wave + i) + (lane >> 3);
    ox[i] = row_of(p) * (uint32_t)K + 16 * pc8((lane & 7) ^ swz(p & 15));
  }
  constexpr int kPosWave = POS / kWaves, kSI = (2 * kPosWave + 63) / 64;  // the wave's positions; the loads of eight blocks of their scale words: half a position's a lane
  uint32_t oxs[kSI];
#pragma unroll
  for (int i = 0; i < kSI; ++i) {
    const int p = kPosWave * wave + min((64 * i + lane) >> 1, kPosWave - 1);
    oxs[i] = row_of(p) * (uint32_t)G + (KB >= 8 ? 16 * sc_half(p & 15, lane) : 0);
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem;
  const uint32_t ring0 = lds0 + (uint32_t)wave * (S::kRing * S::kTileB);
  // Weight tile i of the wave's sequence (tile i % 4 of turn i / 4, clamped: past the end the last turn again, into a slot nobody
  // reads) goes to slot i % kRing of the wave's own ring, whose rows no other wave reads: a slot is free as soon as the wave has read
  // its fragments. Activations: a stage a turn.
  const int TN = KB / TB;
  auto issue_w = [&](int t, int i, int slot, int hh) {
    pf8::dma16_w<STREAM>(wt[i] + (size_t)min(t, TN - 1) * S::kRowB, ow[hh], uni(ring0 + (uint32_t)slot * S::kTileB + hh * 1024));
  };
  auto issue_x = [&](int t) {
    const uint32_t xbase = lds0 + S::kOffX + (uint32_t)(t % S::kStages) * (TB * S::kStageX) + (uint32_t)wave * (S::kHX * 1024);
#pragma unroll
    for (int b = 0; b < TB; ++b)
#pragma unroll
      for (int i = 0; i < S::kHX; ++i) {
        if (i >= nhx) break;
        dma16(g.aq + (size_t)min(t, TN - 1) * (128 * TB) + 128 * b, ox[i], uni(xbase + b * S::kStageX + i * 1024));
      }
  };
  // The scale words of the group that turn t opens (blocks 8 q ... 8 q + 7; the last ones of a row from its end): the weight rows'
  // into the wave's one buffer, which is free when the group's last words are read (R: into two); the positions' into two. A line of L2 holds a
  // row's words of 32 blocks and has left L2 when the next group comes, so what counts is how often it is named. Rows of fewer than
  // eight blocks: their words are put in place by hand.
  constexpr int kGroupTurns = 8 / TB;
  auto first_block = [&](int q) { return min(8 * q, KB - 8); };
  auto issue_scales = [&](int t) {
    const int q = t / kGroupTurns, kb = first_block(q);
#pragma unroll
    for (int i = 0; i < 2; ++i) dma16(pws[i] + 4 * kb, uni(lds0 + S::kOffS + (R ? (uint32_t)(q & 1) * S::kScaleW : 0) + (uint32_t)wave * 2048 + i * 1024));
#pragma unroll
    for (int i = 0; i < kSI; ++i)
      if (nhx > 0 && 64 * i + lane < 2 * kPosWave) dma16(g.as + 4 * kb, oxs[i], uni(lds0 + S::kOffSX + (uint32_t)(q & 1) * S::kScaleX + (uint32_t)wave * (32 * kPosWave) + i * 1024));
  };
  if (KB >= 8) {
    issue_scales(0);
  } else {
    uint32_t w[2][7], x[kSI][7];
#pragma unroll
    for (int i = 0; i < 7; ++i) {
      const int o = 4 * min(i, KB - 1);
      w[0][i] = ldg_u32(pws[0] + o), w[1][i] = ldg_u32(pws[1] + o);
#pragma unroll
      for (int k = 0; k < kSI; ++k) x[k][i] = ldg_u32(g.as + oxs[k] + o);
    }
    if (!(lane & 1)) {
      const int r = lane >> 1;
#pragma unroll
      for (int i = 0; i < 7; ++i) {
#pragma unroll
        for (int k = 0; k < 2; ++k) reinterpret_cast<uint32_t*>(smem + S::kOffS)[(64 * wave + 32 * k + r) * 8 + 4 * sc_half(r & 15, i >> 2) + (i & 3)] = w[k][i];
#pragma unroll
        for (int k = 0; k < kSI; ++k) {
          const int p = kPosWave * wave + 32 * k + r;
          if (32 * k + r < kPosWave) reinterpret_cast<uint32_t*>(smem + S::kOffSX)[p * 8 + 4 * sc_half(p & 15, i >> 2) + (i & 3)] = x[k][i];
        }
      }
    }
  }
  issue_x(0);
#pragma unroll
  for (int i = 0; i < S::kRing; ++i) {
    if (R && i > 0 && i % 4 == 0) issue_x(i / 4);
#pragma unroll
    for (int hh = 0; hh < S::LT; ++hh) issue_w(i / 4, i % 4, i, hh);
  }

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
    const u32x4_t lo = *reinterpret_cast<const u32x4_t*>(t + (TB == 2 ? rd4b[b] : rd4));
    return v8i_t{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, 0, 0, 0, 0};
  };
  const int rsh = 8 * part;

  v4f_t acc[S::RA][S::kSub];
#pragma unroll
  for (int t = 0; t < S::RA; ++t)
#pragma unroll
    for (int j = 0; j < S::kSub; ++j) acc[t][j] = v4f_t{0.f, 0.f, 0.f, 0.f};

  auto run = [&](auto nj_c) {
    constexpr int NJ = decltype(nj_c)::value;
    int slot = 0;  // of the turn's first weight tile: 4 t % kRing
    for (int t = 0; t < TN; ++t) {
      // this wave's loads of turn t have landed (weight tiles of later turns may be in flight; R: all of R - 1 later turns, loads of scales
      // among them only make the wait longer); after the barrier everyone's have, and everyone is done reading the stage of turn
      // t - 1, which the activations of turn t + kAhead now overwrite
      wait_loads<R ? (R - 1) * (4 * S::LT + S::kHX) : S::LT * (S::kRing - 4)>();
      __syncthreads();
      const int q = t / kGroupTurns, word = TB * t - (KB >= 8 ? first_block(q) : 0);  // the turn's first word of its group's
      // (a turn of two blocks begins at an even word: both lie in one half)
      const int at = r16 * 32 + 16 * sc_half(r16, word >> 2) + 4 * (word & 3);  // the lane's row's words of the turn in a 16-row (16-position) tile's 512 bytes; its byte: `part`
      const uint8_t* WS = smem + S::kOffS + (R ? (q & 1) * S::kScaleW : 0) + wave * 2048 + at;
      const uint8_t* XS = smem + S::kOffSX + (size_t)(q & 1) * S::kScaleX + at;
      const uint8_t* X = smem + S::kOffX + (size_t)(t % S::kStages) * (TB * S::kStageX);
      int sl[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) sl[i] = slot + i >= S::kRing ? slot + i - S::kRing : slot + i;
      v8i_t fa[TB][S::RA];
      int fs[TB][S::RA];
#pragma unroll
      for (int b = 0; b < TB; ++b)
#pragma unroll
        for (int i = 0; i < S::RA; ++i) {
          const uint8_t* W = smem + wave * (S::kRing * S::kTileB) + sl[i] * S::kTileB;
          fa[b][i] = F4 ? frag4(W, b) : frag8(W);
          fs[b][i] = (*reinterpret_cast<const uint32_t*>(WS + i * 512 + 4 * b) >> rsh) & 0xFFu;
        }
      if (R && (t + S::kAhead) % kGroupTurns == 0 && t + S::kAhead < TN) issue_scales(t + S::kAhead);
      issue_x(t + S::kAhead);
#pragma unroll
      for (int b = 0; b < TB; ++b)  // (read: what holds them may be written from here on)
        asm volatile("" : "+v"(fa[b][0]), "+v"(fa[b][1]), "+v"(fa[b][2]), "+v"(fa[b][3]), "+v"(fs[b][0]), "+v"(fs[b][1]), "+v"(fs[b][2]), "+v"(fs[b][3]));
      if (!R && (t + 1) % kGroupTurns == 0 && t + 1 < TN) issue_scales(t + 1);
      // (R: a wave has its SIMD for itself, so the next step's fragment is read before this one's MFMAs)
      v8i_t fn;
      int xn;
      auto next = [&](int j) { fn = frag8(X + j * 2048), xn = (*reinterpret_cast<const uint32_t*>(XS + j * 512) >> rsh) & 0xFFu; };
      if constexpr (R) next(0);
      static_for<NJ>([&](auto jc) {
        constexpr int j = decltype(jc)::value;
        v8i_t fb[TB];
        int xsb[TB];
        if constexpr (R) {
          fb[0] = fn, xsb[0] = xn;
          if (j + 1 < NJ) next(j + 1);
        } else {
#pragma unroll
          for (int b = 0; b < TB; ++b) {
            fb[b] = frag8(X + b * S::kStageX + j * 2048);
            xsb[b] = (*reinterpret_cast<const uint32_t*>(XS + j * 512 + 4 * b) >> rsh) & 0xFFu;
          }
        }
        // (the weights' loads one by one between the MFMAs)
#pragma unroll
        for (int i = 0; i < 4 * S::LT; ++i)
          if (i * NJ / (4 * S::LT) == j) issue_w(t + (S::kRing + i / S::LT) / 4, (S::kRing + i / S::LT) % 4, sl[i / S::LT], i % S::LT);
#pragma unroll
        for (int b = 0; b < TB; ++b)
#pragma unroll
          for (int i = 0; i < S::RA; ++i) acc[i][j] = mfma_mx<CBSZ>(fa[b][i], fb[b], acc[i][j], fs[b][i], xsb[b]);
      });
      slot = slot + 4 >= S::kRing ? slot + 4 - S::kRing : slot + 4;
    }
  };
  auto run_nj = [&](auto self, auto n) {
    constexpr int N = decltype(n)::value;
    if (N == S::kSub || nmt == N) run(n);
    else if constexpr (N < S::kSub) self(self, std::integral_constant<int, N + 1>{});
  };
  run_nj(run_nj, std::integral_constant<int, F4 && POS == 64 ? 3 : !F4 && POS == 128 ? 5 : 1>{});
  wait_loads<0>();
  __syncthreads();

  // register q of lane l is weight row 4 (l / 16) + q of the 16-row tile, position l % 16 of the 16 positions
  if (UP) {
    const int I = g.I;
    const float lim = g.limit;
    static_for<S::kSub>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      if (j >= nmt) return;
      const int p = 16 * j + r16;
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
        const int ch = 16 * (S::RA / 2 * wave + b) + 4 * part;
        const int piece = (ch >> 3) ^ (p & 15);
        *reinterpret_cast<uint2*>(smem + p * 256 + piece * 16 + (ch & 4) * 2) = make_uint2(pack_bf16(hv[0], hv[1]), pack_bf16(hv[2], hv[3]));
      }
    });
    __syncthreads();
    // 16 lanes a position, 8 channels a lane: a scale group (32 channels) is 4 lanes. The scale byte is the exponent of
    // max(amax, 1e-4) / 448 rounded up to a power of two (ds41f engine/kernels/common.cuh:53-66); codes e4m3(h * 2^(127 - e)).
    const int l16 = tid & 15;
    for (int p = tid >> 4; p < 16 * nmt; p += kThreads4 / 16) {
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
    // position = 8 bytes of bf16), read back as whole rows (64 rows = 128 bytes a position), 8 lanes a position
    const int H = g.H;
    uint8_t* my = smem + wave * 2048;
    const int row0 = r0 + 16 * S::RA * wave;
    static_for<S::kSub>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      if (j >= nmt) return;
#pragma unroll
      for (int t = 0; t < S::RA; ++t) {
        const uint32_t lo = pack_bf16(acc[t][j][0], acc[t][j][1]), hi = pack_bf16(acc[t][j][2], acc[t][j][3]);
        const int c = 2 * t + (part >> 1);  // the 16-byte piece: rows 16 t + 4 part ... are bytes 32 t + 8 part ...
        *reinterpret_cast<uint2*>(my + r16 * 128 + ((c ^ r16) & 7) * 16 + (part & 1) * 8) = make_uint2(lo, hi);
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int p = 8 * i + (lane >> 3), c = lane & 7;
        const u32x4_t v = *reinterpret_cast<const u32x4_t*>(my + p * 128 + ((c ^ p) & 7) * 16);
        const int pos = m0 + 16 * j + p;
        if (pos < mend) __builtin_nontemporal_store(v, reinterpret_cast<u32x4_t*>(g.d + (size_t)pos * H + row0 + 8 * c));
      }
    });
  }
}

constexpr int kLds = std::max({Shape<kMaxPos, DSGX_FMT_MXFP4_G32, 1>::kLds, Shape<64, DSGX_FMT_MXFP4_G32, 2>::kLds, Shape<32, DSGX_FMT_MXFP4_G32, 2>::kLds,
                               Shape<128, DSGX_FMT_FP8_B32E, 1>::kLds, Shape<64, DSGX_FMT_FP8_B32E, 1>::kLds});
static_assert(2 * kLds <= 160 * 1024, "two workgroups a CU");

// The tile of the shared expert's rows from m0 on (e4m3 weights), in the smallest shape that holds them
template <bool UP>
__device__ __forceinline__ void shared_tile(const Args& g, uint8_t* smem, int m0, int mend, int ns) {
  constexpr int F8 = DSGX_FMT_FP8_B32E;
  if (mend - m0 > 64) gemm_tile<UP, 128, F8, 1>(g, smem, -1, m0, mend, ns);
  else gemm_tile<UP, 64, F8, 1>(g, smem, -1, m0, mend, ns);
}
// The shared expert (tile_e null: tiles of 128 rows over [0, nrows)).
template <bool UP>
__global__ void __launch_bounds__(kThreads4, 2) k_gemm(Args g) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const int NS = UP ? g.I / (kWgRows / 2) : g.H / kWgRows;
  int tile, ns;
  pf8::task_of<true>(NS, tile, ns, blockIdx.x, g.map);
  if (ns >= NS || tile * 128 >= g.nrows) return;
  shared_tile<UP>(g, smem, tile * 128, g.nrows, ns);
}
// ... in no more tiles than the chip has CUs: one workgroup a CU, which has the CU's LDS for loads in flight.
template <bool UP, int POS, int R>
__global__ void __launch_bounds__(kThreads4, 2) k_few(Args g) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const int NS = UP ? g.I / (kWgRows / 2) : g.H / kWgRows;
  int tile, ns;
  pf8::task_of<true>(NS, tile, ns, blockIdx.x, g.map);
  if (ns >= NS || tile * POS >= g.nrows) return;
  gemm_tile<UP, POS, DSGX_FMT_FP8_B32E, 1, false, R>(g, smem, -1, tile * POS, g.nrows, ns);
}
// Whether the routed experts' rows go in tiles of 128 positions instead of 160. Many rounds of workgroups over the chip: 160, an expert's
// weights are read less often. Up to two: what the rounds take by the tallest tile of each, from the very counts of tiles (a fortieth of a
// round does not count: its workgroups find the slots of small tiles). Top-4 of 32, 160 / 128: hidden 1024, intermediate 512, T = 1000 / 2000 / 3000 /
// 4500 / 6000 50.8 / 45.3, 55.6 / 57.4, 68.1 / 61.5, 77.7 / 91, 111.5 / 102.4 us, hidden 2048 62.9 / 56.4, 70.8 / 78.3, 98.2 / 89.3, 112 / 129, 155.5 /
// 149.5. As kernels of eight waves and 256 positions 58, 60.4, 62.7, 102, 105 and 70.6, 83.3, 88.1, 138, 154.
constexpr int kLowPos = 128;
__device__ __forceinline__ bool lower_tiles(const Args& g, int NS) {
  if (!g.slots) return false;
  const int shared = g.sh.grid ? (g.nrows + 127) / 128 : 0;
  auto rounds = [&](int n) { return (40 * (n + shared) * NS + 39 * g.slots - 1) / (40 * g.slots); };
  const int r = rounds(*g.ntiles);
  return r <= 2 && rounds(*g.ntiles_low) * kLowPos < r * kMaxPos;
}
// The routed experts' list of tiles, an expert's tiles next to each other.
// A tile of up to 64 rows runs two blocks a turn where K is pairs of blocks; where K is an odd number (only down) every tile takes the
// one shape without pairs (down of hidden 2048, intermediate 384, top-6 of 64, T = 17 / 100 / 600, whole call, kernels of eight waves with 128 positions for
// those tiles / this: 41.7 / 50.2 / 80.3 and 30.3 / 43.1 / 62.9 us; 5120 x 1152, top-6 of 256, T = 40 / 250 / 1500 242 / 485 / 730 and 177 / 393 / 625).
template <bool UP>
__global__ void __launch_bounds__(kThreads4, 2) k_gemm_mixed(Args g) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  constexpr int F4 = DSGX_FMT_MXFP4_G32;
  const int NS = UP ? g.I / (kWgRows / 2) : g.H / kWgRows;
  int tile, ns;
  if (blockIdx.x < g.sh.grid) {  // (the same for the whole workgroup)
    pf8::task_of<true>(NS, tile, ns, blockIdx.x, g.map);
    if (ns >= NS || tile * 128 >= g.nrows) return;
    Args q = g;
    q.aq = g.sh.aq, q.as = g.sh.as, q.gather = nullptr, q.posw = nullptr, q.wstride = q.sstride = 0;
    q.wa = g.sh.wa, q.sa = g.sh.sa, q.wb = g.sh.wb, q.sb = g.sh.sb, q.h = g.sh.h, q.hq = g.sh.hq, q.hs = g.sh.hs, q.d = g.sh.d;
    shared_tile<UP>(q, smem, tile * 128, g.nrows, ns);
    return;
  }
  pf8::task_of<false>(NS, tile, ns, blockIdx.x - g.sh.grid, g.map);
  const bool low = lower_tiles(g, NS);
  const int *tile_e = low ? g.tile_e_low : g.tile_e, *tile_m0 = low ? g.tile_m0_low : g.tile_m0;
  if (ns >= NS || tile >= *(low ? g.ntiles_low : g.ntiles)) return;
  const int e = tile_e[tile];
  const int m0 = g.off[e] + tile_m0[tile], mend = min(g.off[e + 1], m0 + (low ? kLowPos : kMaxPos));
  const bool pairs = (UP ? g.H : g.I) % 256 == 0;
  if (mend - m0 > 64 || !pairs) gemm_tile<UP, kMaxPos, F4, 1>(g, smem, e, m0, mend, ns);
  else if (mend - m0 > 32) gemm_tile<UP, 64, F4, 2>(g, smem, e, m0, mend, ns);
  else if (g.stream && tile_m0[tile] == 0) gemm_tile<UP, 32, F4, 2, true>(g, smem, e, m0, mend, ns);
  else gemm_tile<UP, 32, F4, 2>(g, smem, e, m0, mend, ns);
}

}  // namespace pfmx
}  // namespace dsgx
