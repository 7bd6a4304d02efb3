// The grouped GEMMs of the prefill step for INT4 (group 32) experts with bf16 activations - the altar-1 contract
// (altar1-4xgx10-switchless/engine/experts/prefill.cu:337-352, 772-831 of the reference): a weight is the bf16 value
// W = bf16((u - u_z) s), products are summed in f32 by v_mfma_f32_16x16x32_bf16, whose accumulators the MFMA carries across K.
//
// The structure is pf_gemm_fp8.cuh's: a workgroup (8 waves) computes up to 128 positions against 256 weight rows (UP: 128
// channels, gate and up), a wave 32 rows x every position; both operands and the weights' scales and zero points go from
// memory straight into rings in LDS (global_load_lds, hand-counted waits, one workgroup barrier a 128-k block), a turn's loads
// are issued one at a time between its MFMAs. What is its own:
//   * a weight row of a block is 64 bytes of packed nibbles (four lanes a row, piece q of row r at slot q ^ sw4(r)), or 128 of two;
//     lane (row, part) reads ONE piece = the 32 values of one scale group, its bf16 scale and its zero-point word, decodes
//     them in registers (the decode kernels' routine: one rounding of the exact product) into the A fragments of four MFMAs;
//     MFMA j takes the lane's values 8 j .. 8 j + 7, i.e. k = 32 part + 8 j + [0, 8), and the activation fragment of MFMA j
//     holds the same k (the permutation of k inside a block is invisible to the sums);
//   * an activation row of a block is 256 bytes of bf16: sixteen 16-byte pieces, piece c of position r at slot c ^ sw16(r), four
//     instructions a 16-position tile; a lane's piece for MFMA j is 4 part + j;
//   * a block's weights are decoded a turn ahead, between the MFMAs of the block before: vector unit and matrix unit run
//     beside each other.
// The k order of the sums - block after block, inside a block the four MFMAs j = 0 .. 3 - is k_pf_gemm16's, so the bits
// are the ones that kernel gave.
#pragma once
#include "pf_gemm_b16.cuh"

namespace dsgx {
namespace pfi4 {

using pf8::dma16;
using pf8::kThreads;
using pf8::kWgRows;
using pf8::sw4;
using pf8::v4f_t;
using pf8::wait_loads;
typedef __bf16 v8bf_t __attribute__((ext_vector_type(8)));

// A tile's shape by its positions, 64 or 128, and PAIR: LDS holds three rings of three slots each, activations (a slot a 128-k block),
// nibbles (PAIR: a slot two blocks, whole lines of a weight row, for 64 positions where K is pairs of blocks; else a block) and the
// scales and zero points of two blocks. A
// wave's weights, scales and zero points are its own, so their slot is free as soon as the wave has opened the block, a turn
// before its MFMAs: a load has two turns to land in either shape.
// What the launch waits for besides is the lines that its loads name (pf_gemm_mx.cuh): 8 bytes of scales a row and block were 32
// lines an instruction, 64 bytes of weights a row and block named every line twice. Hidden 6144, intermediate 2048, 168
// experts, gate/up with 16 / 32 / 64 / 128 rows an expert: 686 / 741 / 855 / 1301 us with a stage of every operand a block and its
// scales in it, 606 / 690 / 840 / 1180 like this (with the weights in the caches 540 / 600 / 742 / 1032).
template <int POS, bool PAIR>
struct Shape {
  static constexpr int kPos = POS;
  static constexpr int kSub = POS / 16;
  static constexpr bool kPair = PAIR;                    // two blocks a weight slot
  static constexpr int kX = POS * 256;                   // bf16 rows of a block
  static constexpr int kW = kWgRows * (kPair ? 128 : 64);
  static constexpr int kS = kWgRows * 16, kZ = (kWgRows / 8) * 32;  // two blocks: eight bf16 scales a row, eight zero-point words a group of eight rows
  static constexpr int kOffW = 3 * kX, kOffS = kOffW + 3 * kW, kOffZ = kOffS + 3 * kS;
  static constexpr int kLds = kOffZ + 3 * kZ;            // 162,816 (the epilogues reuse it: UP POS x 256 B, DOWN 8 x 2 KiB)
  static constexpr int kLoadsX = POS / 32, kLoads = 1 + 2 + kLoadsX;  // a wave's loads a turn: scales or zero points, weights, activations
};
constexpr int kLds = Shape<128, false>::kLds;
static_assert(kLds == Shape<64, true>::kLds && kLds > Shape<64, false>::kLds, "one launch, any shape");
static_assert(pfb16::kLds <= kLds, "a launch may hold the shared expert's tiles");
constexpr int kLdsRun = kLds + kThreads / 64 * 4;  // ... and a word a wave: whether it met a scale above the fast decode's range

struct Args {
  const uint16_t* x;   // activations bf16 [rows][K]
  const int* gather;   // position -> activation row (null: the position itself)
  const int* tile_e;   // 128-position tiles: expert, first position inside the expert's bucket
  const int* tile_m0;
  const int* ntiles;
  const int* off;
  dsgx_layer_w L;
  uint16_t* h;         // UP: h bf16 [position][I]
  float* d;            // DOWN: f32 [position][H]
  unsigned sh_grid;    // the shared expert's workgroups in this launch (pf8::grid_of of them, so the others keep their XCDs; 0: none)
  pfb16::Args sh;
};

// Where piece q of a row lies. A 16-byte LDS read of 64 lanes is served sixteen lanes at a time, and the sixteen are lanes
// 0-3, 12-15, 20-27 (and 4-11, 16-19, 28-31; the same from 32 on): rows 0-3 and 12-15 of one k part beside rows 4-11 of the
// next. Slots q ^ (r / 4 % 4) (64-byte rows) and c ^ r (256-byte rows), one-to-one on sixteen neighbouring rows, put two lanes
// of such a set on every bank (gate/up at T = 1111: 7.2e7 conflicts in 1.55e8 LDS cycles; 3e5 in 8.3e7 with the slots below).
// sw4 takes rows 0-3, 4-7, 8-11, 12-15 to 0, 2, 3, 1 and sw16 exchanges rows 4-7 and 12-15: one-to-one on both kinds of sixteen.
__device__ __forceinline__ int sw16(int r) { return r ^ ((r & 4) << 1); }

template <bool UP, int POS, bool PAIR>
__device__ __forceinline__ void gemm_tile(const Args& g, uint8_t* smem, int e, int m0, int mend, int ns) {
  using S = Shape<POS, PAIR>;
  constexpr int kPos = S::kPos;
  const int K = UP ? g.L.H : g.L.I, N = UP ? g.L.I : g.L.H, KB = K / 128, G = K / 32;
  if (mend > m0 + kPos) mend = m0 + kPos;
  const dsgx_mat_desc* dsc = g.L.desc + (size_t)e * 3;
  const size_t soff = ((size_t)N * K / 2 + 255) / 256 * 256, zoff = soff + ((size_t)N * G * 2 + 255) / 256 * 256;
  const uint8_t* ma = g.L.pool + dsc[UP ? 0 : 2].off;   // UP: gate; DOWN: down
  const uint8_t* mb = UP ? g.L.pool + dsc[1].off : ma;  // UP: up
  const float s2a = UP ? dsc[0].s2 : 1.f, s2b = UP ? dsc[1].s2 : 1.f;
  const int tid = threadIdx.x, lane = tid & 63, wave = uni(tid >> 6), r16 = lane & 15, part = lane >> 4;
  const int c0 = ns * (kWgRows / 2), r0 = ns * kWgRows;
  // the wave's two 16-row tiles: UP the gate rows and the up rows of channels c0 + 16 wave ...; DOWN rows r0 + 32 wave + 16 t ...
  auto tile_row = [&](int t, const uint8_t*& base) {
    base = (UP && t) ? mb : ma;
    return UP ? c0 + 16 * wave : r0 + 32 * wave + 16 * t;
  };
  const int nmt = uni(min(S::kSub, (mend - m0 + 15) / 16));

  // ---- what this lane fetches ----
  // weights: 64-byte rows: one instruction a tile, lane -> row lane / 4, piece (lane % 4) ^ sw4(row); 128-byte rows: two
  // instructions a tile (rows 0-7, 8-15), lane -> row lane / 8, piece (lane % 8) ^ (row % 8)
  const uint8_t* pw[2];
  const uint8_t* psc;  // scales, lanes 0-31: the 16 bytes of tile lane / 16, row lane % 16
  const uint8_t* pzp;  // zero points, lanes 0-7: 16 of the 32 bytes of tile lane / 4, octet lane / 2 % 2
  {
    const uint8_t* base;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int row = tile_row(t, base), rl = lane >> (S::kPair ? 3 : 2);
      pw[t] = base + (size_t)(row + rl) * (K / 2) + 16 * (S::kPair ? (lane & 7) ^ rl : (lane & 3) ^ sw4(rl));
    }
    const int rows = tile_row((lane >> 4) & 1, base);
    psc = base + soff + (size_t)(rows + r16) * G * 2;
    const int rowz = tile_row((lane >> 2) & 1, base);
    pzp = base + zoff + (size_t)((rowz >> 3) + ((lane >> 1) & 1)) * G * 4 + (KB > 1 ? 16 * (lane & 1) : 0);
  }
  // activations: the wave brings positions kPos / 8 wave ... (none if they lie past a small tile's end); instruction i: position
  // 4 i + lane / 16 of them, piece (lane % 16) ^ sw16(position)
  const bool brings_x = POS > 64 || m0 + 8 * wave < mend;
  const uint8_t* px[S::kLoadsX];
#pragma unroll
  for (int i = 0; i < S::kLoadsX; ++i) {
    const int p = kPos / 8 * wave + 4 * i + (lane >> 4);
    const int pos = min(m0 + p, mend - 1);  // (a ragged tile re-reads its last row: never stored)
    px[i] = reinterpret_cast<const uint8_t*>(g.x) + (size_t)(g.gather ? g.gather[pos] : pos) * K * 2 + 16 * ((lane & 15) ^ sw16(p & 15));
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem;
  // The loads, each clamped past K's end (the last block again, into a slot nobody reads). Scales and zero points: pair q of
  // blocks; the last pair of an odd number of blocks starts a block early.
  auto first_block = [&](int q) { return max(0, min(2 * q, KB - 2)); };
  auto load_s = [&](int q) {
    if (lane < 32) dma16(psc + 8 * first_block(q), uni(lds0 + S::kOffS + (uint32_t)(q % 3) * S::kS + (uint32_t)wave * 512));
  };
  auto load_z = [&](int q) {
    if (lane < 8) dma16(pzp + 16 * first_block(q), uni(lds0 + S::kOffZ + (uint32_t)(q % 3) * S::kZ + (uint32_t)wave * 128));
  };
  auto load_x = [&](int kb, int i) {
    if (brings_x) dma16(px[i] + (size_t)min(kb, KB - 1) * 256, uni(lds0 + (uint32_t)(kb % 3) * S::kX + (uint32_t)wave * (kPos * 32) + i * 1024));
  };
  auto load_w = [&](int q, int t, int hh) {  // slot q: block q, or pair q (its rows 8 hh ...)
    const int last = S::kPair ? KB / 2 - 1 : KB - 1;
    dma16(pw[t] + (S::kPair ? (size_t)hh * 4 * K : 0) + (size_t)min(q, last) * (S::kPair ? 128 : 64),  // (rows 8-15: the same pieces)
          uni(lds0 + S::kOffW + (uint32_t)(q % 3) * S::kW + (uint32_t)wave * (S::kPair ? 4096 : 2048) + t * (S::kPair ? 2048 : 1024) + hh * 1024));
  };
  // load i of turn kb: activations of block kb + 2, weights of block kb + 3, or half the rows of pair kb / 2 + 2, scales (even
  // turns) or zero points (odd turns) of pair kb / 2 + 2; the small ones first, then the activations (L2 hits mostly), the weights
  // last (a wave's loads return in issue order: the ones that wait for HBM hold back every later one)
  auto issue_one = [&](int kb, int i) {
    const int q = (kb >> 1) + 2;
    if (i == 0) {
      if (kb & 1) load_z(q);
      else load_s(q);
    } else if (i <= S::kLoadsX) {
      load_x(kb + 2, i - 1);
    } else {
      const int t = i - 1 - S::kLoadsX;
      if (S::kPair) load_w(q, t, kb & 1);
      else load_w(kb + 3, t, 0);
    }
  };
  // what the first turns need: blocks 0 (and 1, opened in turn 0), then block 1's activations and the next weights
  auto fill = [&]() {
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      load_s(n), load_z(n);
#pragma unroll
      for (int i = 0; i < S::kLoadsX; ++i) load_x(n, i);
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        if (S::kPair) load_w(n, t, 0), load_w(n, t, 1);
        else if (n == 0) load_w(0, t, 0), load_w(1, t, 0);
        else load_w(2, t, 0);
      }
    }
  };
  constexpr int kSecond = 2 + S::kLoadsX + (S::kPair ? 4 : 2);  // a wave's loads of fill's second pass
  fill();

  // fragment reads: the lane's 32 nibbles (row r16, group `part` of the block), its bf16 scale, its zero-point word (the row's
  // nibble: r16 % 8), the activation piece of MFMA j: 4 part + j of position r16
  const int rdw = S::kPair ? (r16 >> 3) * 1024 + (r16 & 7) * 128 + (part ^ (r16 & 7)) * 16 : r16 * 64 + (part ^ sw4(r16)) * 16;  // (a pair's second block: ^ 64)
  const int rds = r16 * 16 + part * 2, rdz = (r16 >> 3) * 32 + part * 4;
  const uint32_t zsh = 4 * (r16 & 7);
  int rdx[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) rdx[j] = r16 * 256 + ((4 * part + j) ^ sw16(r16)) * 16;

  v4f_t acc[2][8];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[t][j] = v4f_t{0.f, 0.f, 0.f, 0.f};

  // A block's weights are decoded a turn ahead, a piece (one MFMA's fragment) at a time between the MFMAs of the turn before:
  // the decode is vector-unit work and the MFMAs run beside it. (Decoded in front of its own MFMAs it stood in their way: both
  // waves of a SIMD reach it together behind the barrier: 1.39 -> 1.1 ms for gate/up.)
  u32x4_t raw[2];
  I4Group grp[2];
  uint32_t uz[2];
  float smax = 0.f;  // the largest scale that this lane has met (in magnitude; a NaN decodes to NaN by either routine)
  auto open_block = [&](int kb) {  // the lane's raw words, scale and zero point of the wave's two tiles of block kb
    const int q = kb >> 1, o = kb - first_block(q);  // the pair whose scales and zero points the block's are among, which of the two
    const uint8_t* W = smem + S::kOffW + (size_t)((S::kPair ? q : kb) % 3) * S::kW + wave * (S::kPair ? 4096 : 2048) + (S::kPair ? rdw ^ ((kb & 1) * 64) : rdw);
    const uint8_t* SC = smem + S::kOffS + (size_t)(q % 3) * S::kS + wave * 512 + 8 * o + rds;
    const uint8_t* Z = smem + S::kOffZ + (size_t)(q % 3) * S::kZ + wave * 128 + 16 * o + rdz;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      raw[t] = *reinterpret_cast<const u32x4_t*>(W + t * (S::kPair ? 2048 : 1024));
      uz[t] = (*reinterpret_cast<const uint32_t*>(Z + t * 64) >> zsh) & 15u;
      grp[t] = i4_group(bf16_bits_to_f32(*reinterpret_cast<const uint16_t*>(SC + t * 256)), uz[t]);
    }
    smax = fmaxf(smax, fmaxf(fabsf(grp[0].s), fabsf(grp[1].s)));
  };
  auto piece = [&](auto any, u32x4_t (&fa)[2][4], int pc) {  // piece pc = 4 t + j of the opened block
    const int t = pc >> 2, j = pc & 3;
    const uint32_t w = j == 0 ? raw[t].x : j == 1 ? raw[t].y : j == 2 ? raw[t].z : raw[t].w;
    uint32_t o[4];
    if constexpr (decltype(any)::value) i4x8_to_bf16_any(w, grp[t].s, -((float)uz[t] * grp[t].s), o);
    else i4x8_to_bf16(w, grp[t], o);
    fa[t][j] = u32x4_t{o[0], o[1], o[2], o[3]};
  };
  auto run = [&](auto nj_c, auto any) {  // any: decode by the routine for every scale
    constexpr int NJ = decltype(nj_c)::value;
    u32x4_t fa[2][4], fn[2][4];
    // fill's first pass has landed (the second may be in flight)
    if (brings_x) wait_loads<kSecond>();
    else wait_loads<kSecond - S::kLoadsX>();
    __syncthreads();
    open_block(0);
#pragma unroll
    for (int pc = 0; pc < 8; ++pc) piece(any, fa, pc);
    auto turn = [&](int kb, u32x4_t (&fa)[2][4], u32x4_t (&fn)[2][4]) {
      // what turn kb - 2 asked for has landed: the activations of block kb, the weights of block kb + 1 (turn kb - 1's loads may be
      // in flight; turn 0: fill's first pass)
      if (kb > 0) {
        if (brings_x) wait_loads<S::kLoads>();
        else wait_loads<S::kLoads - S::kLoadsX>();
      }
      __syncthreads();
      open_block(min(kb + 1, KB - 1));
      const uint8_t* X = smem + (size_t)(kb % 3) * S::kX;
#pragma unroll
      for (int mt = 0; mt < 8; ++mt) {
        // (the turn's loads between its MFMAs; a ragged tile issues what is left behind its last 16-position tile)
#pragma unroll
        for (int i = 0; i < S::kLoads; ++i)
          if (mt < NJ && i * NJ / S::kLoads == mt) issue_one(kb, i);
        piece(any, fn, mt);
        if (mt >= NJ) continue;
        u32x4_t fb[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) fb[j] = *reinterpret_cast<const u32x4_t*>(X + mt * 4096 + rdx[j]);
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int t = 0; t < 2; ++t)
            acc[t][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf_t, fa[t][j]), __builtin_bit_cast(v8bf_t, fb[j]), acc[t][mt], 0, 0, 0);
      }
    };
    for (int kb = 0; kb < KB; kb += 2) {  // (two turns a pass: the two fragment buffers swap roles without copies)
      turn(kb, fa, fn);
      if (kb + 1 < KB) turn(kb + 1, fn, fa);
    }
  };
  switch (nmt) {
    case 1: run(std::integral_constant<int, 1>{}, std::false_type{}); break;
    case 2: run(std::integral_constant<int, 2>{}, std::false_type{}); break;
    case 3: run(std::integral_constant<int, 3>{}, std::false_type{}); break;
    default:
      if constexpr (S::kSub == 4) {
        run(std::integral_constant<int, 4>{}, std::false_type{});
      } else {
        switch (nmt) {
          case 4: run(std::integral_constant<int, 4>{}, std::false_type{}); break;
          case 5: run(std::integral_constant<int, 5>{}, std::false_type{}); break;
          case 6: run(std::integral_constant<int, 6>{}, std::false_type{}); break;
          case 7: run(std::integral_constant<int, 7>{}, std::false_type{}); break;
          default: run(std::integral_constant<int, 8>{}, std::false_type{}); break;
        }
      }
      break;
  }
  // A tile that met a scale which i4x8_to_bf16 is not for (2^116 or more, none in a checkpoint) is done once more, by the routine
  // for every scale. The turns only keep the maximum: with a vote and the second decode in every turn (two copies in each of
  // fourteen bodies, 21,500 instructions of gate/up against 16,600) tiles of few positions, which wait for their loads, were
  // slower than before the fast decode: gate/up at T = 64, hidden 6144, intermediate 2048: 468 -> 492 us, 472 like this.
  int* met = reinterpret_cast<int*>(smem + kLds);
  const bool large = i4_any_large(smax);
  if (lane == 0) met[wave] = large;
  wait_loads<0>();
  __syncthreads();
  int any_met = 0;
#pragma unroll
  for (int i = 0; i < kThreads / 64; ++i) any_met |= met[i];
  if (__builtin_expect(uni(any_met), 0)) {  // (the same in every wave)
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[t][j] = v4f_t{0.f, 0.f, 0.f, 0.f};
    fill();
    run(std::integral_constant<int, S::kSub>{}, std::true_type{});
    wait_loads<0>();
    __syncthreads();
  }

  if (UP) pfb16::store_h(smem, acc, nmt, s2a, s2b, m0, mend, c0, g.L.I, g.h);
  else pfb16::store_d(smem, acc, nmt, m0, mend, r0, g.L.H, g.d);
}

// The routed experts' tiles, and in front of them (workgroups 0 .. sh_grid - 1) the BF16 shared expert's, if the launch holds those.
// PAIR: K is an even number of 128-k blocks; only down has an odd number (up to 64 rows of one: in the 128-position shape every wave
// fetches activations that nobody reads; whole call of hidden 2048, intermediate 384, 64 experts, T = 17 / 60: 69.5 / 75.7 us there, 68.1 /
// 74.8 like this). A kernel of its own: as a third shape of one kernel it cost the others up to 1.3% (hidden 6144, intermediate 2048, 168
// experts, T = 17 / 40 / 60: 396.5 / 551 / 685 us, 391.5 / 544 / 677.5 like this). The check of K under PAIR is always true; it is
// there for the code that the compiler makes of it: without it 394 / 547.5 / 681.
template <bool UP, bool PAIR>
__global__ void __launch_bounds__(kThreads) k_gemm(Args g) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  if (blockIdx.x < g.sh_grid) {  // (the same for the whole workgroup)
    pfb16::tiles<UP>(g.sh, smem, blockIdx.x);
    return;
  }
  const int NS = UP ? g.L.I / (kWgRows / 2) : g.L.H / kWgRows;
  int tile, ns;
  pf8::task_of<false>(NS, tile, ns, blockIdx.x - g.sh_grid);
  if (ns >= NS || tile >= *g.ntiles) return;
  const int e = g.tile_e[tile];
  const int m0 = g.off[e] + g.tile_m0[tile], mend = g.off[e + 1];
  if (mend - m0 <= 64 && (!PAIR || (UP ? g.L.H : g.L.I) % 256 == 0)) gemm_tile<UP, 64, PAIR>(g, smem, e, m0, mend, ns);
  else gemm_tile<UP, 128, false>(g, smem, e, m0, mend, ns);
}

}  // namespace pfi4
}  // namespace dsgx
