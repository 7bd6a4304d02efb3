// The grouped GEMMs of the prefill step for INT4 (group 32) experts with bf16 activations - the altar-1 contract
// (altar1-4xgx10-switchless/engine/experts/prefill.cu:337-352, 772-831 of the reference): a weight is the bf16 value
// W = bf16((u - u_z) s), products are summed in f32 by the bf16 MFMA, whose accumulators it carries across K.
//
// The structure is pf_gemm_fp8.cuh's: a workgroup (4 waves, two workgroups a CU) computes up to 128 positions against 256 weight rows
// (UP: 128 channels, gate and up), a wave 64 rows x every position; both operands and the weights' scales and zero points go from
// memory straight into LDS (global_load_lds, hand-counted waits), a turn's loads are issued one at a time between its MFMAs. What
// is its own:
//   * a weight row of a 128-k block is 64 bytes of packed nibbles, four pieces of the 32 values of one scale group each. MT = 16: lane (row, lp) of
//     a 16-row tile takes piece lp, MT = 32: lane (row, lp) of a 32-row tile takes pieces lp and 2 + lp, with their bf16 scales and zero-point
//     words, and decodes them in registers (the decode kernels' routine: one rounding of the exact product) into the A fragments of steps (j, a),
//     j = 0 .. 3, a = 0 or 0, 1: the values 8 j .. 8 j + 7 of piece 2 a + lp, i.e. k = 32 (2 a + lp) + 8 j + [0, 8), and the activation
//     fragment holds the same k (the permutation of k inside a block is invisible to the sums);
//   * an activation row of a block is 256 bytes of bf16, sixteen 16-byte pieces; a lane's piece of step (j, a) is 4 (2 a + lp) + j;
//   * the MFMAs of a step of all positions stand together, so that only their fragments of the weights and the next step's have to be held;
//     the next step's are decoded between them: vector unit and matrix unit run beside each other.
// The k order of the sums - block after block, inside a block j after j, the two steps of a j of v_mfma_f32_32x32x16_bf16 together one
// 16 x 16 x 32 (pf_gemm_b16.cuh) - is k_pf_gemm16's, so the bits are the ones that kernel gave.
//
// Tiles of more than 64 positions take MT = 32, which leaves the vector unit its issue slots (with the 16 x 16 x 32 instruction the busy times of the
// two units added up to the launch); smaller ones MT = 16, whose last tile has fewer empty positions. Two workgroups of four waves a CU,
// as their barriers, first loads and epilogues are not each other's, against one of eight waves of 32 rows: gate/up of hidden
// 6144, intermediate 2048, 168 experts with 8 / 32 / 64 / 96 / 128 rows an expert 732 / 711 / 846 / 985 / 1150 -> 512 / 608 / 748 / 885 / 1010 us,
// down 350 / 385 / 467 / 577 / 672 -> 258 / 325 / 424 / 527 / 612. (MT = 32 for every tile: gate/up 564 / 601 / 746 / 904 / 1086.) What bounds it
// now: few rows an expert the decode (2.4 vector instructions a value, 60% of the issue slots) beside the weights' way from HBM; many rows
// the chip's power: at 96 rows an expert the MFMAs' 16 x 16 x 32 form took 1.43e7 clocks at 1.77 GHz, the 32 x 32 x 16 form 1.1e7 at 1.4.
#pragma once
#include "pf_gemm_b16.cuh"

namespace dsgx {
namespace pfi4 {


using pf8::dma16;
using pf8::dma16_w;
using pf8::kThreads4;
using pf8::kWaves;
using pf8::kWgRows;
using pf8::sw4;
using pf8::swz;
using pf8::v4f_t;
using pf8::wait_loads;
using pfb16::v8bf_t;

// PAIR: K is pairs of 128-k blocks. A block is two turns, of the MFMAs j = 0, 1 and 2, 3. LDS holds three stages of a turn's activations,
// the waves' own nibbles (PAIR: a slot of two blocks, whole lines of a weight row; else two slots of a block) and the scales and zero points
// of two blocks. A wave reads a pair's words, scales and zero points into registers together: their slot is free then, and the next
// pair's have most of two blocks to land. What the launch waits for besides is the lines that its loads name (pf_gemm_mx.cuh): 8 bytes of
// scales a row and block were 32 lines an instruction, 64 bytes of weights a row and block named every line twice.
constexpr int kMaxPos = 128;  // positions of a tile of the list
constexpr int stages(int pos) { return pos > 96 ? 2 : 3; }    // of a turn's activations, `pos` positions x 64 k: what 80 KiB of LDS hold beside the rest
constexpr int kW = 8192, kS = 64 * 16, kZ = 8 * 32;           // a wave's: nibbles; two blocks' scales a row; two blocks' zero-point words an octet of rows
constexpr int kOffW = 3 * 96 * 128, kOffS = kOffW + kWaves * kW, kOffZ = kOffS + kWaves * kS;
constexpr int kLds = std::max(kOffZ + kWaves * kZ, pfb16::kLds);  // (the epilogues reuse it: UP 128 x 256 B, DOWN 4 x 8 KiB)
constexpr int kLdsRun = kLds + kWaves * 4;  // ... and a word a wave: whether it met a scale above the fast decode's range
static_assert(2 * kLdsRun <= 160 * 1024, "two workgroups a CU");
// What a turn asks for behind the activations of the turn after the next (a wave's loads return in issue order: the ones that wait for
// HBM hold back every later one), turn i of a pair's four: PAIR, the first: the next pair's scales, zero points and weights; else a block's
// first: the weights of the block after the next, a pair's first also the next pair's scales and zero points.
constexpr int loads(bool pair, int i) {
  i = (i + 4) % 4;
  return pair ? (i == 0 ? 10 : 0) : i == 0 ? 6 : i == 2 ? 4 : 0;
}
constexpr int loads_x(int pos) { return (pos + 31) / 32; }    // a wave's instructions for a stage of activations, eight positions each
// how many of a wave's loads may be in flight at the start of turn i, which needs the activations that turn i - stages + 1 asked for first
constexpr int young(bool pair, int pos, int i) { return stages(pos) == 2 ? loads(pair, i - 1) : loads(pair, i - 2) + loads_x(pos) + loads(pair, i - 1); }

// Which workgroups share an XCD: four tiles x four row groups (gate/up with 8 / 64 / 224 rows an expert, eight tiles x four groups 622 / 756 /
// 1846 us, one x eight 511 / 737 / 1924, this 512 / 748 / 1828; whole calls, this / 1 x 8 / 8 x 4 / 4 x 2: 6144 x 2048, 168 experts, T = 250 / 1200 / 2500 887 / 888 /
// 897 / 893, 1413 / 1439 / 1421 / 1426, 2184 / 2219 / 2231 / 2233; 3072 x 1536, 48 experts, T = 250 / 1200 139 / 141 / 159 / 142, 295 / 305 / 304 / 306; 2048 x 768, 64
// experts, T = 2500 175 / 179 / 186 / 175; 16 experts of 6144 x 2048, T = 250 219 / 220 / 214 / 201).
__host__ __device__ inline pf8::Map map_of(int NS) { return pf8::map_of(2, 2, NS); }

struct Args {
  const uint16_t* x;   // activations bf16 [rows][K]
  const int* gather;   // position -> activation row (null: the position itself)
  const int* tile_e;   // tiles of kMaxPos positions: expert, first position inside the expert's bucket
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
// 0-3, 12-15, 20-27 (and 4-11, 16-19, 28-31; the same from 32 on). Of 128-byte rows two fill the banks, of 64-byte rows four. Tiles of 32 rows:
// the sixteen read one piece of sixteen rows: slot q ^ (r / 2 % 8) (64-byte rows: q ^ (r / 4 % 4)) is one-to-one on the even rows of either set and on
// the odd ones. Tiles of 16 rows: they read one part's piece of rows 0-3 and 12-15 and the next part's of rows 4-11; the next part's differs in
// bit 1 of 2 part + j (activations: swz) and in bit 0 of the nibbles' part (r % 8; 64-byte rows sw4).
template <int MT>
__device__ __forceinline__ int slot_x(int r) { return MT == 16 ? swz(r) : (r >> 1) & 7; }
template <int MT>
__device__ __forceinline__ int slot_w(int r) { return MT == 16 ? r & 7 : (r >> 1) & 7; }
template <int MT>
__device__ __forceinline__ int slot_w64(int r) { return MT == 16 ? sw4(r) : (r >> 2) & 3; }

template <bool UP, bool PAIR, int MT>
__device__ __forceinline__ void gemm_tile(const Args& g, uint8_t* smem, int e, int m0, int mend, int ns) {
  const int K = UP ? g.L.H : g.L.I, N = UP ? g.L.I : g.L.H, KB = K / 128, G = K / 32;
  if (mend > m0 + kMaxPos) mend = m0 + kMaxPos;
  const dsgx_mat_desc* dsc = g.L.desc + (size_t)e * 3;
  const size_t soff = ((size_t)N * K / 2 + 255) / 256 * 256, zoff = soff + ((size_t)N * G * 2 + 255) / 256 * 256;
  const uint8_t* ma = g.L.pool + dsc[UP ? 0 : 2].off;   // UP: gate; DOWN: down
  const uint8_t* mb = UP ? g.L.pool + dsc[1].off : ma;  // UP: up
  const float s2a = UP ? dsc[0].s2 : 1.f, s2b = UP ? dsc[1].s2 : 1.f;
  const int tid = threadIdx.x, lane = tid & 63, wave = uni(tid >> 6), r = lane % MT, lp = lane / MT;
  constexpr int NT = 64 / MT, NA = MT / 16, kPt = MT == 16 ? 4 : kMaxPos / 32;  // a wave's row tiles; a lane's pieces of a row's block; position tiles
  const int c0 = ns * (kWgRows / 2), r0 = ns * kWgRows;
  // the wave's row tiles: UP the gate rows (t even) and the up rows (t odd) of channels c0 + 32 wave + MT (t / 2) ...; DOWN rows
  // r0 + 64 wave + MT t ...
  auto tile_row = [&](int t, const uint8_t*& base) {
    base = (UP && (t & 1)) ? mb : ma;
    return UP ? c0 + 32 * wave + MT * (t >> 1) : r0 + 64 * wave + MT * t;
  };
  const int npt = uni((mend - m0 + MT - 1) / MT);  // the position tiles that hold rows

  // ---- what this lane fetches ----
  // weights: 128-byte rows: eight instructions of eight rows each: row lane / 8, slot lane % 8; 64-byte rows: four of sixteen
  // rows: row lane / 4, slot lane % 4
  const uint8_t* wt[NT];
  const uint8_t* psc;  // scales: the 16 bytes of tile lane / MT, row lane % MT
  const uint8_t* pzp;  // zero points, lanes 0-15: 16 of the 32 bytes of octet lane / 2 of the wave's eight
  {
    const uint8_t* base;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int row = tile_row(t, base);
      wt[t] = base + (size_t)row * (K / 2);
    }
    const int rows = tile_row(lp, base);
    psc = base + soff + (size_t)(rows + r) * G * 2;
    const int oct = lane >> 1 & 7, rowz = tile_row(oct / (MT / 8), base);
    pzp = base + zoff + (size_t)((rowz >> 3) + oct % (MT / 8)) * G * 4 + (KB > 1 ? 16 * (lane & 1) : 0);
  }
  uint32_t ow[2];  // (128-byte rows: of every second eight)
#pragma unroll
  for (int i = 0; i < 2; ++i)
    ow[i] = (uint32_t)(lane >> (PAIR ? 3 : 2)) * (K / 2) + 16 * (PAIR ? (lane & 7) ^ slot_w<MT>(8 * i + (lane >> 3)) : (lane & 3) ^ slot_w64<MT>(lane >> 2));
  // activations: half a block's of eight positions an instruction: group wave + 4 i of eights (of an odd number of 16-position tiles the
  // last waves bring two groups that others bring), position lane / 8 of them, slot lane % 8 holds piece 2 part + j % 2
  const uint8_t* x0 = reinterpret_cast<const uint8_t*>(g.x) + (g.gather ? 0 : (size_t)m0 * K * 2);
  constexpr int kXL = loads_x(MT * kPt);
  auto x_group = [&](int npt_, int i) { return wave + 4 * i < npt_ * (MT / 8) ? wave + 4 * i : wave + 4 * i - 2; };
  uint32_t ox[kXL];  // (T rows of gathered activations are under 4 GiB: dsgx_moe_prefill)
#pragma unroll
  for (int i = 0; i < kXL; ++i) {
    const int p = 8 * x_group(npt, i) + (lane >> 3), pos = min(m0 + p, mend - 1);  // (a ragged tile re-reads its last row: never stored)
    const int pc = (lane & 7) ^ slot_x<MT>(p % MT);
    ox[i] = (uint32_t)(g.gather ? g.gather[pos] : pos - m0) * (uint32_t)(K * 2) + 64 * (pc >> 1) + 16 * (pc & 1);
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem;
  // The loads, each clamped past K's end (the last block again, into a slot nobody reads). Scales and zero points: pair q of
  // blocks; the last pair of an odd number of blocks starts a block early.
  auto first_block = [&](int q) { return max(0, min(2 * q, KB - 2)); };
  auto load_s = [&](int q) { dma16(psc + 8 * first_block(q), uni(lds0 + kOffS + (uint32_t)wave * kS)); };
  auto load_z = [&](int q) {
    if (lane < 16) dma16(pzp + 16 * first_block(q), uni(lds0 + kOffZ + (uint32_t)wave * kZ));
  };
  auto load_x = [&](auto nj_c, int turn, int stage) {  // turn: two a block
    constexpr int NJ = decltype(nj_c)::value;
    const int kb = min(turn >> 1, KB - 1);
#pragma unroll
    for (int i = 0; i < loads_x(MT * NJ); ++i)
      dma16(x0 + (size_t)kb * 256 + (turn & 1) * 32, ox[i], uni(lds0 + (uint32_t)(stage * (NJ * MT * 128) + x_group(NJ, i) * 1024)));
  };
  // (small tiles' weights as streaming loads, mostly their expert's only tile: gate/up with 8 / 64 rows an expert 539 / 753 -> 506 / 726 us; tall
  // tiles' not, their expert has others that find them in L2: hidden 3840, intermediate 768, 20 experts, T = 1500 406 -> 381)
  auto load_w = [&](int q, int i) {  // PAIR: pair q, rows 8 i ... of the wave's; else block q, rows 16 i ...
    constexpr int kRows = PAIR ? 8 : 16;
    const int t = kRows * i / MT;
    dma16_w<MT == 16>(wt[t] + (size_t)min(q, PAIR ? KB / 2 - 1 : KB - 1) * (PAIR ? 128 : 64) + (size_t)(kRows * i % MT) * (K / 2), ow[PAIR ? i & 1 : 0],
             uni(lds0 + kOffW + (uint32_t)wave * kW + (PAIR ? 0 : (q & 1) * 4096) + i * 1024));
  };
  auto load_b = [&](int kb, bool odd, int i) {  // load i of loads()
    if (!odd && i == 0) load_s((kb >> 1) + 1);
    else if (!odd && i == 1) load_z((kb >> 1) + 1);
    else load_w(PAIR ? (kb >> 1) + 1 : kb + 2, odd ? i : i - 2);
  };

  // fragment reads: the lane's 32 nibbles of piece lp (piece 2 + lp: ^ 32; a pair's second block: ^ 64), its activation piece of the
  // turn's first step (second j: ^ 16, a = 1: ^ 64)
  const int rdw = PAIR ? r * 128 + (lp ^ slot_w<MT>(r)) * 16 : r * 64 + (lp ^ slot_w64<MT>(r)) * 16;
  const int rds = r * 16 + lp * 2, rdz = (r >> 3) * 32 + lp * 4;
  const uint32_t zsh = 4 * (r & 7);
  const int rdx = r * 128 + ((2 * lp) ^ slot_x<MT>(r)) * 16;

  pfb16::acc_t<MT> acc[NT][kPt];
  auto zero = [&]() {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int j = 0; j < kPt; ++j)
#pragma unroll
        for (int i = 0; i < MT * MT / 64; ++i) acc[t][j][i] = 0.f;
  };
  zero();

  u32x4_t raw[PAIR ? 2 : 1][NT][NA];  // [PAIR: a pair's blocks][tile][a]
  I4Group grp[NT][NA];
  uint32_t uz[NT][NA], later[NT][NA];  // later: the second block's scale above its zero point
  float smax = 0.f;  // the largest scale that this lane has met (in magnitude; a NaN decodes to NaN by either routine)
  auto open_block = [&](int kb, bool odd) {  // the lane's words, scales and zero points of block kb
    const uint8_t* W = smem + kOffW + wave * kW;
    const int o0 = kb - first_block(kb >> 1), o1 = KB > 1 ? 1 : 0;  // where a pair's two blocks are among its scales (an odd K's last one is second)
    auto scale = [&](int t, int a, int o) { return (uint32_t)*reinterpret_cast<const uint16_t*>(smem + kOffS + wave * kS + t * (MT * 16) + 8 * o + 4 * a + rds); };
    auto zero_point = [&](int t, int a, int o) { return (*reinterpret_cast<const uint32_t*>(smem + kOffZ + wave * kZ + t * (MT * 4) + 16 * o + 8 * a + rdz) >> zsh) & 15u; };
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int a = 0; a < NA; ++a) {
        uint32_t sc;
        if constexpr (!PAIR) raw[0][t][a] = *reinterpret_cast<const u32x4_t*>(W + (kb & 1) * 4096 + t * (MT * 64) + (rdw ^ (32 * a)));
        if (odd) {
          sc = later[t][a] >> 16, uz[t][a] = later[t][a] & 15u;
        } else {
          if constexpr (PAIR) {
#pragma unroll
            for (int b = 0; b < 2; ++b) raw[b][t][a] = *reinterpret_cast<const u32x4_t*>(W + t * (MT * 128) + (rdw ^ (32 * a + 64 * b)));
          }
          sc = scale(t, a, o0), uz[t][a] = zero_point(t, a, o0);
          later[t][a] = scale(t, a, o1) << 16 | zero_point(t, a, o1);
        }
        grp[t][a] = i4_group(bf16_bits_to_f32(sc), uz[t][a]);
        smax = fmaxf(smax, fabsf(grp[t][a].s));
      }
  };
  auto keep_raw = [&]() {  // (read: their slots may be written from here on)
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int a = 0; a < NA; ++a) {
        asm volatile("" : "+v"(raw[0][t][a]), "+v"(later[t][a]));
        if constexpr (PAIR) asm volatile("" : "+v"(raw[1][t][a]));
      }
  };
  auto piece = [&](auto any, bool odd, int t, int step) {  // the fragment of step NA j + a of tile t of the opened block
    const int j = step / NA, a = step % NA;
    const u32x4_t& r = raw[PAIR && odd ? 1 : 0][t][a];
    const uint32_t w = j == 0 ? r.x : j == 1 ? r.y : j == 2 ? r.z : r.w;
    uint32_t o[4];
    if constexpr (decltype(any)::value) i4x8_to_bf16_any(w, grp[t][a].s, -((float)uz[t][a] * grp[t][a].s), o);
    else i4x8_to_bf16(w, grp[t][a], o);
    return u32x4_t{o[0], o[1], o[2], o[3]};
  };
  auto run = [&](auto nj_c, auto any) {  // nj: position tiles; any: decode by the routine for every scale
    constexpr int NJ = decltype(nj_c)::value;
    // what the first turns need (not PAIR: and the second block's weights)
    constexpr int kStages = stages(MT * NJ);
#pragma unroll
    for (int t = 0; t < kStages - 1; ++t) load_x(nj_c, t, t);
    load_s(0), load_z(0);
#pragma unroll
    for (int i = 0; i < 8; ++i) PAIR ? load_w(0, i) : load_w(i >> 2, i & 3);
    constexpr int kSteps = 2 * NA;  // a turn's
    u32x4_t fa[NT], fn[NT];
    wait_loads<PAIR ? 0 : 4>();  // (the wave's own: no barrier)
    open_block(0, false);
#pragma unroll
    for (int t = 0; t < NT; ++t) fa[t] = piece(any, false, t, 0);
    keep_raw();
    int stage = 0;  // of the turn's activations
    // turn th of block kb, odd: its parity
    auto turn = [&](int kb, auto odd_c, auto th_c) {
      constexpr bool odd = decltype(odd_c)::value;
      constexpr int th = decltype(th_c)::value, in_pair = 2 * odd + th, kLoads = loads(PAIR, in_pair);
      // The turn's activations have landed, and with them everything asked for before them: in a pair's last turn the next pair's words, scales
      // and zero points; not PAIR, in a block's second the next block's. After the barrier everyone's have, and everyone is done reading
      // the stage that the ones asked for now overwrite.
      wait_loads<young(PAIR, MT * NJ, in_pair)>();
      __syncthreads();
      const uint8_t* X = smem + (size_t)stage * (NJ * MT * 128);
      load_x(nj_c, 2 * kb + th + kStages - 1, stage == 0 ? kStages - 1 : stage - 1);
      stage = stage == kStages - 1 ? 0 : stage + 1;
      // a turn's fragments of the activations in the order of their use: step (j % 2, a), position tile; two on their way
      auto frag_x = [&](auto nc) {
        constexpr int n = decltype(nc)::value, st = n / NJ;
        return *reinterpret_cast<const u32x4_t*>(X + (n % NJ) * (MT * 128) + (rdx ^ (16 * (st / NA) + 64 * (st % NA))));
      };
      u32x4_t bn[2];
      bn[0] = frag_x(std::integral_constant<int, 0>{}), bn[1] = frag_x(std::integral_constant<int, 1>{});
      pf8::static_for<kSteps * NJ>([&](auto nc) {
        constexpr int n = decltype(nc)::value, st = n / NJ, pt = n % NJ, step = kSteps * th + st;  // of the turn, of the block
        if constexpr (step == 2 * kSteps - 1 && pt == 0) open_block(min(kb + 1, KB - 1), !odd);
        const u32x4_t fb = bn[n & 1];
        if constexpr (n + 2 < kSteps * NJ) bn[n & 1] = frag_x(std::integral_constant<int, n + 2>{});
        if constexpr (kLoads > 0) {
#pragma unroll
          for (int i = 0; i < kLoads; ++i)
            if (i * kSteps * NJ / kLoads == n) load_b(kb, odd, i);
        }
#pragma unroll
        for (int t = 0; t < NT; ++t)
          if (t * NJ / NT == pt) fn[t] = step == 2 * kSteps - 1 ? piece(any, !odd, t, 0) : piece(any, odd, t, (step + 1) % (2 * kSteps));
#pragma unroll
        for (int t = 0; t < NT; ++t)
          if constexpr (MT == 16) acc[t][pt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf_t, fa[t]), __builtin_bit_cast(v8bf_t, fb), acc[t][pt], 0, 0, 0);
          else acc[t][pt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf_t, fa[t]), __builtin_bit_cast(v8bf_t, fb), acc[t][pt], 0, 0, 0);
        if constexpr (pt == NJ - 1) {
#pragma unroll
          for (int t = 0; t < NT; ++t) fa[t] = fn[t];
          if constexpr (step == 2 * kSteps - 1) keep_raw();
        }
      });
    };
    auto block = [&](int kb, auto odd_c) {
      turn(kb, odd_c, std::integral_constant<int, 0>{});
      turn(kb, odd_c, std::integral_constant<int, 1>{});
    };
    for (int kb = 0; kb < KB; kb += 2) {
      block(kb, std::false_type{});
      if (PAIR || kb + 1 < KB) block(kb + 1, std::true_type{});
    }
  };
  auto run_npt = [&](auto self, auto n) {
    constexpr int NJ = decltype(n)::value;
    if (NJ == kPt || npt == NJ) run(n, std::false_type{});
    else if constexpr (NJ < kPt) self(self, std::integral_constant<int, NJ + 1>{});
  };
  run_npt(run_npt, std::integral_constant<int, MT == 16 ? 1 : 3>{});
  // A tile that met a scale which i4x8_to_bf16 is not for (2^116 or more, none in a checkpoint) is done once more, by the routine
  // for every scale. The turns only keep the maximum: with a vote and the second decode in every turn (as kernels of eight waves: two copies
  // in each of fourteen bodies, 21,500 instructions of gate/up against 16,600) tiles of few positions were slower than
  // before the fast decode: gate/up at T = 64, hidden 6144, intermediate 2048: 468 -> 492 us, 472 like this.
  int* met = reinterpret_cast<int*>(smem + kLds);
  const bool large = i4_any_large(smax);
  if (lane == 0) met[wave] = large;
  wait_loads<0>();
  __syncthreads();
  int any_met = 0;
#pragma unroll
  for (int i = 0; i < kWaves; ++i) any_met |= met[i];
  if (__builtin_expect(uni(any_met), 0)) {  // (the same in every wave)
    zero();
    run(std::integral_constant<int, kPt>{}, std::true_type{});  // (positions past the tile's own: rows that nobody stores)
    wait_loads<0>();
    __syncthreads();
  }

  if (UP) pfb16::store_h<MT>(smem, acc, s2a, s2b, m0, mend, c0, g.L.I, g.h);
  else pfb16::store_d<MT>(smem, acc, m0, mend, r0, g.L.H, g.d);
}

// The routed experts' tiles, and in front of them (workgroups 0 .. sh_grid - 1) the BF16 shared expert's, if the launch holds those.
// PAIR: K is an even number of 128-k blocks; only down has an odd number. A kernel of its own: its shapes in the other's code cost
// that up to 1.3% when a workgroup was eight waves.
template <bool UP, bool PAIR>
__global__ void __launch_bounds__(kThreads4, 2) k_gemm(Args g) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  if (blockIdx.x < g.sh_grid) {  // (the same for the whole workgroup)
    pfb16::tiles<UP>(g.sh, smem, blockIdx.x);
    return;
  }
  const int NS = UP ? g.L.I / (kWgRows / 2) : g.L.H / kWgRows;
  int tile, ns;
  pf8::task_of<false>(NS, tile, ns, blockIdx.x - g.sh_grid, map_of(NS));
  if (ns >= NS || tile >= *g.ntiles) return;
  const int e = g.tile_e[tile];
  const int m0 = g.off[e] + g.tile_m0[tile], mend = g.off[e + 1];
  if (mend - m0 <= 64) gemm_tile<UP, PAIR, 16>(g, smem, e, m0, mend, ns);
  else gemm_tile<UP, PAIR, 32>(g, smem, e, m0, mend, ns);
}

}  // namespace pfi4
}  // namespace dsgx
