// The FP8 x FP8 grouped GEMM of the prefill step (gate/up + SwiGLU, and down), DeepSeek's block-scaled contract
// (ds41f-4xgx10-switchless/ref/torchref/kernel.py:105-125, ref/inference/kernel.py:207-274 of the reference): per 128-k
// block the e4m3 x e4m3 products summed in f32 from zero, then acc = fma(x_scale * w_scale, partial, acc).
//
// A workgroup (4 waves, two workgroups a CU) computes one tile of up to 32 or 160 positions against 256 weight rows (UP: 128
// channels, gate and up): a wave owns 64 weight rows and every position. Two workgroups a CU, because their barriers, first loads
// and epilogues are not each other's: as one workgroup of eight waves and 256 positions, a tile's first stage and epilogue (4 and
// 12 of 84 us) and every wait for its slowest load left the CU idle (hidden 4096, intermediate 2048, 256 experts, whole call,
// T = 8192: 2975 -> 2813 us; 3.45M -> 2.88M clocks of gate/up). What bounds it now is what L2 does not hold: 8.6 GB of lines missed
// in gate/up at T = 8192 (4.3 of them the weights once), which come at 5.3 to 6 TB/s whatever their kind; the chip also lowers its
// clock in this launch (1.8 GHz). Hence 160 positions and not 128 (an expert's weights are read again for each of its tiles: T = 3000
// 1744 -> 1718, T = 8192 2858 -> 2836; 160 is what 256 registers a lane hold), and the scales' loads below.
// Weights are the MFMA's A operand, so a lane's four accumulators of a 16 x 16 tile belong to ONE position and the
// block's combined scale is one value a lane.
//
// Both operands go from memory straight into LDS (global_load_lds_dwordx4: no registers, no LDS store instructions).
// Such a load puts lane l's 16 bytes at (base) + 16 l, so the LDS layout is chosen by what each lane fetches: a 16-row
// tile is two instructions of eight rows, eight consecutive lanes fetch the eight 16-byte pieces of one row's 128 bytes
// (one full line of the caches) in the order piece = q ^ swz(row), swz(r) = (r % 8) ^ (r / 8), which leaves piece c of
// row r at slot 8 r + (c ^ swz(r)): the MFMA-order reads (consecutive lanes = consecutive rows, one piece) then touch
// different bank groups, whether the LDS serves 8 lanes (128 bytes) or 16 lanes (256 bytes) a clock: swz is one-to-one
// on rows 0-7, on rows 8-15, on the even rows and on the odd rows (measured: no bank conflicts).
// The loads are written as inline assembly with the waits counted by hand (the compiler would otherwise wait for every
// outstanding load before each LDS read): a wave's loads return in issue order, and a turn issues its weights last, so
// vmcnt(the weight loads still allowed in flight) = "the block of this turn has landed". Addresses are a scalar base and a lane's
// offset, so that a load costs the vector unit nothing.
//
// The number of live 16-position tiles of a wave (ragged tiles: most experts of a chunk hold fewer rows than a tile) is
// a template parameter of the loop: a turn is straight-line code, the MFMAs take the constant 0 as their addend, and
// tiles past the end cost nothing.
//
// Epilogues go through LDS so that every store instruction writes whole 128-byte lines (a lane's accumulators are four
// consecutive weight rows of one position: stored directly, each line would be written in pieces by several
// instructions, which the memory system pays for several times over). UP also quantises h for the down projection
// (act_quant over the workgroup's 128 channels = one scale block) on the way out.
#pragma once
#include <algorithm>
#include <type_traits>
#include <utility>

#include "abi_internal.h"
#include "common.cuh"

namespace dsgx {
namespace pf8 {

typedef int v8i_t __attribute__((ext_vector_type(8)));
typedef float v4f_t __attribute__((ext_vector_type(4)));

constexpr int kWgRows = 256;      // weight rows a workgroup (UP: 128 channels)
constexpr int kWaves = 4, kThreads4 = 64 * kWaves;

// LDS of one of two workgroups on a CU: the waves' own rings of weight tiles (a slot is free when its fragments are read, so RING - 4
// tiles come two turns ahead and four one turn), two stages of activations, two buffers of scales. Deeper rings are no gain where many
// tiles are in flight: a shape of 64 positions and 7 tiles was slower than the widest with 4 (T = 1200 1361 -> 1308 us), and
// dsgx_moe_prefill says where 32 positions take 8.
constexpr int kMaxPos = 160;
// R > 0: a shape for one workgroup a CU (k_few): weights and activations R blocks ahead.
template <int POS, int RING = 4, int R = 0>
struct Shape {
  static_assert(R == 0 || RING == 4 * R, "R blocks of weights");
  static constexpr int kPos = POS;                 // positions of a tile
  static constexpr int kSub = POS / 16;            // its 16-position tiles
  static constexpr int RA = 4;                     // 16-row tiles a wave
  static constexpr int kRing = RING;               // the wave's own ring of weight tiles, 2 KiB each
  static constexpr int kHX = POS / 32;             // 8-position half tiles that a wave brings
  static constexpr int kStageX = POS * 128;        // a block's activations
  static constexpr int kAhead = R ? R : 1, kStages = kAhead + 1;
  static constexpr int kOffX = kWaves * kRing * 2048, kOffS = kOffX + kStages * kStageX;
  static constexpr int kSB = POS == kMaxPos ? 4 : 8;  // blocks whose scales of the positions come together; two such buffers behind the stages
  static constexpr int kGroup = POS * 4 * kSB;
  static constexpr int kLds = kOffS + 2 * kGroup;  // (the epilogues reuse it: UP kPos x 256 B, DOWN 4 x 4 KiB)
};
constexpr int kLds = std::max({Shape<kMaxPos>::kLds, Shape<32, 5>::kLds, Shape<32, 8>::kLds});
static_assert(2 * kLds <= 160 * 1024, "two workgroups a CU");

// Workgroup -> (position tile, group of weight rows): blocks of 2^tl consecutive tiles x 2^nl row groups get consecutive workgroup
// numbers of ONE XCD (numbers x, x + 8, x + 16, ...), so that what they share (a tile's activations, an expert's weights) is fetched
// into that XCD's L2 once. Which blocks: dsgx_moe_prefill and dsgx_dsk_moe_prefill.
struct Map {
  int tl, nl;
};
constexpr Map kMap{3, 2};
// ... with as many row groups as divide NS: a block of fewer groups than the others always falls to the same XCDs where the blocks of a tile
// are 2, 4 or 8 (ten row groups as 8 + 2: four XCDs with four times the others' work; hidden 2560, intermediate 1280, 256 experts, as many groups as nl
// says / this: FP8 T = 200 467 / 386 us, T = 1000 691 / 568, T = 8192 1237 / 1141, MXFP4 T = 4000 501 / 459, INT4 T = 200 337 / 313, T = 4000 989 / 921)
__host__ __device__ inline Map map_of(int tl, int nl, int NS) {
  while (nl > 0 && NS % (1 << nl)) --nl;
  return Map{tl, nl};
}
// ... of a launch with fewer workgroups than CUs: a row group's tiles (up to eight) on one XCD, the row groups over all of them
inline Map map_of_few(int tiles) {
  int tl = 0;
  while (tl < 3 && (1 << tl) < tiles) ++tl;
  return Map{tl, 0};
}
constexpr int kXcds = 8;
__host__ __device__ inline unsigned grid_of(int tiles, int NS, Map m = kMap) {
  const int blocks = ((tiles + (1 << m.tl) - 1) >> m.tl) * ((NS + (1 << m.nl) - 1) >> m.nl);
  return ((unsigned)((blocks + kXcds - 1) / kXcds) * kXcds) << (m.tl + m.nl);
}
// TILE_MINOR: neighbouring workgroup numbers are neighbouring tiles of one row group (the shared expert, whose tiles all stream the same
// weights: in a whole call of 4096 x 2048, 64 experts, T = 2500 827 against 847 us, 256 experts, T = 8192 2762 / 2784; alone no difference); else the row
// groups of one tile (the routed experts' list: 256 experts, T = 5000 / 8192 1977 / 2770 against 2067 / 2852).
template <bool TILE_MINOR>
__device__ __forceinline__ void task_of(int NS, int& tile, int& ns, unsigned wg = blockIdx.x, Map m = kMap) {
  const int x = wg % kXcds, j = wg / kXcds;
  const int b = (j >> (m.tl + m.nl)) * kXcds + x, i = j & ((1 << (m.tl + m.nl)) - 1);
  const int NG = (NS + (1 << m.nl) - 1) >> m.nl;
  tile = ((b / NG) << m.tl) + (TILE_MINOR ? i & ((1 << m.tl) - 1) : i >> m.nl);
  ns = ((b % NG) << m.nl) + (TILE_MINOR ? i >> m.tl : i & ((1 << m.nl) - 1));
}

// The shared expert's side of a launch that holds both its tiles and the routed experts' (k_gemm_mixed): the first `grid`
// workgroups are its tiles' (grid_of of them, so the others keep their XCDs).
struct SharedRows {
  unsigned grid;
  const uint8_t* aq;
  const float* as;
  uint16_t* h;
  uint8_t* hq;
  float* hs;
  float* d;
};
struct Args {
  const uint8_t* aq;   // activations, e4m3 [rows][K]
  const float* as;     // their scales [rows][K / 128]
  const int* gather;   // position -> activation row (null: the position itself)
  const int* tile_e;   // the list of tiles of kMaxPos positions (null: one pseudo-expert -1 holding rows [0, nrows): the shared expert)
  Map map;
  const int* tile_m0;
  const int* ntiles;
  const int* off;
  int nrows;           // the shared expert's rows: T
  int fast_act;        // UP: SwiGLU by the plain formula (swiglu4)
  int deep;            // small tiles take deep rings
  int height;          // k_gemm: rows of a tile
  dsgx_layer_w L;
  uint16_t* h;         // UP: h bf16 [position][I]
  uint8_t* hq;         // UP: h quantised, e4m3 [position][I]
  float* hs;           // UP: its scales [position][I / 128]
  float* d;            // DOWN: f32 [position][H]
  SharedRows sh;       // k_gemm_mixed: the shared expert's rows in the same launch (grid 0: not in it)
#ifdef DSGX_PF_TRACE
  unsigned long long* trace;  // (diagnostic build: thread 0's wall-clock stamps, 8 a workgroup of the routed experts' grid)
#endif
};
#ifdef DSGX_PF_TRACE
#define PF_STAMP(g, k) do { if ((g).trace && threadIdx.x == 0) (g).trace[(size_t)(blockIdx.x - (g).sh.grid) * 8 + (k)] = wall_clock64(); } while (0)
#else
#define PF_STAMP(g, k) do { } while (0)
#endif

// lane l's 16 bytes from `src` to LDS at lds_base + 16 l (lds_base wave-uniform)
__device__ __forceinline__ void dma16(const uint8_t* src, uint32_t lds_base) {
  asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds_base), "v"(src) : "memory");
}
// ... from a wave-uniform address and the lane's offset
__device__ __forceinline__ void dma16(const uint8_t* base, uint32_t off, uint32_t lds_base) {
  asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_base), "v"(off), "s"(base) : "memory");
}
// ... as a streaming load, for what one workgroup of an XCD reads once
__device__ __forceinline__ void dma16_nt(const uint8_t* base, uint32_t off, uint32_t lds_base) {
  asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2 nt" ::"s"(lds_base), "v"(off), "s"(base) : "memory");
}
template <bool STREAM>
__device__ __forceinline__ void dma16_w(const uint8_t* base, uint32_t off, uint32_t lds_base) {
  if constexpr (STREAM) dma16_nt(base, off, lds_base);
  else dma16(base, off, lds_base);
}
// f(0), f(1), ... f(N - 1) as constants (a loop over 40 accumulators with a way out in it is past the size that the compiler unrolls)
template <int... I, class F>
__device__ __forceinline__ void static_for(std::integer_sequence<int, I...>, F f) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F f) {
  static_for(std::make_integer_sequence<int, N>{}, f);
}
template <int N>
__device__ __forceinline__ void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ int swz(int r) { return (r & 7) ^ (r >> 3); }
// Where half h of row r's 32 bytes of scales lies: rows 8-15 exchange their halves, so that sixteen rows' words of one block lie on
// different banks.
__device__ __forceinline__ int sc_half(int r, int h) { return (h ^ (r >> 3)) & 1; }
// the slot of a 64-byte row's piece q is q ^ sw4(row), in the INT4 and MXFP4 kernels (why: pf_gemm_i4.cuh)
__device__ __forceinline__ int sw4(int r) { return (((r >> 2) ^ (r >> 3)) & 1) << 1 | ((r >> 3) & 1); }

// one tile: expert e (-1: the shared expert), rows [m0, mend) of the activations' positions, row group ns
template <bool UP, int POS, int RING, bool STREAM, int R = 0>
__device__ __forceinline__ void gemm_tile(const Args& g, uint8_t* smem, int e, int m0, int mend, int ns) {
  using S = Shape<POS, RING, R>;
  const int K = UP ? g.L.H : g.L.I, KB = K / 128;
  if (mend > m0 + S::kPos) mend = m0 + S::kPos;  // (the tile's own rows)
  const uint8_t *wa, *wb;  // UP: gate, up; DOWN: down twice
  const float *sa, *sb;
  float s2a = 1.f, s2b = 1.f;
  const size_t NK = (size_t)g.L.H * g.L.I;
  if (e < 0) {
    if (UP) wa = g.L.sh.g, sa = g.L.sh.gs, wb = g.L.sh.u, sb = g.L.sh.us;
    else wa = wb = g.L.sh.d, sa = sb = g.L.sh.ds;
  } else {
    const dsgx_mat_desc* d = g.L.desc + (size_t)e * 3;
    if (UP) wa = g.L.pool + d[0].off, wb = g.L.pool + d[1].off, s2a = d[0].s2, s2b = d[1].s2;
    else wa = wb = g.L.pool + d[2].off;
    sa = reinterpret_cast<const float*>(wa + (NK + 255) / 256 * 256);
    sb = reinterpret_cast<const float*>(wb + (NK + 255) / 256 * 256);
  }
  const int tid = threadIdx.x, lane = tid & 63, wave = uni(tid >> 6), r16 = lane & 15, part = lane >> 4;
  // The workgroup's sixteen 16-row tiles, four a wave. UP: tile 2 c is the gate rows, tile 2 c + 1 the up rows of channels
  // c0 + 16 c ... (so a wave's tiles come in gate/up pairs of the same channels); DOWN: tile i is rows r0 + 16 i ...
  const int c0 = ns * (kWgRows / 2), r0 = ns * kWgRows;
  const uint8_t* wt[S::RA];  // the wave's tiles: their first rows
#pragma unroll
  for (int t = 0; t < S::RA; ++t) {
    const int i = S::RA * wave + t;
    wt[t] = UP ? ((i & 1) ? wb : wa) + (size_t)(c0 + 16 * (i >> 1)) * K : wa + (size_t)(r0 + 16 * i) * K;
  }
  const int nmt = uni(min(S::kSub, (mend - m0 + 15) / 16));  // the tile's 16-position tiles that hold rows

  // ---- what this lane fetches: row lr = lane / 8 of an 8-row half, piece (lane % 8) ^ swz(row of the 16) ----
  const int lr = lane >> 3, lq = lane & 7;
  uint32_t ow[2];  // rows 0-7 and 8-15 of a weight tile
#pragma unroll
  for (int hh = 0; hh < 2; ++hh) ow[hh] = (uint32_t)(8 * hh + lr) * K + 16 * (lq ^ swz(8 * hh + lr));
  auto row_of = [&](int p) {  // the activation row of the tile's position p (a ragged tile re-reads its last row: never stored)
    const int pos = min(m0 + p, mend - 1);
    return (uint32_t)(g.gather ? g.gather[pos] : pos);
  };
  uint32_t ox[S::kHX];  // the 8-position half tiles this wave brings (kHX wave, ...)
#pragma unroll
  for (int i = 0; i < S::kHX; ++i) {
    const int p = 8 * (S::kHX * wave + i) + lr;
    ox[i] = row_of(p) * (uint32_t)K + 16 * (lq ^ swz(p & 15));
  }
  constexpr int kPosWave = 8 * S::kHX, kPc = S::kSB / 4;  // the wave's positions, 16-byte pieces of their scales
  const int sp = kPosWave * wave + min(lane / kPc, kPosWave - 1);
  const uint32_t oxs = row_of(sp) * (uint32_t)KB * 4 + (kPc == 2 && KB >= 8 ? 16 * sc_half(sp & 15, lane) : 0);  // lanes 0 .. kPc kPosWave - 1: a piece of a position's scales
  // (the dynamic segment's address inside LDS: the pointer in the LDS address space is that 32-bit offset)
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem;
  // the half tiles this wave brings that hold rows: a ragged tile's others are not fetched (R: they are, so that every wave has as many
  // loads in flight as its waits count)
  const int nhx = R ? S::kHX : uni(min(S::kHX, max(0, (mend - m0 + 7) / 8 - S::kHX * wave)));
  // Weight tile i of the wave's sequence (tile i % 4 of block i / 4, clamped: past the end the last block again, into a slot nobody
  // reads) goes to slot i % kRing of the wave's own ring, whose rows no other wave reads: a slot is free as soon as the wave has read
  // its fragments. Activations: a stage a block.
  const uint32_t ring0 = lds0 + (uint32_t)wave * (S::kRing * 2048);
  auto issue_w = [&](int kb, int t, int slot, int hh) {
    dma16_w<STREAM>(wt[t] + (size_t)min(kb, KB - 1) * 128, ow[hh], uni(ring0 + (uint32_t)slot * 2048 + hh * 1024));
  };
  auto issue_x = [&](int kb) {
    const uint32_t xbase = lds0 + S::kOffX + (uint32_t)(kb % S::kStages) * S::kStageX + (uint32_t)wave * (1024 * S::kHX);
#pragma unroll
    for (int i = 0; i < S::kHX; ++i) {
      if (i >= nhx) break;
      dma16(g.aq + (size_t)min(kb, KB - 1) * 128, ox[i], uni(xbase + i * 1024));
    }
  };
  // The positions' scales come for kSB = 8 blocks at a time, 32 bytes a position, into two buffers (blocks 8 q ... 8 q + 7, the last
  // ones of a row from its end), lane -> position lane / 2, half sc_half(lane); in the widest tile, where LDS is short, for four. A
  // row's scales are one line of L2 for 32 blocks, and that line has left L2 when the next group comes, so it is missed once a group.
  // Rows of fewer than kSB blocks: put in place by hand, their loads in flight together.
  auto first_block = [&](int q) { return min(S::kSB * q, KB - S::kSB); };
  auto issue_scales = [&](int q) {
    if (nhx > 0 && lane < kPc * kPosWave)
      dma16(reinterpret_cast<const uint8_t*>(g.as + first_block(q)), oxs, uni(lds0 + S::kOffS + (uint32_t)(q & 1) * S::kGroup + (uint32_t)wave * (16 * kPc * kPosWave)));
  };
  // The wave's weight scales: lane l holds those of block l; one value
  // a 16-row tile pair (UP: gate and up; DOWN: all of a wave's rows lie in one 128-row block). They are loaded with
  // ordinary loads and WAITED FOR before any of the loads above is issued (the compiler's own wait for them would
  // otherwise count those as well and drain the pipeline). Rows of up to 64 blocks (8192 k), which the host checks.
  const int srow = (UP ? c0 : r0 + 16 * S::RA * wave) / 128;
  const float* swa = sa + (size_t)srow * KB;
  const float* swb = UP ? sb + (size_t)srow * KB : swa;
  PF_STAMP(g, 2);
  float xw[S::kSB - 1];  // (KB < kSB: the positions' scales, on their way with the weights')
  if (KB < S::kSB) {
#pragma unroll
    for (int i = 0; i < S::kSB - 1; ++i) xw[i] = *(const DSGX_GLOBAL float*)(uintptr_t)(reinterpret_cast<const uint8_t*>(g.as + min(i, KB - 1)) + oxs);
  }
  const int kl = min(lane, KB - 1);
  float wsa_l = swa[kl], wsb_l = swb[kl];
  asm volatile("" : "+v"(wsa_l), "+v"(wsb_l));  // (uses that make the compiler place its wait here)
  PF_STAMP(g, 3);
  if (KB < S::kSB && lane < kPc * kPosWave && lane % kPc == 0) {
#pragma unroll
    for (int i = 0; i < S::kSB - 1; ++i) reinterpret_cast<float*>(smem + S::kOffS)[sp * S::kSB + 4 * (kPc == 2 ? sc_half(sp & 15, i >> 2) : 0) + (i & 3)] = xw[i];
  }
  issue_x(0);
  if (KB >= S::kSB) issue_scales(0);
#pragma unroll
  for (int i = 0; i < S::kRing; ++i) {
    if (R && i > 0 && i % 4 == 0) issue_x(i / 4);
    issue_w(i / 4, i % 4, i, 0), issue_w(i / 4, i % 4, i, 1);
  }

  // fragment reads: lane (row r16, part) takes pieces 2 part and 2 part + 1 of its row (32 consecutive k)
  const int rd0 = (r16 >> 3) * 1024 + (r16 & 7) * 128 + ((2 * part) ^ swz(r16)) * 16;
  const int rd1 = (r16 >> 3) * 1024 + (r16 & 7) * 128 + ((2 * part + 1) ^ swz(r16)) * 16;
  auto frag = [&](const uint8_t* t) {
    const u32x4_t lo = *reinterpret_cast<const u32x4_t*>(t + rd0), hi = *reinterpret_cast<const u32x4_t*>(t + rd1);
    return v8i_t{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
  };

  v4f_t acc[S::RA][S::kSub];
#pragma unroll
  for (int t = 0; t < S::RA; ++t)
#pragma unroll
    for (int j = 0; j < S::kSub; ++j) acc[t][j] = v4f_t{0.f, 0.f, 0.f, 0.f};

  auto run = [&](auto nj_c) {
    constexpr int NJ = decltype(nj_c)::value;
    int slot = 0;  // of the block's first weight tile: 4 kb % kRing
    for (int kb = 0; kb < KB; ++kb) {
      // this wave's loads of block kb have landed (weight tiles of later blocks may be in flight; R: all of R - 1 later blocks, a load of
      // scales among them only makes the wait longer); after the barrier everyone's have, and everyone is done reading the stage of
      // block kb - 1, which the activations of block kb + kAhead now overwrite
      wait_loads<R ? (R - 1) * (8 + S::kHX) : 2 * (S::kRing - 4)>();
      __syncthreads();
      if (kb == 0) PF_STAMP(g, 4);
      if ((kb + S::kAhead) % S::kSB == 0 && kb + S::kAhead < KB) issue_scales((kb + S::kAhead) / S::kSB);
      int sl[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) sl[t] = slot + t >= S::kRing ? slot + t - S::kRing : slot + t;
      v8i_t fa[S::RA];
#pragma unroll
      for (int t = 0; t < S::RA; ++t) fa[t] = frag(smem + wave * (S::kRing * 2048) + sl[t] * 2048);
      issue_x(kb + S::kAhead);
      const float wsa = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, wsa_l), kb & 63));
      const float wsb = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, wsb_l), kb & 63));
      const uint8_t* X = smem + S::kOffX + (kb % S::kStages) * S::kStageX;
      const int sw = kb - (KB >= S::kSB ? first_block(kb / S::kSB) : 0);
      const uint8_t* XS = smem + S::kOffS + ((kb / S::kSB) & 1) * S::kGroup + r16 * (4 * S::kSB) + 16 * (kPc == 2 ? sc_half(r16, sw >> 2) : 0) + 4 * (sw & 3);
      v8i_t fn = frag(X);
      float xn = *reinterpret_cast<const float*>(XS);
      asm volatile("" : "+v"(fa[0]), "+v"(fa[1]), "+v"(fa[2]), "+v"(fa[3]));  // (read: their slots may be written from here on)
      static_for<NJ>([&](auto jc) {
        constexpr int j = decltype(jc)::value;
        const v8i_t fb = fn;
        const float xv = xn;
        if (j + 1 < NJ) fn = frag(X + (j + 1) * 2048), xn = *reinterpret_cast<const float*>(XS + (j + 1) * (64 * S::kSB));
#pragma unroll
        for (int i = 0; i < 8; ++i)
          if (i * NJ / 8 == j) issue_w(kb + (S::kRing + i / 2) / 4, (S::kRing + i / 2) % 4, sl[i / 2], i & 1);
        const float s0 = __fmul_rn(xv, wsa), s1 = __fmul_rn(xv, wsb);
#pragma unroll
        for (int t = 0; t < S::RA; ++t) {
          const v4f_t p = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fa[t], fb, v4f_t{0.f, 0.f, 0.f, 0.f}, 0, 0, 0, 0, 0, 0);
          const float sc = (UP && (t & 1)) ? s1 : s0;
#pragma unroll
          for (int q = 0; q < 4; ++q) acc[t][j][q] = fmaf(sc, p[q], acc[t][j][q]);
        }
      });
      slot = slot + 4 >= S::kRing ? slot + 4 - S::kRing : slot + 4;
    }
  };
  auto run_nj = [&](auto self, auto n) {
    constexpr int N = decltype(n)::value;
    if (N == S::kSub || nmt == N) run(n);
    else if constexpr (N < S::kSub) self(self, std::integral_constant<int, N + 1>{});
  };
  run_nj(run_nj, std::integral_constant<int, POS == kMaxPos ? 3 : 1>{});
  wait_loads<0>();   // the trailing loads into unused slots: nothing may still be landing in LDS from here on
  __syncthreads();   // ... in any wave's part of it: the epilogues reuse the stages
  PF_STAMP(g, 5);

  // register q of lane l is weight row 4 (l / 16) + q of the 16-row tile, position l % 16 of the 16 positions
  if (UP) {
    // h = bf16(bf16(silu(bf16 g)) * bf16 u) for the workgroup's 128 channels of every position into an LDS tile
    // [position][256 bytes], 16-byte pieces exchanged by position so that writes and reads spread over the banks; then 16
    // lanes a position: h to memory as whole lines, act_quant over the 128 channels (the scale block of the down
    // projection: amax clamped at 1e-4, scale = amax * f32(1 / 448), e4m3 codes of h / scale clamped to +-448).
    const int I = g.L.I;
    const bool fast = uni(g.fast_act) != 0;
    static_for<S::kSub>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      if (j >= nmt) return;
      const int p = 16 * j + r16;  // position within the tile
#pragma unroll
      for (int b = 0; b < S::RA / 2; ++b) {
        float gv[4], uv[4];
        bf16_round4(acc[2 * b][j], s2a, gv), bf16_round4(acc[2 * b + 1][j], s2b, uv);
        const int ch = 16 * (S::RA / 2 * wave + b) + 4 * part;  // first of the lane's four channels (of the workgroup's 128)
        const int piece = (ch >> 3) ^ (p & 15);
        *reinterpret_cast<uint2*>(smem + p * 256 + piece * 16 + (ch & 4) * 2) = swiglu4(gv, uv, fast);
      }
    });
    __syncthreads();
    const int l16 = tid & 15;
    for (int p = tid >> 4; p < 16 * nmt; p += kThreads4 / 16) {  // (whole rows of 16 lanes take the same turns)
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
      amax = dpp_max<0x141>(amax);
      amax = dpp_max<0x140>(amax);
      amax = fmaxf(amax, 1e-4f);
      const float sc = __fmul_rn(amax, 1.0f / 448.0f), rsc = __builtin_amdgcn_rcpf(sc);
      float qv[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) qv[i] = fminf(448.f, fmaxf(-448.f, div_by(v[i], sc, rsc)));
      uint32_t o0 = __builtin_amdgcn_cvt_pk_fp8_f32(qv[0], qv[1], 0, false), o1 = __builtin_amdgcn_cvt_pk_fp8_f32(qv[4], qv[5], 0, false);
      o0 = __builtin_amdgcn_cvt_pk_fp8_f32(qv[2], qv[3], o0, true), o1 = __builtin_amdgcn_cvt_pk_fp8_f32(qv[6], qv[7], o1, true);
      if (pos < mend) {
        __builtin_nontemporal_store(hv, reinterpret_cast<u32x4_t*>(g.h + (size_t)pos * I + c0 + 8 * l16));
        *reinterpret_cast<uint2*>(g.hq + (size_t)pos * I + c0 + 8 * l16) = make_uint2(o0, o1);
        if (l16 == 0) g.hs[(size_t)pos * (I / 128) + ns] = sc;
      }
    }
  } else {
    // the wave's 16 positions x 64 rows of one 16-position tile at a time through its own piece of LDS (4 KiB):
    // written as held, read back as whole rows, 16 lanes a position. Streaming stores, here and of h above, which only a caller's view reads: a
    // chunk's d is 26 MB to 1 GB that would push the weights out of L2 (T = 700 / 1500 / 3000 / 8192 1202 / 1374 / 1682 / 2833 -> 1178 / 1332 / 1652 /
    // 2810 us; MXFP4 T = 3000 1467 -> 1452, its h as well: no change).
    const int H = g.L.H;
    uint8_t* my = smem + wave * 4096;
    const int row0 = r0 + 16 * S::RA * wave;
    static_for<S::kSub>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      if (j >= nmt) return;
#pragma unroll
      for (int t = 0; t < S::RA; ++t) {
        const int c = 4 * t + part;  // the 16-byte piece: rows 16 t + 4 part ...
        *reinterpret_cast<v4f_t*>(my + r16 * 256 + ((c & ~7) | ((c ^ r16) & 7)) * 16) = acc[t][j];
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int p = 4 * i + part, c = r16;
        const v4f_t v = *reinterpret_cast<const v4f_t*>(my + p * 256 + ((c & ~7) | ((c ^ p) & 7)) * 16);
        const int pos = m0 + 16 * j + p;
        if (pos < mend) __builtin_nontemporal_store(v, reinterpret_cast<v4f_t*>(g.d + (size_t)pos * H + row0 + 4 * c));
      }
    });
  }
  PF_STAMP(g, 6);
}

// A tile in the shape that its rows take. `only`: it is its expert's only one. Nobody else reads its weights then, and as streaming loads they
// leave what others share (activations, scales) in L2: T = 20 / 60 / 200 / 700 / 1500 345 / 590 / 964 / 1241 / 1380 -> 316 / 552 / 900 / 1199 /
// 1373 us; a remainder's weights as well, T = 8192 2825 -> 2880, and the widest tiles' too, T = 200 929, T = 8192 3400.
template <bool UP>
__device__ __forceinline__ void any_tile(const Args& g, uint8_t* smem, int e, int m0, int mend, int ns, bool only) {
  if (mend - m0 > 32) gemm_tile<UP, kMaxPos, 4, false>(g, smem, e, m0, mend, ns);
  else if (g.deep) gemm_tile<UP, 32, 8, true>(g, smem, e, m0, mend, ns);
  else if (only) gemm_tile<UP, 32, 5, true>(g, smem, e, m0, mend, ns);
  else gemm_tile<UP, 32, 5, false>(g, smem, e, m0, mend, ns);
}
// The shared expert alone: tiles of g.height rows (up to kMaxPos) over [0, nrows).
template <bool UP>
__global__ void __launch_bounds__(kThreads4, 2) k_gemm(Args g) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const int NS = UP ? g.L.I / (kWgRows / 2) : g.L.H / kWgRows;
  int tile, ns;
  task_of<true>(NS, tile, ns, blockIdx.x, g.map);
  const int m0 = tile * g.height;
  if (ns >= NS || m0 >= g.nrows) return;
  any_tile<UP>(g, smem, -1, m0, min(g.nrows, m0 + g.height), ns, false);
}
// ... in no more tiles than the chip has CUs: one workgroup a CU, which has the CU's LDS for loads in flight (Shape's R). A launch of few
// workgroups waits for its loads' latency, turn after turn (0.47 us a block with four blocks ahead).
template <bool UP, int POS, int R>
__global__ void __launch_bounds__(kThreads4, 2) k_few(Args g) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const int NS = UP ? g.L.I / (kWgRows / 2) : g.L.H / kWgRows;
  int tile, ns;
  task_of<true>(NS, tile, ns, blockIdx.x, g.map);
  if (ns >= NS || tile * POS >= g.nrows) return;
  gemm_tile<UP, POS, 4 * R, false, R>(g, smem, -1, tile * POS, g.nrows, ns);
}
// The routed experts' list, an expert's tiles next to each other, behind the shared expert's tiles.
template <bool UP>
__global__ void __launch_bounds__(kThreads4, 2) k_gemm_mixed(Args g) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const int NS = UP ? g.L.I / (kWgRows / 2) : g.L.H / kWgRows;
  int tile, ns;
  if (blockIdx.x < g.sh.grid) {  // (the same for the whole workgroup)
    task_of<true>(NS, tile, ns, blockIdx.x, g.map);
    const int m0 = tile * kMaxPos, mend = g.nrows;
    if (ns >= NS || m0 >= mend) return;
    Args q = g;
#ifdef DSGX_PF_TRACE
    q.trace = nullptr;
#endif
    q.aq = g.sh.aq, q.as = g.sh.as, q.gather = nullptr, q.h = g.sh.h, q.hq = g.sh.hq, q.hs = g.sh.hs, q.d = g.sh.d;
    any_tile<UP>(q, smem, -1, m0, mend, ns, tile == 0);
    return;
  }
  PF_STAMP(g, 0);
  task_of<false>(NS, tile, ns, blockIdx.x - g.sh.grid, g.map);
  if (ns >= NS || tile >= *g.ntiles) return;
  const int e = g.tile_e[tile];
  const int m0 = g.off[e] + g.tile_m0[tile], mend = g.off[e + 1];
  if (m0 >= 0) PF_STAMP(g, 1);
#ifdef DSGX_PF_TRACE
  if (g.trace && threadIdx.x == 0) g.trace[(size_t)(blockIdx.x - g.sh.grid) * 8 + 7] = min(mend - m0, kMaxPos);
#endif
  any_tile<UP>(g, smem, e, m0, mend, ns, g.tile_m0[tile] == 0);
}

}  // namespace pf8
}  // namespace dsgx
