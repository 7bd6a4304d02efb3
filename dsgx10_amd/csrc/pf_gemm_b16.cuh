// The BF16 shared expert of an INT4 layer's prefill step: dense GEMMs of bf16 rows against stored bf16 weights (gate and up
// interleaved in one matrix, row 2 c gate and 2 c + 1 up of channel c; altar1-4xgx10-switchless/engine/experts/prefill.cu:
// 337-352 of the reference), summed in f32 by v_mfma_f32_32x32x16_bf16.
//
// Staged as pf_gemm_fp8.cuh's tiles: 64 k of bf16 are the 128 bytes a row that 128 k of e4m3 are. A workgroup (4 waves, two
// workgroups a CU) computes up to 128 positions against 256 weight rows (UP: the gate and up rows of 128 channels), a wave 64 rows
// x every position; two stages of the positions' 64 k, a ring of the wave's own for its weights (tiles of 16 rows), whose slots are free
// when their fragments are read; both operands by global_load_lds, the weights' loads between a turn's MFMAs. Piece c of row
// r lies at slot c ^ (r / 2 % 8): a 16-byte read is served sixteen lanes at a time (pf_gemm_i4.cuh), rows 0-3, 12-15, 20-27 of a tile or the
// others, and the even rows of either set (and the odd ones) go to eight slots one-to-one.
// The sums' order: the 32 x 32 x 16 instruction adds the eight products of a lane's registers as one group and the two halves' groups
// to the accumulator one after the other, the 16 x 16 x 32 one its four parts' in the same way, so two of the former (k = 16 s + 8 half)
// are one of the latter (k = 8 part), bit for bit; and the former leaves the vector unit more of its issue slots (a loop with three
// vector instructions a 16 x 16 x 32's worth: 17.6 against 23.1 clocks, without any 16.4 against 17.9).
// A whole step runs these tiles in the routed experts' launches (pfi4::k_gemm), in front of them: as launches of their own (k_few, k_gemm) they
// are 16 and 24 workgroups a 128 rows, most of the chip idle. (Hidden 6144, intermediate 2048, 168 experts, kernels of eight waves, T = 1111:
// 1660 -> 1590 us; hidden 3840, intermediate 768, 16 experts, T = 200: 244 -> 134.)
#pragma once
#include "pf_gemm_fp8.cuh"

namespace dsgx {
namespace pfb16 {

using pf8::dma16;
using pf8::kThreads4;
using pf8::kWaves;
using pf8::kWgRows;
using pf8::v4f_t;
using pf8::wait_loads;
typedef __bf16 v8bf_t __attribute__((ext_vector_type(8)));
typedef float v16f_t __attribute__((ext_vector_type(16)));

constexpr int kPos = 128;
// The waves' rings of weight tiles, 2 KiB each, and the stages of activations. R > 0: for one workgroup a CU (k_few), both R turns ahead.
template <int POS = kPos, int R = 0>
struct Shape {
  static constexpr int kRing = R ? 4 * R : 5, kAhead = R ? R : 1, kStages = kAhead + 1;
  static constexpr int kStageX = POS * 128, kOffX = kWaves * kRing * 2048;
  static constexpr int kLds = kOffX + kStages * kStageX;
};
constexpr int kLds = Shape<>::kLds;  // 73,728
static_assert(2 * kLds <= 160 * 1024, "two workgroups a CU");

struct Args {
  const uint16_t* x;  // bf16 [rows][K]
  const uint8_t* w;   // bf16; UP: [2 I][H] interleaved; DOWN: [H][I]
  int rows, H, I;
  uint16_t* h;        // UP: bf16 [rows][I]
  float* d;           // DOWN: f32 [rows][H]
};

// The accumulators of a wave's 64 rows x MT NS positions, by tiles of MT rows x MT positions of v_mfma_f32_16x16x32_bf16 or 32x32x16, and the
// four consecutive rows `u` that a lane holds of a tile (MT = 16: one such four): rows 4 (l / 16), or 8 u + 4 (l / 32), position l % MT
template <int MT>
using acc_t = std::conditional_t<MT == 16, v4f_t, v16f_t>;
template <int MT>
__device__ __forceinline__ v4f_t four(const acc_t<MT>& a, int u) {
  if constexpr (MT == 16) return a;
  else return v4f_t{a[4 * u], a[4 * u + 1], a[4 * u + 2], a[4 * u + 3]};
}
// The epilogues, shared with the INT4 experts' kernel.
// UP (tiles t even gate, t odd up of channels 32 wave + MT (t / 2) ... of the workgroup's 128): h = bf16(bf16(silu(bf16 g)) * bf16 u) into an
// LDS tile [position][256 bytes] (16-byte pieces exchanged by position: writes and reads spread over the banks), then whole lines to
// memory, 16 lanes a position
template <int MT, int NS>
__device__ __forceinline__ void store_h(uint8_t* smem, const acc_t<MT> (&acc)[64 / MT][NS], float s2a, float s2b, int m0, int mend, int c0, int I, uint16_t* h) {
  const int tid = threadIdx.x, lane = tid & 63, wave = uni(tid >> 6);
  pf8::static_for<NS>([&](auto jc) {
    constexpr int pt = decltype(jc)::value;
    if (m0 + MT * pt >= mend) return;
    const int p = MT * pt + lane % MT;
    pf8::static_for<MT == 16 ? 2 : 4>([&](auto uc) {
      constexpr int u = decltype(uc)::value, t = MT == 16 ? 2 * u : 0;
      float gv[4], uv[4];
      bf16_round4(four<MT>(acc[t][pt], u), s2a, gv), bf16_round4(four<MT>(acc[t + 1][pt], u), s2b, uv);
      const int ch = 32 * wave + (MT == 16 ? 16 : 8) * u + 4 * (lane / MT);  // first of the lane's four channels (of the workgroup's 128)
      *reinterpret_cast<uint2*>(smem + p * 256 + ((ch >> 3) ^ (p & 15)) * 16 + (ch & 4) * 2) = swiglu4(gv, uv, false);
    });
  });
  __syncthreads();
  const int l16 = tid & 15;
  for (int pos = m0 + (tid >> 4); pos < mend; pos += kThreads4 / 16) {
    const int p = pos - m0;
    *reinterpret_cast<u32x4_t*>(h + (size_t)pos * I + c0 + 8 * l16) = *reinterpret_cast<const u32x4_t*>(smem + p * 256 + (l16 ^ (p & 15)) * 16);
  }
}
// DOWN: MT positions at a time through the wave's own MT x 256 bytes: written as held (four rows of a position: 16 bytes), read back
// as whole rows (64 rows = 256 bytes a position, 16 lanes a position)
template <int MT, int NS>
__device__ __forceinline__ void store_d(uint8_t* smem, const acc_t<MT> (&acc)[64 / MT][NS], int m0, int mend, int r0, int H, float* d) {
  const int tid = threadIdx.x, lane = tid & 63, wave = uni(tid >> 6), r = lane % MT;
  uint8_t* my = smem + wave * (MT * 256);
  const int row0 = r0 + 64 * wave;
  pf8::static_for<NS>([&](auto jc) {
    constexpr int pt = decltype(jc)::value;
    if (m0 + MT * pt >= mend) return;
#pragma unroll
    for (int t = 0; t < 64 / MT; ++t)
#pragma unroll
      for (int u = 0; u < (MT == 16 ? 1 : 4); ++u) {
        const int c = MT / 4 * t + 2 * u + lane / MT;  // the 16-byte piece: rows 4 c ...
        *reinterpret_cast<v4f_t*>(my + r * 256 + (c ^ (r & 15)) * 16) = four<MT>(acc[t][pt], u);
      }
#pragma unroll
    for (int i = 0; i < MT / 4; ++i) {
      const int p = 4 * i + (lane >> 4), c = lane & 15;
      const v4f_t v = *reinterpret_cast<const v4f_t*>(my + p * 256 + (c ^ (p & 15)) * 16);
      const int pos = m0 + MT * pt + p;
      if (pos < mend) __builtin_nontemporal_store(v, reinterpret_cast<v4f_t*>(d + (size_t)pos * H + row0 + 4 * c));
    }
  });
}

// rows [m0, mend) against row group ns
template <bool UP, int POS = kPos, int R = 0>
__device__ __forceinline__ void gemm_tile(const Args& g, uint8_t* smem, int m0, int mend, int ns) {
  using S = Shape<POS, R>;
  constexpr int kRing = S::kRing, kStageX = S::kStageX, kOffX = S::kOffX, kXL = POS / 32;  // kXL: a wave's loads of a stage of activations
  const int K = UP ? g.H : g.I, TN = K / 64;
  if (mend > m0 + POS) mend = m0 + POS;
  const int tid = threadIdx.x, lane = tid & 63, wave = uni(tid >> 6), r32 = lane & 31, half = lane >> 5;
  const int npt = uni((mend - m0 + 31) / 32);
  // what this lane fetches: row lane / 8 of eight, slot lane % 8. The wave's four 16-row tiles: UP the gate rows (t < 2) and
  // the up rows of channels 128 ns + 32 wave + 16 (t % 2) ...; DOWN rows 256 ns + 64 wave + 16 t ...
  const int lr = lane >> 3;
  const uint8_t* wt[4];
  uint32_t ow[2];
#pragma unroll
  for (int t = 0; t < 4; ++t) wt[t] = g.w + (size_t)(kWgRows * ns + 64 * wave + (UP ? 32 * (t & 1) + (t >> 1) : 16 * t)) * K * 2;
#pragma unroll
  for (int hh = 0; hh < 2; ++hh) ow[hh] = (uint32_t)(8 * hh + lr) * (UP ? 4 : 2) * K + 16 * ((lane & 7) ^ (4 * hh + (lane >> 4)));
  const uint8_t* px[kXL];  // positions 8 (wave + 4 i) ...
#pragma unroll
  for (int i = 0; i < kXL; ++i)  // (a ragged tile re-reads its last row: never stored)
    px[i] = reinterpret_cast<const uint8_t*>(g.x) + (size_t)min(m0 + 8 * (wave + 4 * i) + lr, mend - 1) * K * 2 + 16 * ((lane & 7) ^ (4 * (wave & 1) + (lane >> 4)));
  // ... and its empty eights are not fetched (R: they are, so that every wave has as many loads in flight as its waits count)
  const int nhx = R ? kXL : uni(min(kXL, max(0, ((mend - m0 + 7) / 8 - wave + 3) / 4)));
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem;
  // (past the end: the last turn's again, into slots nobody reads)
  auto issue_x = [&](int t) {
    const size_t off = (size_t)min(t, TN - 1) * 128;
#pragma unroll
    for (int i = 0; i < kXL; ++i) {
      if (i >= nhx) break;
      dma16(px[i] + off, uni(lds0 + kOffX + (uint32_t)(t % S::kStages) * kStageX + (uint32_t)(wave + 4 * i) * 1024));
    }
  };
  auto issue_w = [&](int t, int tile, int slot, int hh) {  // half hh of the tile
    dma16(wt[tile] + (size_t)min(t, TN - 1) * 128, ow[hh], uni(lds0 + (uint32_t)wave * (kRing * 2048) + (uint32_t)slot * 2048 + hh * 1024));
  };
  issue_x(0);
#pragma unroll
  for (int i = 0; i < kRing; ++i) {
    if (R && i > 0 && i % 4 == 0) issue_x(i / 4);
    issue_w(i / 4, i % 4, i, 0), issue_w(i / 4, i % 4, i, 1);
  }
  const int rd = (half ^ ((r32 >> 1) & 7)) * 16;  // (step s: ^ 32 s)
  v16f_t acc[2][POS / 32];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int j = 0; j < POS / 32; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[t][j][r] = 0.f;

  auto run = [&](auto nj_c) {
    constexpr int NJ = decltype(nj_c)::value;
    int slot = 0;  // of the turn's first weight tile: 4 t % kRing
    for (int t = 0; t < TN; ++t) {
      wait_loads<R ? (R - 1) * (8 + kXL) : 2 * (kRing - 4)>();  // (the next turn's first tiles may be in flight, or all of R - 1 turns)
      __syncthreads();
      int sl[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) sl[i] = slot + i >= kRing ? slot + i - kRing : slot + i;
      const uint8_t* X = smem + kOffX + (t % S::kStages) * kStageX + r32 * 128;
      u32x4_t fa[2][4], fn;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const uint8_t* W = smem + wave * (kRing * 2048) + (sl[2 * i] + (r32 >> 4) * (sl[2 * i + 1] - sl[2 * i])) * 2048 + (r32 & 15) * 128;
#pragma unroll
        for (int s = 0; s < 4; ++s) fa[i][s] = *reinterpret_cast<const u32x4_t*>(W + (rd ^ (32 * s)));
      }
      issue_x(t + S::kAhead);
      fn = *reinterpret_cast<const u32x4_t*>(X + rd);
#pragma unroll
      for (int i = 0; i < 2; ++i) asm volatile("" : "+v"(fa[i][0]), "+v"(fa[i][1]), "+v"(fa[i][2]), "+v"(fa[i][3]));  // (read: their slots may be written from here on)
      pf8::static_for<4 * NJ>([&](auto jc) {
        constexpr int n = decltype(jc)::value, pt = n >> 2, s = n & 3;
        const u32x4_t fb = fn;
        if constexpr (n + 1 < 4 * NJ) fn = *reinterpret_cast<const u32x4_t*>(X + ((n + 1) >> 2) * 4096 + (rd ^ (32 * ((n + 1) & 3))));
#pragma unroll
        for (int i = 0; i < 8; ++i)
          if (i * 4 * NJ / 8 == n) issue_w(t + (kRing + i / 2) / 4, (kRing + i / 2) % 4, sl[i / 2], i & 1);
#pragma unroll
        for (int i = 0; i < 2; ++i)
          acc[i][pt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf_t, fa[i][s]), __builtin_bit_cast(v8bf_t, fb), acc[i][pt], 0, 0, 0);
      });
      slot = slot + 4 >= kRing ? slot + 4 - kRing : slot + 4;
    }
  };
  if (POS == 32 || npt <= 1) run(std::integral_constant<int, 1>{});
  else if (POS == 64 || npt <= 2) run(std::integral_constant<int, std::min(2, POS / 32)>{});
  else if (R && npt <= 3) run(std::integral_constant<int, std::min(3, POS / 32)>{});
  else run(std::integral_constant<int, POS / 32>{});
  wait_loads<0>();
  __syncthreads();
  if (UP) store_h<32>(smem, acc, 1.f, 1.f, m0, mend, ns * (kWgRows / 2), g.I, g.h);
  else store_d<32>(smem, acc, m0, mend, ns * kWgRows, g.H, g.d);
}

// workgroup wg of the grid_of(ceil(rows / 128), row groups) that hold the rows
template <bool UP>
__device__ __forceinline__ void tiles(const Args& g, uint8_t* smem, unsigned wg) {
  const int NS = UP ? g.I / (kWgRows / 2) : g.H / kWgRows;
  int tile, ns;
  pf8::task_of<true>(NS, tile, ns, wg);
  if (ns >= NS || tile * kPos >= g.rows) return;
  gemm_tile<UP>(g, smem, tile * kPos, g.rows, ns);
}
template <bool UP>
__global__ void __launch_bounds__(kThreads4, 2) k_gemm(Args g) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  tiles<UP>(g, smem, blockIdx.x);
}
// The rows in no more tiles than the chip has CUs: one workgroup a CU, which has the CU's LDS for loads in flight.
template <bool UP, int POS, int R>
__global__ void __launch_bounds__(kThreads4, 2) k_few(Args g, pf8::Map map, int height) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const int NS = UP ? g.I / (kWgRows / 2) : g.H / kWgRows;
  int tile, ns;
  pf8::task_of<true>(NS, tile, ns, blockIdx.x, map);
  const int m0 = tile * height;
  if (ns >= NS || m0 >= g.rows) return;
  gemm_tile<UP, POS, R>(g, smem, m0, min(g.rows, m0 + height), ns);
}

}  // namespace pfb16
}  // namespace dsgx
