// The BF16 shared expert of an INT4 layer's prefill step: dense GEMMs of bf16 rows against stored bf16 weights (gate and up
// interleaved in one matrix, row 2 c gate and 2 c + 1 up of channel c; altar1-4xgx10-switchless/engine/experts/prefill.cu:
// 337-352 of the reference), summed in f32 by v_mfma_f32_16x16x32_bf16.
//
// Staged as pf_gemm_fp8.cuh's 128-position tiles: 64 k of bf16 are the 128 bytes a row that 128 k of e4m3 are. A workgroup (8
// waves) computes up to 128 positions against 256 weight rows (UP: the gate and up rows of 128 channels), a wave 32 rows x every
// position; three stages of 64 k, both operands by global_load_lds, a turn's six loads a wave between its MFMAs. Piece c of row
// r lies at slot c ^ (r % 8): the lane (row, part) of MFMA j reads piece 4 j + part, k = 32 j + 8 part + [0, 8), and a
// 16-byte read is served rows 0-3 and 12-15 of one part beside rows 4-11 of the next, whose pieces differ in bit 0.
// A whole step runs these tiles in the routed experts' launches (pfi4::k_gemm), in front of them: as launches of their own they are
// 16 and 24 workgroups a 128 rows, most of the chip idle. Hidden 6144, intermediate 2048, 168 experts: the two launches took
// 178 + 124 us of 1660 at T = 1111 with the register-ring kernel that they had (219 us at T = 336; these, alone, 108), the call
// now takes 1590; hidden 3840, intermediate 768, 16 experts, T = 200: 244 -> 134.
#pragma once
#include "pf_gemm_fp8.cuh"

namespace dsgx {
namespace pfb16 {

using pf8::dma16;
using pf8::kThreads;
using pf8::kWgRows;
using pf8::v4f_t;
using pf8::wait_loads;
typedef __bf16 v8bf_t __attribute__((ext_vector_type(8)));

constexpr int kPos = 128, kStages = 3, kLoads = 6;  // a wave's loads a turn: four of its weight rows, two of its 16 positions
constexpr int kStageW = kWgRows * 128, kStageBytes = kStageW + kPos * 128;
constexpr int kLds = kStages * kStageBytes;  // 147,456

struct Args {
  const uint16_t* x;  // bf16 [rows][K]
  const uint8_t* w;   // bf16; UP: [2 I][H] interleaved; DOWN: [H][I]
  int rows, H, I;
  uint16_t* h;        // UP: bf16 [rows][I]
  float* d;           // DOWN: f32 [rows][H]
};

// The epilogues of a 32-row x 128-position wave tile, shared with the INT4 experts' kernel: register q of lane l is weight row 4
// (l / 16) + q of the 16-row tile, position l % 16 of the 16 positions.
// UP (acc[0] gate, acc[1] up of channels 16 wave ... of the workgroup's 128): h = bf16(bf16(silu(bf16 g)) * bf16 u) into an LDS tile
// [position][256 bytes] (16-byte pieces exchanged by position: writes and reads spread over the banks), then whole lines to
// memory, 16 lanes a position
__device__ __forceinline__ void store_h(uint8_t* smem, const v4f_t (&acc)[2][8], int nmt, float s2a, float s2b, int m0, int mend, int c0, int I, uint16_t* h) {
  const int tid = threadIdx.x, lane = tid & 63, wave = uni(tid >> 6), r16 = lane & 15, part = lane >> 4;
#pragma unroll
  for (int mt = 0; mt < 8; ++mt) {
    if (mt >= nmt) break;
    const int p = 16 * mt + r16;
    float gv[4], uv[4];
    bf16_round4(acc[0][mt], s2a, gv), bf16_round4(acc[1][mt], s2b, uv);
    const int ch = 16 * wave + 4 * part;
    const int piece = (ch >> 3) ^ (p & 15);
    *reinterpret_cast<uint2*>(smem + p * 256 + piece * 16 + (ch & 4) * 2) = swiglu4(gv, uv, false);
  }
  __syncthreads();
  const int l16 = tid & 15;
  for (int p = tid >> 4; p < 16 * nmt; p += kThreads / 16) {
    const int pos = m0 + p;
    const u32x4_t hv = *reinterpret_cast<const u32x4_t*>(smem + p * 256 + (l16 ^ (p & 15)) * 16);
    if (pos < mend) *reinterpret_cast<u32x4_t*>(h + (size_t)pos * I + c0 + 8 * l16) = hv;
  }
}
// DOWN: a 16-position tile at a time through the wave's own 2 KiB: written as held (four rows of a position: 16 bytes), read back
// as whole rows (32 rows = 128 bytes a position, 8 lanes a position)
__device__ __forceinline__ void store_d(uint8_t* smem, const v4f_t (&acc)[2][8], int nmt, int m0, int mend, int r0, int H, float* d) {
  const int tid = threadIdx.x, lane = tid & 63, wave = uni(tid >> 6), r16 = lane & 15, part = lane >> 4;
  uint8_t* my = smem + wave * 2048;
  const int row0 = r0 + 32 * wave;
#pragma unroll
  for (int mt = 0; mt < 8; ++mt) {
    if (mt >= nmt) break;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int c = 4 * t + part;
      *reinterpret_cast<v4f_t*>(my + r16 * 128 + ((c ^ r16) & 7) * 16) = acc[t][mt];
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int idx = i * 64 + lane, p = idx >> 3, c = idx & 7;
      const v4f_t v = *reinterpret_cast<const v4f_t*>(my + p * 128 + ((c ^ p) & 7) * 16);
      const int pos = m0 + 16 * mt + p;
      if (pos < mend) *reinterpret_cast<v4f_t*>(d + (size_t)pos * H + row0 + 4 * c) = v;
    }
  }
}

// rows [m0, mend) against row group ns
template <bool UP>
__device__ __forceinline__ void gemm_tile(const Args& g, uint8_t* smem, int m0, int mend, int ns) {
  const int K = UP ? g.H : g.I, TN = K / 64;
  if (mend > m0 + kPos) mend = m0 + kPos;
  const int tid = threadIdx.x, lane = tid & 63, wave = uni(tid >> 6), r16 = lane & 15, part = lane >> 4;
  const int nmt = uni((mend - m0 + 15) / 16);
  // what this lane fetches: row lane / 8 of an 8-row half, piece (lane % 8) ^ (row % 8). The wave's two 16-row tiles: UP the
  // gate rows and the up rows of channels 128 ns + 16 wave ...; DOWN rows 256 ns + 32 wave + 16 t ...
  const int lr = lane >> 3, lp = 16 * ((lane & 7) ^ lr);
  const uint8_t* pw = g.w + (size_t)(kWgRows * ns + 32 * wave + (UP ? 2 : 1) * lr) * K * 2 + lp;
  const size_t tile1 = (size_t)(UP ? 1 : 16) * K * 2, half1 = (size_t)(UP ? 16 : 8) * K * 2;  // bytes to the second tile, to a tile's second half
  const uint8_t* px[2];
#pragma unroll
  for (int hh = 0; hh < 2; ++hh)  // (a ragged tile re-reads its last row: never stored)
    px[hh] = reinterpret_cast<const uint8_t*>(g.x) + (size_t)min(m0 + 16 * wave + 8 * hh + lr, mend - 1) * K * 2 + lp;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem;
  // load i of turn t (past the end: the last turn's again, into a stage nobody reads): the activations, then the weights
  auto issue_one = [&](int t, int i) {
    const size_t off = (size_t)min(t, TN - 1) * 128;
    const uint32_t st = lds0 + (uint32_t)(t % kStages) * kStageBytes;
    if (i < 2) dma16(px[i] + off, uni(st + kStageW + (uint32_t)wave * 2048 + i * 1024));
    else dma16(pw + ((i - 2) >> 1) * tile1 + (i & 1) * half1 + off, uni(st + (uint32_t)wave * 4096 + (i - 2) * 1024));
  };
#pragma unroll
  for (int s = 0; s + 1 < kStages; ++s)
#pragma unroll
    for (int i = 0; i < kLoads; ++i) issue_one(s, i);
  int rd[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) rd[j] = r16 * 128 + ((4 * j + part) ^ (r16 & 7)) * 16;
  v4f_t acc[2][8];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[t][j] = v4f_t{0.f, 0.f, 0.f, 0.f};

  auto run = [&](auto nj_c) {
    constexpr int NJ = decltype(nj_c)::value;
    for (int t = 0; t < TN; ++t) {
      wait_loads<(kStages - 2) * kLoads>();
      __syncthreads();
      const uint8_t* W = smem + (size_t)(t % kStages) * kStageBytes + wave * 4096;
      const uint8_t* X = smem + (size_t)(t % kStages) * kStageBytes + kStageW;
      u32x4_t fa[2][2];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) fa[i][j] = *reinterpret_cast<const u32x4_t*>(W + i * 2048 + rd[j]);
#pragma unroll
      for (int mt = 0; mt < NJ; ++mt) {
        u32x4_t fb[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) fb[j] = *reinterpret_cast<const u32x4_t*>(X + mt * 2048 + rd[j]);
#pragma unroll
        for (int i = 0; i < kLoads; ++i)
          if (i * NJ / kLoads == mt) issue_one(t + kStages - 1, i);
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int i = 0; i < 2; ++i)
            acc[i][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf_t, fa[i][j]), __builtin_bit_cast(v8bf_t, fb[j]), acc[i][mt], 0, 0, 0);
      }
    }
  };
  if (nmt <= 1) run(std::integral_constant<int, 1>{});
  else if (nmt <= 2) run(std::integral_constant<int, 2>{});
  else if (nmt <= 4) run(std::integral_constant<int, 4>{});
  else run(std::integral_constant<int, 8>{});
  wait_loads<0>();
  __syncthreads();
  if (UP) store_h(smem, acc, nmt, 1.f, 1.f, m0, mend, ns * (kWgRows / 2), g.I, g.h);
  else store_d(smem, acc, nmt, m0, mend, ns * kWgRows, g.H, g.d);
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
__global__ void __launch_bounds__(kThreads) k_gemm(Args g) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  tiles<UP>(g, smem, blockIdx.x);
}

}  // namespace pfb16
}  // namespace dsgx
