// Dense GEMV for 1-16 activation rows over FP8-128x128, INT4-g32 and BF16 weights: the gfx950 counterpart of the
// reference's glm::gemv (altar1-4xgx10-switchless/engine/attn/gemv.cu:173-333, attn.h:59-123).
//
//   y[r][n] = sum_k x[r][k] W[n][k], f32 accumulation, outputs bf16 / f32 / SwiGLU (gemv.cu:138-170).
//   FP8: per 128-k block the unscaled f32 sum, then acc = fma(S, sum, acc) (gemv.cu:230-244, micro/gemv.cu:512);
//   INT4: W = bf16_rne((u - u_z) s) per element in registers (attn_common.cuh:65-76), then as BF16.
//
// One wavefront owns RB rows of W and the whole of K (rowdot.cuh); the grid is sized to the chip and walks the row
// batches round-robin. The order of the adds inside a dot product is not the reference's (not part of its contract).
#include "abi_internal.h"
#include "addnorm.cuh"
#include "rowdot.cuh"

namespace dsgx {
namespace {

constexpr int kMaxSegs = 4;  // attn.h:94
struct GemvSegDev {
  MatDev m;
  void* y;
  int n, ldy, row0;
};
struct GemvArgs {
  const uint16_t* x;
  int ldx, K, nq, nsegk, nsegs, total_rows, out, splitk;
  GemvSegDev sg[kMaxSegs];
  NormIn norm;  // norm.part set: the rows are not read from x but made here, xn = RMSNorm(bf16(res + part)) (dsgx_add_norm_gemv)
};

// The activation rows into LDS: from x, or (fused add + norm) computed by this workgroup from the partial sums and the
// residual - every workgroup makes all M rows for itself (M H values: a few KB from L2), workgroup 0 also writes the new
// residual and the normed rows to memory for the kernels that follow.
// (add_norm_rows is 256 threads' work: a workgroup of another size, NORM false, has no code for it.)
template <int KL, int M, bool NORM>
__device__ __forceinline__ void stage_rows(uint4* xs, const GemvArgs& a, float* red) {
  if (!NORM || !a.norm.part) {
    stage_x<KL>(xs, a.x, a.ldx, M, a.K, a.nq * 8);
    return;
  }
  add_norm_rows<M>(a.norm, 0, a.K, xs, red, true, blockIdx.x == 0, [&](int m, int q) { return (size_t)m * a.nq + xchunk_index<KL>(q); });
}

// the lanes of a row's last segment that lie inside K
template <int FMT>
__device__ __forceinline__ int last_seg_lanes(int K, int nsegk) { return (K - (nsegk - 1) * FmtT<FMT>::SEGK + FmtT<FMT>::KL - 1) / FmtT<FMT>::KL; }

// A slice of a batch's rows (segments seg0, seg0 + sk, ...) by the INT4 routine for every scale, for the waves of k_gemv whose faster one
// has met a scale of 2^116 or more (none in a checkpoint). The loop only keeps the largest (and these lines stand once, behind it: as part of
// every step's code they made a call's first pass 10 us longer): 6144 x 16384 at 1 / 2 / 4 rows 17.9 / 19.7 / 24.1 ->
// 17.2 / 19.1 / 23.3 us a call, 16384 x 2048 at one 9.2 -> 8.6 (a vote and both routines in every step were 4% slower than the long one alone).
// k_gemv_sk's calls are over before it pays (768 x 6144 over 4 at one row 6.2 -> 6.45). Nor where one wave walks the slices of eight rows
// (SPLIT, M = 8): there the largest scale and the code of the second pass are registers past 128 (136; 120 with the long routine) and more instructions between
// the slices: 5120 x 1024 over 2 8.8 -> 9.6, 4096 x 4096 11.85 -> 12.35, 8064 x 2048 11.3 -> 11.6 us; at five to seven rows the two are within 2% (mean
// +0.7 to +2.3%), unsplit at eight +1.3%.
template <int M, int RB>
__device__ __forceinline__ void dot_any_scale(const GemvArgs& a, int row_, int seg0, int sk, const uint4* xs, int lane, float (&acc)[RB][M]) {
  constexpr int FMT = DSGX_FMT_INT4_G32;
  const int row = uni(row_);
  int si = 0;
#pragma unroll
  for (int i = 1; i < kMaxSegs; ++i)
    if (i < a.nsegs && row >= a.sg[i].row0) si = i;
  RowSrc src[RB];
#pragma unroll
  for (int i = 0; i < RB; ++i) {
    src[i] = row_src<FMT>(a.sg[si].m, row - a.sg[si].row0 + i, a.K);
#pragma unroll
    for (int m = 0; m < M; ++m) acc[i][m] = 0.f;
  }
  for (int seg = seg0; seg < a.nsegk; seg += sk) {
    const uint32_t le = lane < (seg == a.nsegk - 1 ? last_seg_lanes<FMT>(a.K, a.nsegk) : kWave) ? lane : 0;
    Raw r[RB];
#pragma unroll
    for (int i = 0; i < RB; ++i) load_row<FMT>(r[i], src[i], seg, le, 0, acc[i][0]);
    step_dot<FMT, M, RB, true>(r, xs, a.nq, seg, lane, acc, a.K);
  }
}

// NW: wavefronts a workgroup, in groups of four: the first batches of the walk go to every workgroup's first group, so that
// fewer batches than wavefronts still spread over all CUs. SPLIT: the split-K order of adds (k_gemv_sk's slices, in their
// order, the same bits) by one wavefront that walks the slices one after the other.
// Bound by the vector unit (INT4, or from 3 activation rows) or by latency: eight wavefronts a CU in ONE workgroup stage the
// activations once a CU and keep two wavefronts a SIMD where 64 KB and more of activations left room for one workgroup of
// four (INT4 6144 x 16384, 4 rows: 36.1 us with four waves, 27.1 with eight - 25.8 since they hold no code of the add + norm
// prologue -, 29.6 with sixteen; FP8 12000 x 8192, 8 rows: 41.6, 33.8, 52.5). Two rows a wavefront: four leave half the waves
// without a batch or make a longer last round (INT4 16384 x 2048, 1 row: 13.4 against 10.6).
template <int FMT, int M, int RB, int D, int NW, bool SPLIT>
__global__ void __launch_bounds__(NW * 64) k_gemv(GemvArgs a) {
  extern __shared__ uint4 xs[];
  __shared__ float red[4 * M];
  const int lane = threadIdx.x & 63;
  // (the wave's number is the same in every lane: said so, which keeps the row cursors and the segment's descriptor on the
  // scalar unit - read from a vector register they came through vector loads of the kernel's arguments, which a wave's
  // weight loads then queued behind, one ring entry after the other)
  const int wave = uni(threadIdx.x >> 6);
  const int gw = uni((wave >> 2) * (int)gridDim.x * 4 + (int)blockIdx.x * 4 + (wave & 3)), GW = gridDim.x * NW;
  const int nbatch = a.total_rows / RB;
  const int nmine = gw < nbatch ? (nbatch - gw + GW - 1) / GW : 0;
  const int nsteps = nmine * a.nsegk;
  const int sk = SPLIT ? a.splitk : 1, slices = SPLIT ? min(sk, a.nsegk) : 1;  // the K slices of a row, and those that hold a segment

  auto locate = [&](int row, int& si) {
    si = 0;
#pragma unroll
    for (int i = 1; i < kMaxSegs; ++i)
      if (i < a.nsegs && row >= a.sg[i].row0) si = i;
  };
  Raw w[D][RB];
  float acc[RB][M];
#pragma unroll
  for (int r = 0; r < RB; ++r)
#pragma unroll
    for (int m = 0; m < M; ++m) acc[r][m] = 0.f;
  int lt = 0, lj = 0, lsl = 0, lseg = 0;  // the load cursor: step, batch number of this wave, slice, segment
  // the rows of the batch under the load cursor: their addresses are set up on the scalar unit when the cursor enters a batch, and a
  // step's loads are a scalar base and a lane offset each. (With 64-bit addresses made on the lanes for every load there were 85
  // instructions between one load and the next, which is what the waves' first loads waited for: INT4 6144 x 16384 at one / four rows
  // 20.4 / 27.6 us a call -> 19.4 / 26.2, 1536 x 6144 at one row 6.8 -> 6.4, FP8 16384 x 1536 8.7 -> 8.45, 1000 x 1152 4.25 -> 4.03.)
  // (a call with one segment, the common one, fetches its descriptor once: every later fetch would be two dependent scalar round trips)
  MatDev lm = a.sg[0].m;
  RowSrc src[RB];
  auto enter = [&]() {
    const int row = uni(min((gw + lj * GW) * RB, a.total_rows - RB));  // (a wave without a batch: rows of its own as far as there are)
    int row0 = 0;
    if (a.nsegs > 1) {
      int si;
      locate(row, si);
      lm = a.sg[si].m, row0 = a.sg[si].row0;
    }
#pragma unroll
    for (int i = 0; i < RB; ++i) src[i] = row_src<FMT>(lm, row - row0 + i, a.K);
  };
  enter();
  // past the last step the ring's loads go, scales and zero points too, to the first bytes of the wave's last rows: one cached line of
  // the wave's own (with a line for each kind of load, 2048 x 4096 over 2 took 5.9 us, 5.4 like this)
  auto park = [&]() {
#pragma unroll
    for (int i = 0; i < RB; ++i) src[i].w = src[i].a = src[i].z = src[0].w;
  };
  if (nsteps == 0) park();
  const int last_lanes = last_seg_lanes<FMT>(a.K, a.nsegk);
  auto load = [&](Raw (&r)[RB]) {
    const bool ok = lt < nsteps;
    ++lt;
    const uint32_t le = lane < uni(ok ? (lseg == a.nsegk - 1 ? last_lanes : kWave) : 0) ? lane : 0;
#pragma unroll
    for (int i = 0; i < RB; ++i) load_row<FMT>(r[i], src[i], uni(ok ? lseg : 0), le, lm.lks, acc[i][0]);
    if (ok && (lseg += sk) >= a.nsegk) {
      if (++lsl == slices) {
        lsl = 0, ++lj;
        if (lt < nsteps) enter();
        else park();
      }
      lseg = lsl;
    }
  };
  int cj = 0, csl = 0, cseg = 0;
  float mine = 0.f, mine2 = 0.f;  // lane r * M + m: output (row r, activation row m) of the batch, and the pair's other row (SwiGLU)
  constexpr bool kFast = FMT == DSGX_FMT_INT4_G32 && !(SPLIT && M == 8);  // (dot_any_scale)
  float smax = 0.f;  // the largest scale that the wave has met
  // a slice is complete: add the lanes' partials, then the slices' sums in their order
  auto slice_done = [&]() {
    float v1 = 0.f, v2 = 0.f;
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int m = 0; m < M; ++m) {
        const float v = wave_sum(acc[i][m]);
        acc[i][m] = 0.f;
        if (lane == i * M + m) v1 = v;
        if (lane == (i ^ 1) * M + m) v2 = v;
      }
    mine = SPLIT && csl ? __fadd_rn(mine, v1) : v1, mine2 = SPLIT && csl ? __fadd_rn(mine2, v2) : v2;
    cseg = ++csl;
    if (SPLIT && csl < slices) return;
    if (SPLIT && slices < sk) mine = __fadd_rn(mine, 0.f), mine2 = __fadd_rn(mine2, 0.f);  // (an empty slice's sum, as k_gemv_sk adds it)
    csl = cseg = 0;
    const int row = (gw + cj * GW) * RB;
    ++cj;
    if (lane >= RB * M) return;
    int si = 0;
    if (a.nsegs > 1) locate(row, si);
    const GemvSegDev& sg = a.sg[si];
    const int r = lane / M, m = lane % M, n = row - sg.row0 + r;
    if (a.out == DSGX_OUT_BF16) {
      static_cast<uint16_t*>(sg.y)[(size_t)m * sg.ldy + n] = (uint16_t)f32_to_bf16_bits(mine);
    } else if (a.out == DSGX_OUT_F32) {
      static_cast<float*>(sg.y)[(size_t)m * sg.ldy + n] = mine;
    } else if ((r & 1) == 0) {  // SwiGLU: row 2i gate, 2i + 1 up -> column i (gemv.cu:164-168)
      static_cast<uint16_t*>(sg.y)[(size_t)m * sg.ldy + n / 2] = (uint16_t)swiglu_bits(bf16_round(mine), bf16_round(mine2));
    }
  };
  auto compute = [&](const Raw (&raw)[RB]) {
    step_dot<FMT, M, RB, true, kFast>(raw, xs, a.nq, cseg, lane, acc, a.K, &smax);
    if ((cseg += sk) >= a.nsegk) slice_done();
  };
  // the first weight loads are issued before the activations are staged: one memory round trip, not two, before the
  // first product (these calls are a few microseconds long: latency is most of them)
#pragma unroll
  for (int d = 0; d < D; ++d) load(w[d]);
  stage_rows<FmtT<FMT>::KL, M, NW == 4>(xs, a, red);
  __syncthreads();
  for (int t = 0; t < nsteps; t += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      if (t + d < nsteps) compute(w[d]);
      load(w[d]);
    }
  }
  if constexpr (kFast) {
    if (__builtin_expect(i4_any_large(smax), 0)) {  // all of the wave's rows once more, each lane over its own results
      cj = csl = 0;
      while (cj < nmine) {
        dot_any_scale<M, RB>(a, (gw + cj * GW) * RB, csl, sk, xs, lane, acc);
        slice_done();
      }
    }
  }
}

// Split-K (engine/attn/attn.h:119 of the reference: warps of a CTA share a tile's k range, for small N): a workgroup of
// four waves holds 4 / SK row batches, the SK waves of a batch take the K segments slice, slice + SK, ... of its rows;
// the waves' sums meet in LDS and the batch's first wave adds them in slice order (a fixed order, as the reference's
// finish(), gemv.cu:138-151), then the epilogue of k_gemv. One batch a group and launch: this form is for matrices of
// few rows, where whole-K waves would leave most of the chip idle and walk K in several dependent round trips; the others
// take the same slices one after the other in k_gemv.
template <int FMT, int M, int RB, int SK>
__global__ void __launch_bounds__(256) k_gemv_sk(GemvArgs a) {
  extern __shared__ uint4 xs[];
  __shared__ float part[4][RB * M];
  __shared__ float red[4 * M];
  const int lane = threadIdx.x & 63, wave = uni(threadIdx.x >> 6);  // (uniform: the segment's descriptor stays on the scalar unit)
  constexpr int GPW = 4 / SK;  // batches a workgroup
  const int grp = wave / SK, slice = wave % SK;
  const int nbatch = a.total_rows / RB;
  const int batch = blockIdx.x * GPW + grp;
  const bool live = batch < nbatch;
  const int row = uni(live ? batch * RB : 0);
  int si = 0;
#pragma unroll
  for (int i = 1; i < kMaxSegs; ++i)
    if (i < a.nsegs && row >= a.sg[i].row0) si = i;
  const GemvSegDev& sg = a.sg[si];
  const int nmine = live && slice < a.nsegk ? (a.nsegk - slice + SK - 1) / SK : 0;  // this wave's segments
  constexpr int D = 4;
  Raw w[D][RB];
  float acc[RB][M];
#pragma unroll
  for (int r = 0; r < RB; ++r)
#pragma unroll
    for (int m = 0; m < M; ++m) acc[r][m] = 0.f;
  RowSrc src[RB];
#pragma unroll
  for (int i = 0; i < RB; ++i) src[i] = row_src<FMT>(sg.m, row - sg.row0 + i, a.K);
  const int last_lanes = last_seg_lanes<FMT>(a.K, a.nsegk);
  int lt = 0;
  auto load = [&](Raw (&r)[RB]) {
    const bool ok = lt < nmine;
    if (lt == nmine)  // past the last step: the first bytes of this wave's rows (k_gemv's park)
#pragma unroll
      for (int i = 0; i < RB; ++i) src[i].w = src[i].a = src[i].z = src[0].w;
    const int seg = uni(ok ? slice + lt * SK : 0);
    ++lt;
    const uint32_t le = lane < uni(ok ? (seg == a.nsegk - 1 ? last_lanes : kWave) : 0) ? lane : 0;
#pragma unroll
    for (int i = 0; i < RB; ++i) load_row<FMT>(r[i], src[i], seg, le, sg.m.lks, acc[i][0]);
  };
#pragma unroll
  for (int d = 0; d < D; ++d) load(w[d]);
  stage_rows<FmtT<FMT>::KL, M, true>(xs, a, red);
  __syncthreads();
  for (int t = 0; t < nmine; t += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      if (t + d < nmine) step_dot<FMT, M, RB, true>(w[d], xs, a.nq, slice + (t + d) * SK, lane, acc, a.K);
      load(w[d]);
    }
  }
  // the wave's sums over its lanes, value (i, m) kept by lane i * M + m
  float mine = 0.f;
#pragma unroll
  for (int i = 0; i < RB; ++i)
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const float v = wave_sum(acc[i][m]);
      if (lane == i * M + m) mine = v;
    }
  if (lane < RB * M) part[wave][lane] = mine;
  __syncthreads();
  if (!live || slice != 0 || lane >= RB * M) return;
  float sum = part[grp * SK][lane];
#pragma unroll
  for (int k = 1; k < SK; ++k) sum = __fadd_rn(sum, part[grp * SK + k][lane]);
  const int r = lane / M, m = lane % M, n = row - sg.row0 + r;
  if (a.out == DSGX_OUT_BF16) {
    static_cast<uint16_t*>(sg.y)[(size_t)m * sg.ldy + n] = (uint16_t)f32_to_bf16_bits(sum);
  } else if (a.out == DSGX_OUT_F32) {
    static_cast<float*>(sg.y)[(size_t)m * sg.ldy + n] = sum;
  } else if ((r & 1) == 0) {  // SwiGLU: row 2i gate, 2i + 1 up -> column i; the up row's sum sits M lanes further
    float up = part[grp * SK][lane + M];
#pragma unroll
    for (int k = 1; k < SK; ++k) up = __fadd_rn(up, part[grp * SK + k][lane + M]);
    static_cast<uint16_t*>(sg.y)[(size_t)m * sg.ldy + n / 2] = (uint16_t)swiglu_bits(bf16_round(sum), bf16_round(up));
  }
}

template <int FMT, int M, int SK>
int launch_gemv_sk(const GemvArgs& a, hipStream_t st) {
  constexpr int RB = 2;
  const size_t lds = (size_t)M * a.nq * 16;
  const int nbatch = a.total_rows / RB, gpw = 4 / SK;
  auto kern = k_gemv_sk<FMT, M, RB, SK>;
  if (int rc = allow_dynamic_lds(reinterpret_cast<const void*>(kern), lds)) return rc;
  hipLaunchKernelGGL(kern, dim3((nbatch + gpw - 1) / gpw), dim3(256), lds, st, a);
  DSGX_HIP(hipGetLastError());
  return DSGX_OK;
}

template <int FMT, int M, int NW, bool SPLIT>
int launch_gemv_nw(const GemvArgs& a, hipStream_t st) {
  constexpr int RB = 2, D = 4;
  if (NW != 4 && a.norm.part) return fail(DSGX_EINVAL, "gemv: the add + norm prologue runs in workgroups of four wavefronts");
  const size_t lds = (size_t)M * a.nq * 16;
  const int nbatch = a.total_rows / RB;
  // never more workgroups than it takes to give every group of four wavefronts a batch
  const int per_cu = NW == 4 && lds <= 64 * 1024 ? 2 : 1;
  int grid = num_cus_cached() * per_cu;
  if (grid > (nbatch + 3) / 4) grid = (nbatch + 3) / 4;
  if (grid < 1) grid = 1;
  auto kern = k_gemv<FMT, M, RB, D, NW, SPLIT>;
  if (int rc = allow_dynamic_lds(reinterpret_cast<const void*>(kern), lds)) return rc;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(NW * 64), lds, st, a);
  DSGX_HIP(hipGetLastError());
  return DSGX_OK;
}
template <int FMT, int M, int NW>
int launch_gemv(const GemvArgs& a, hipStream_t st) {
  return a.splitk > 1 ? launch_gemv_nw<FMT, M, NW, true>(a, st) : launch_gemv_nw<FMT, M, NW, false>(a, st);
}
template <int FMT, int M>
int launch_gemv_rows(const GemvArgs& a, hipStream_t st) {
  const int nbatch = a.total_rows / 2, cus = num_cus_cached(), sk = a.splitk;
  constexpr bool kBf16 = FMT == DSGX_FMT_BF16;
  const size_t lds = (size_t)M * a.nq * 16;
  // Slices on waves of their own (k_gemv_sk): a workgroup stages all activation rows for 4 / sk batches, so what counts is how
  // many of its workgroups a CU holds at once. (us below: own waves / one wave walking the slices in k_gemv)
  //   one a CU: always (BF16 1000 x 4096 over 2, 8 rows: 8.1 / 9.5; FP8 384 x 2048 over 4, 1 row: 4.4 / 4.6);
  //   two: BF16, whose steps are short, from two segments a row (1024 x 6144 over 4, 6 rows: 9.4 / 11.8; 2048 x 512 over 2 only
  //   at many rows: 8 rows 5.3 / 5.7); the others only where slices are long: over 4 from four segments (INT4 1000 x 12288,
  //   2 rows: 10.1 / 11.2; FP8 768 x 2048, 3 rows: 5.7 / 5.6), three at one or two rows (INT4 768 x 6144, 1 row: 6.5 / 6.9), over
  //   2 at one row from five (INT4 1152 x 10240: 8.4 / 9.3);
  //   three, which registers allow at one BF16 row: from six segments (1152 x 8192 over 2: 7.7 / 8.1);
  //   more, a second round: never (INT4 6144 x 16384 over 4, 4 rows: 125 / 28).
  const long waves = (long)nbatch * sk;
  bool own = sk > 1 && waves <= 4 * cus;
  // (under the add + norm prologue every workgroup makes the rows: one a CU or none. FP8 768 x 4096 over 4, 3 rows: 18.7 / 14.8)
  if (sk > 1 && !a.norm.part) {
    const bool two_fit = waves <= 8 * cus && 2 * (lds + 1024) <= 160 * 1024;
    own = own || (two_fit && (kBf16 ? a.nsegk >= 2 || M >= 4 : sk == 4 ? a.nsegk >= (M <= 2 ? 3 : 4) : M == 1 && a.nsegk >= 5));
    own = own || (kBf16 && M == 1 && waves <= 12 * cus && a.nsegk >= 6);
  }
  if (own) return sk == 2 ? launch_gemv_sk<FMT, M, 2>(a, st) : launch_gemv_sk<FMT, M, 4>(a, st);
  // Two workgroups of four a CU under the add + norm prologue (256 threads' work), and for few and short BF16 rows, which are
  // over before eight waves' staging returns anything (1024 x 2048, 1 row: 4.8 us, 5.1 with eight a workgroup; 1024 x 8192,
  // 8 rows, beyond 32 KB of activations: 14.2 and 12.9). FP8 and INT4 take eight at every size (64 x 1024: the same time).
  if (a.norm.part || (kBf16 && nbatch <= 4 * cus && lds <= 32 * 1024)) return launch_gemv<FMT, M, 4>(a, st);
  return launch_gemv<FMT, M, 8>(a, st);
}
template <int FMT>
int launch_gemv_m(int M, const GemvArgs& a, hipStream_t st) {
  switch (M) {
    case 1: return launch_gemv_rows<FMT, 1>(a, st);
    case 2: return launch_gemv_rows<FMT, 2>(a, st);
    case 3: return launch_gemv_rows<FMT, 3>(a, st);
    case 4: return launch_gemv_rows<FMT, 4>(a, st);
    case 5: return launch_gemv_rows<FMT, 5>(a, st);
    case 6: return launch_gemv_rows<FMT, 6>(a, st);
    case 7: return launch_gemv_rows<FMT, 7>(a, st);
    case 8: return launch_gemv_rows<FMT, 8>(a, st);
  }
  return fail(DSGX_EINVAL, "gemv: %d rows a launch", M);
}

int ilog2_exact(int v) {
  int l = 0;
  while ((1 << l) < v) ++l;
  return (1 << l) == v ? l : -1;
}

// one launch: the segments of one format (gemv_one of the reference, gemv.cu:459-516)
int gemv_one(int fmt, const uint16_t* x, int ldx, int rows, int K, const dsgx_gemv_seg* segs, int nseg, int out, int splitk, hipStream_t st,
             const NormIn* norm = nullptr) {
  GemvArgs a{};
  a.x = x, a.ldx = ldx, a.K = K, a.out = out, a.nsegs = nseg;
  if (norm) a.norm = *norm;
  const int segk = fmt == DSGX_FMT_FP8_B128 ? 1024 : fmt == DSGX_FMT_INT4_G32 ? 2048 : 512;
  a.nsegk = (K + segk - 1) / segk;
  a.nq = a.nsegk * segk / 8;
  int row0 = 0;
  for (int i = 0; i < nseg; ++i) {
    const dsgx_gemv_seg& g = segs[i];
    GemvSegDev& d = a.sg[i];
    d.m.w = static_cast<const uint8_t*>(g.w);
    d.m.s = static_cast<const uint8_t*>(g.s);
    d.m.zp = static_cast<const uint8_t*>(g.zp);
    d.m.s2 = 1.f;
    if (!g.w || !g.y) return fail(DSGX_EINVAL, "gemv: segment %d has a null weight or output", i);
    if (fmt == DSGX_FMT_FP8_B128) {
      d.m.lrs = ilog2_exact(g.rs), d.m.lks = ilog2_exact(g.ks);
      if (!g.s || d.m.lrs < 0 || d.m.lks < 4 || K % g.ks) return fail(DSGX_EINVAL, "gemv: FP8 segment %d scale block %dx%d (powers of two, k >= 16)", i, g.rs, g.ks);
      if (out == DSGX_OUT_SWIGLU) return fail(DSGX_EUNSUPPORTED, "gemv: SwiGLU output over FP8 weights is not built");
      d.m.srow = K >> d.m.lks;
    } else if (fmt == DSGX_FMT_INT4_G32) {
      if (!g.s || !g.zp) return fail(DSGX_EINVAL, "gemv: INT4 segment %d needs scales and zero points", i);
    }
    d.y = g.y, d.n = g.n, d.ldy = g.ldy, d.row0 = row0;
    row0 += g.n;
  }
  a.total_rows = row0;
  // (dsgx_gemv's contract: whole-K sums above 32 rows a CU, whatever split the call asks for. There the slices cost a sum over
  // the wave each and return nothing: FP8 9000 x 4096 over 4, 8 rows: 24.9 us with slices, 19.9 without)
  a.splitk = a.total_rows <= 32 * num_cus_cached() ? splitk : 1;
  if (rows > 8) return fail(DSGX_EINVAL, "gemv_one: %d rows", rows);
  switch (fmt) {
    case DSGX_FMT_FP8_B128: return launch_gemv_m<DSGX_FMT_FP8_B128>(rows, a, st);
    case DSGX_FMT_INT4_G32: return launch_gemv_m<DSGX_FMT_INT4_G32>(rows, a, st);
    case DSGX_FMT_BF16: return launch_gemv_m<DSGX_FMT_BF16>(rows, a, st);
  }
  return fail(DSGX_EFORMAT, "gemv: format %d", fmt);
}

}  // namespace
}  // namespace dsgx

using namespace dsgx;

extern "C" int dsgx_gemv(const uint16_t* x, int ldx, int rows, int K, const dsgx_gemv_seg* segs, int nseg, int out, int splitk,
                         void* stream) {
  // argument checks of the reference (gemv.cu:524-543): it dies, this returns an error
  if (rows < 1 || rows > DSGX_MAX_ROWS) return fail(DSGX_EINVAL, "gemv: %d rows", rows);
  if (!x || !segs || nseg < 1 || nseg > kMaxSegs) return fail(DSGX_EINVAL, "gemv: K %d, %d segments", K, nseg);
  if (K < 32 || K % 32 || ldx < K || ldx % 8) return fail(DSGX_EINVAL, "gemv: K %d (a multiple of 32), ldx %d (>= K, a multiple of 8)", K, ldx);
  if (splitk != 1 && splitk != 2 && splitk != 4) return fail(DSGX_EINVAL, "gemv: splitk %d", splitk);
  if (out != DSGX_OUT_BF16 && out != DSGX_OUT_F32 && out != DSGX_OUT_SWIGLU) return fail(DSGX_EINVAL, "gemv: output kind %d", out);
  for (int i = 0; i < nseg; ++i) {
    const int f = segs[i].fmt;
    if (f != DSGX_FMT_BF16 && f != DSGX_FMT_INT4_G32 && f != DSGX_FMT_FP8_B128)
      return fail(DSGX_EFORMAT, "gemv: segment %d has no supported weight format (%d)", i, f);
    if (segs[i].n < 8 || segs[i].n % 8) return fail(DSGX_EINVAL, "gemv: segment %d has %d rows", i, segs[i].n);
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  // one launch a format, in the order BF16, INT4, FP8 (outputs do not depend on it); more than 8 activation rows run
  // as two passes over the weights
  for (int fmt : {DSGX_FMT_BF16, DSGX_FMT_INT4_G32, DSGX_FMT_FP8_B128}) {
    dsgx_gemv_seg g[kMaxSegs];
    int n = 0;
    for (int i = 0; i < nseg; ++i)
      if (segs[i].fmt == fmt) g[n++] = segs[i];
    if (!n) continue;
    for (int r0 = 0; r0 < rows; r0 += 8) {
      const int nr = rows - r0 < 8 ? rows - r0 : 8;
      dsgx_gemv_seg gg[kMaxSegs];
      for (int i = 0; i < n; ++i) {
        gg[i] = g[i];
        const size_t esz = out == DSGX_OUT_F32 ? 4 : 2;
        gg[i].y = static_cast<uint8_t*>(g[i].y) + (size_t)r0 * g[i].ldy * esz;
      }
      const int rc = gemv_one(fmt, x + (size_t)r0 * ldx, ldx, nr, K, gg, n, out, splitk, st);
      if (rc) return rc;
    }
  }
  return DSGX_OK;
}

// The residual add + RMSNorm of dsgx_add_norm as the GEMV's prologue: x = the normed rows, made inside the GEMV kernel.
extern "C" int dsgx_add_norm_gemv(const dsgx_norm_in* n, int rows, int K, const dsgx_gemv_seg* segs, int nseg, int out, int splitk, void* stream) {
  if (!n || !n->part || !n->res || !n->w) return fail(DSGX_EINVAL, "add_norm_gemv: the partial sums, the residual and the norm's weight are needed");
  if (rows < 1 || rows > 8) return fail(DSGX_EUNSUPPORTED, "add_norm_gemv: %d rows (1..8; more: dsgx_add_norm, then dsgx_gemv)", rows);
  if (K < 2048 || K % 2048 || K > 16384) return fail(DSGX_EINVAL, "add_norm_gemv: hidden %d (a multiple of 2048 up to 16384)", K);
  if (n->res_out == n->res) return fail(DSGX_EINVAL, "add_norm_gemv: res_out must not be res (every workgroup reads the residual while one writes the new one)");
  if (!segs || nseg < 1 || nseg > kMaxSegs) return fail(DSGX_EINVAL, "add_norm_gemv: %d segments", nseg);
  if (splitk != 1 && splitk != 2 && splitk != 4) return fail(DSGX_EINVAL, "add_norm_gemv: splitk %d", splitk);
  if (out != DSGX_OUT_BF16 && out != DSGX_OUT_F32 && out != DSGX_OUT_SWIGLU) return fail(DSGX_EINVAL, "add_norm_gemv: output kind %d", out);
  const int f = segs[0].fmt;
  if (f != DSGX_FMT_BF16 && f != DSGX_FMT_INT4_G32 && f != DSGX_FMT_FP8_B128) return fail(DSGX_EFORMAT, "add_norm_gemv: no supported weight format (%d)", f);
  for (int i = 0; i < nseg; ++i) {
    if (segs[i].fmt != f) return fail(DSGX_EUNSUPPORTED, "add_norm_gemv: the segments of one call share a format (one launch)");
    if (segs[i].n < 8 || segs[i].n % 8) return fail(DSGX_EINVAL, "add_norm_gemv: segment %d has %d rows", i, segs[i].n);
  }
  const NormIn ni{n->part, n->part2, n->res, n->res_out, n->w, n->xn, n->eps, n->round2};
  return gemv_one(f, nullptr, K, rows, K, segs, nseg, out, splitk, static_cast<hipStream_t>(stream), &ni);
}
