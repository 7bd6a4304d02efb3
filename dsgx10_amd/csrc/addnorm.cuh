// The residual add and RMSNorm of rows by a workgroup of 256 threads: the local half of the reference's
// comm::glm::allreduce_add_norm / allreduce2_add_norm (altar1-4xgx10-switchless/engine/comm/glmcoll.h:34-62) at one rank,
// the norm as engine/attn/prep.cu:12-66 (k_rmsnorm):
//   sum        = part                                   (one partial: the reference's decision 8, yr already holds yr + ys)
//              | bf16(bf16(part) + bf16(part2))         (two partials: the old combine, experts.h finalize)
//   h          = bf16(f32(res) + sum)                   (the contract: the f32 sum rounded once, with the residual)
//              | bf16(f32(res) + bf16(sum))             (round2: the sum rounded first)
//   xn         = bf16(w * bf16(h * rstd)),  rstd = 1 / sqrt(mean(h^2) + eps), IEEE division and square root
// mean(h^2) in f32 in a fixed order: a thread's H / 256 contiguous values in order, the wave by a butterfly, the waves in
// order (the reference fixes an order too, its own: the statistics' order is not part of the contract).
// Used by k_add_norm (a launch of its own) and as the prologue of the dense GEMV kernels (the normed rows go straight
// into the GEMV's staged activations): one code, so both give the same bits.
#pragma once
#include "common.cuh"

namespace dsgx {

struct NormIn {
  const float* part;   // f32 [M][H]; null: no add + norm (the GEMV reads x)
  const float* part2;
  const uint16_t* res;
  uint16_t* res_out;   // may be null
  const uint16_t* w;
  uint16_t* xn;        // may be null
  float eps;
  int round2;
};

// M rows at once (rows row0 ... row0 + M - 1) by 256 threads. xs: LDS for the rows' chunks of 8 bf16 values, chunk q of row m at
// xs[at(m, q)]; red: 4 M floats of LDS. h goes to memory (res_out) and the normed rows to xs and memory (xn) if `writer`.
// Bound by latency: the rows' loads are requested together, chunk after chunk of neighbouring threads (a chunk's h does not mind
// who makes it), and the sums of squares, whose order is fixed, are taken from LDS, all rows between the same two barriers. A row
// at a time, each its own loads and barriers, every thread its 16 or 24 contiguous values, was 4 us a row in front of a router
// (168 x 6144, 3 rows: 17.2 us,
// 12.4 like this before the roundings were one instruction; 256 x 4096, one row, 6.8 and 6.1; a launch of its own at 4096, one row, 4.3 and 3.8).
typedef uint32_t f32x4_row_t __attribute__((ext_vector_type(4), aligned(4)));  // (the partial sums' rows are floats: four at any)
template <int M, class At>
__device__ __forceinline__ void add_norm_rows(const NormIn& a, int row0, int H, uint4* xs, float* red, bool want_xn, bool writer, At&& at) {
  const int tid = threadIdx.x, C = H / 2048, n = M * C;  // a thread's chunks of a row: c 256 + tid, c < C <= 8 (the host checks)
  u32x4_t wq[8];
#pragma unroll
  for (int c = 0; c < 8; ++c)
    if (want_xn && c < C) wq[c] = *reinterpret_cast<const DSGX_GLOBAL u32x4_t*>((uintptr_t)(a.w + 8 * (c * 256 + tid)));
  constexpr int B = M == 1 ? 4 : 8;  // chunks in flight
  for (int j0 = 0; j0 < n; j0 += B) {
    u32x4_t r[B], p[B][2];
#pragma unroll
    for (int u = 0; u < B; ++u) {
      const int j = min(j0 + u, n - 1), m = uni(j / C);
      const size_t o = (size_t)(row0 + m) * H + 8 * ((j - m * C) * 256 + tid);
      r[u] = *reinterpret_cast<const DSGX_GLOBAL u32x4_t*>((uintptr_t)(a.res + o));
#pragma unroll
      for (int i = 0; i < 2; ++i) p[u][i] = *reinterpret_cast<const DSGX_GLOBAL f32x4_row_t*>((uintptr_t)(a.part + o + 4 * i));
    }
#pragma unroll
    for (int u = 0; u < B; ++u) {
      if (j0 + u >= n) break;
      const int j = j0 + u, m = uni(j / C), q = (j - m * C) * 256 + tid;
      const size_t o = (size_t)(row0 + m) * H + 8 * q;
      float hs[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        float s = __uint_as_float(p[u][k >> 2][k & 3]);
        if (a.part2) s = __fadd_rn(bf16_round(s), bf16_round(a.part2[o + k])), s = bf16_round(s);
        else if (a.round2) s = bf16_round(s);
        hs[k] = __fadd_rn(k & 1 ? bf16_hi(r[u][k >> 1]) : bf16_lo(r[u][k >> 1]), s);
      }
      const uint32_t ho[4] = {pack_bf16(hs[0], hs[1]), pack_bf16(hs[2], hs[3]), pack_bf16(hs[4], hs[5]), pack_bf16(hs[6], hs[7])};
      if (writer && a.res_out) *reinterpret_cast<u32x4_t*>(a.res_out + o) = u32x4_t{ho[0], ho[1], ho[2], ho[3]};
      if (want_xn) xs[at(m, q)] = make_uint4(ho[0], ho[1], ho[2], ho[3]);
    }
  }
  if (!want_xn) return;
  __syncthreads();
  // the mean's order: a thread's H / 256 contiguous values one after the other, the wave by wave_sum, the waves in order
  float ss[M];
#pragma unroll
  for (int m = 0; m < M; ++m) ss[m] = 0.f;
  for (int c = 0; c < C; ++c)
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const uint4 v = xs[at(m, tid * C + c)];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint32_t w = k == 0 ? v.x : k == 1 ? v.y : k == 2 ? v.z : v.w;
        const float lo = bf16_lo(w), hi = bf16_hi(w);
        ss[m] = __fadd_rn(ss[m], __fmul_rn(lo, lo));
        ss[m] = __fadd_rn(ss[m], __fmul_rn(hi, hi));
      }
    }
#pragma unroll
  for (int m = 0; m < M; ++m) {
    const float t = wave_sum(ss[m]);
    if ((tid & 63) == 0) red[4 * m + (tid >> 6)] = t;
  }
  __syncthreads();
  float rstd[M];
#pragma unroll
  for (int m = 0; m < M; ++m) {
    const float tot = __fadd_rn(__fadd_rn(__fadd_rn(red[4 * m], red[4 * m + 1]), red[4 * m + 2]), red[4 * m + 3]);
    rstd[m] = __fdiv_rn(1.f, sqrtf(__fadd_rn(__fdiv_rn(tot, (float)H), a.eps)));  // (sqrtf: the correctly rounded root)
  }
#pragma unroll
  for (int m = 0; m < M; ++m)
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      if (c >= C) break;
      const int q = c * 256 + tid;
      const uint4 v = xs[at(m, q)];
      const uint32_t hv[4] = {v.x, v.y, v.z, v.w};
      uint32_t o[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint32_t n = pack_bf16(__fmul_rn(bf16_lo(hv[k]), rstd[m]), __fmul_rn(bf16_hi(hv[k]), rstd[m]));
        o[k] = pack_bf16(__fmul_rn(bf16_lo(wq[c][k]), bf16_lo(n)), __fmul_rn(bf16_hi(wq[c][k]), bf16_hi(n)));
      }
      xs[at(m, q)] = make_uint4(o[0], o[1], o[2], o[3]);
      if (writer && a.xn) *reinterpret_cast<u32x4_t*>(a.xn + (size_t)(row0 + m) * H + 8 * q) = u32x4_t{o[0], o[1], o[2], o[3]};
    }
}

}  // namespace dsgx
