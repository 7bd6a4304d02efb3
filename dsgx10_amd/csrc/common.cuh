// Device helpers shared by the gfx950 kernels: bf16 / e4m3 / INT4 decode in registers, wave64 reductions, the
// streaming loads, the activation staging layout and the router's row function.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/dsgx.h"

namespace dsgx {

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));

constexpr int kWave = 64;

// ---- scalar codecs ------------------------------------------------------------------------------------------------
__device__ __forceinline__ float bf16_bits_to_f32(uint32_t b) { return __uint_as_float(b << 16); }
// f32 -> bf16, round to nearest even (engine/experts/formats.cuh:33-37 of the reference): v_cvt_pk_bf16_f32, one instruction (two for
// the rounded f32) where adding half a step by hand is four; the same bits for every number, and a NaN stays a NaN (by hand the carry
// takes some to infinity or -0). A test compares all 2^32.
__device__ __forceinline__ uint32_t f32_to_bf16_bits(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }
__device__ __forceinline__ float bf16_round(float f) { return (float)(__bf16)f; }
// two f32 -> packed bf16 (lo = a, hi = b), round to nearest even: v_cvt_pk_bf16_f32
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
  bf16x2_t v = {(__bf16)a, (__bf16)b};
  return __builtin_bit_cast(uint32_t, v);
}
// acc + a.lo * b.lo + a.hi * b.hi on packed bf16 pairs: v_dot2c_f32_bf16
__device__ __forceinline__ float dot2(uint32_t a, uint32_t b, float acc) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, a), __builtin_bit_cast(bf16x2_t, b), acc, false);
}

// ---- weight decode: 8 consecutive k -> four packed bf16 pairs (k, k+1) ---------------------------------------------------
// FP8 e4m3fn: two 32-bit words (8 codes) -> exact bf16 values (v_cvt_scalef32_pk_bf16_fp8 with scale 1).
__device__ __forceinline__ void fp8x8_to_bf16(uint32_t w0, uint32_t w1, uint32_t (&o)[4]) {
  o[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w0, 1.0f, false));
  o[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w0, 1.0f, true));
  o[2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w1, 1.0f, false));
  o[3] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w1, 1.0f, true));
}
// INT4-g32: one 32-bit word = 8 stored nibbles u (value i at bits 4i) of one group with scale s (f32 of the bf16) and zero
// point u_z: W = bf16_rne((u - u_z) * s). The INT4 streams wait for the vector unit, so what counts is instructions a value:
// the nibbles become f16 numbers by one and-or a PAIR of them (1024 + u of the nibbles at bits 0 and 16 of the word, 1024 +
// 16 u of those at bits 4 and 20: the unit of an f16 in [1024, 2048) is 1), v_fma_mix_f32 takes such a half as its first
// factor and gives (1024 + u) s - (1024 + u_z) s, or (1024 + 16 u) (s / 16) - (64 + u_z) s, and the packed conversion rounds
// once to nearest even: 17 instructions for 8 values where byte conversions and fmas took 23 (the 1024-offset form of a nibble is
// a widely used one). Every product and constant has at most 11 + 8 significant bits, so it is exact in f32, and so is the difference;
// the constants stay finite for |s| < 2^116, which no checkpoint comes near: a decode unit, a GEMV's rows or a prefill tile that meets a larger
// scale is done once more by i4x8_to_bf16_any, whose terms are finite up to 2^124 (dequant_int4's own kernel uses the subtract-first form, for all).
// Hidden 6144, intermediate 2048, 168 experts: gate/up's vector instructions at T = 1111 3.16e8 -> 2.69e8, the decode kernel's at 6
// rows 8.6e7 -> 7.2e7; with the LDS slots that came with it the prefill call takes 1869 -> 1784 us, four decode layers 923 -> 909.
// k_gemv_sk, k_gemv over K slices at eight rows and the vector-unit decode kernels keep i4x8_to_bf16_any.
struct I4Group {
  float s, c0;   // the scale, -(1024 + u_z) s
  float s1, c1;  // s / 16, -(64 + u_z) s
};
constexpr float kI4MaxScale = 0x1p116f;  // I4Group's terms are exact below
__device__ __forceinline__ I4Group i4_group(float s, uint32_t uz) {
  I4Group g;
  g.s = s;
  g.c0 = -__fmul_rn((float)(uz | 1024u), s);
  g.s1 = __fmul_rn(s, 0.0625f);
  g.c1 = fmaf(960.f, s, g.c0);
  return g;
}
// whether any lane of the wave holds a scale that i4x8_to_bf16 is not for
__device__ __forceinline__ bool i4_any_large(float smax) { return __builtin_amdgcn_ballot_w64(!(fabsf(smax) < kI4MaxScale)) != 0; }
__device__ __forceinline__ uint32_t and_or(uint32_t v, uint32_t mask, uint32_t bits) {  // (v_and_or_b32 takes no literals: mask in a scalar register)
  uint32_t r;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(v), "s"(mask), "v"(bits));
  return r;
}
// half H (0 low, 1 high) of two f16 times s, plus c, rounded once to f32
template <int H>
__device__ __forceinline__ float fma_f16(uint32_t h, float s, float c) {
  float f;
  if (H == 0) asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel_hi:[1,0,0]" : "=v"(f) : "v"(h), "v"(s), "v"(c));
  else asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(f) : "v"(h), "v"(s), "v"(c));
  return f;
}
__device__ __forceinline__ void i4x8_to_bf16(uint32_t w, const I4Group& g, uint32_t (&o)[4]) {
  constexpr uint32_t k1024 = 0x64006400u;
  const uint32_t v = w >> 8;
  const uint32_t a = and_or(w, 0x000F000Fu, k1024), b = and_or(w, 0x00F000F0u, k1024);  // values 0 and 4, 1 and 5
  const uint32_t c = and_or(v, 0x000F000Fu, k1024), d = and_or(v, 0x00F000F0u, k1024);  // values 2 and 6, 3 and 7
  o[0] = pack_bf16(fma_f16<0>(a, g.s, g.c0), fma_f16<0>(b, g.s1, g.c1));
  o[1] = pack_bf16(fma_f16<0>(c, g.s, g.c0), fma_f16<0>(d, g.s1, g.c1));
  o[2] = pack_bf16(fma_f16<1>(a, g.s, g.c0), fma_f16<1>(b, g.s1, g.c1));
  o[3] = pack_bf16(fma_f16<1>(c, g.s, g.c0), fma_f16<1>(d, g.s1, g.c1));
}
// byte k of a word as a float, in one instruction (written as shifts and masks the compiler turns the masked nibbles
// back into a bit-field extract followed by a conversion: two instructions a value)
template <int K>
__device__ __forceinline__ float ubyte_to_f32(uint32_t w) {
  float f;
  if (K == 0) asm("v_cvt_f32_ubyte0 %0, %1" : "=v"(f) : "v"(w));
  else if (K == 1) asm("v_cvt_f32_ubyte1 %0, %1" : "=v"(f) : "v"(w));
  else if (K == 2) asm("v_cvt_f32_ubyte2 %0, %1" : "=v"(f) : "v"(w));
  else asm("v_cvt_f32_ubyte3 %0, %1" : "=v"(f) : "v"(w));
  return f;
}
// the same for every scale with a finite u_z * s (|s| < 2^124); nzs = -(u_z * s): fma(u, s, nzs) is the exact product
__device__ __forceinline__ void i4x8_to_bf16_any(uint32_t w, float s, float nzs, uint32_t (&o)[4]) {
  const uint32_t lo = w & 0x0F0F0F0Fu, hi = (w >> 4) & 0x0F0F0F0Fu;  // lo: values 0,2,4,6; hi: 1,3,5,7
  o[0] = pack_bf16(fmaf(ubyte_to_f32<0>(lo), s, nzs), fmaf(ubyte_to_f32<0>(hi), s, nzs));
  o[1] = pack_bf16(fmaf(ubyte_to_f32<1>(lo), s, nzs), fmaf(ubyte_to_f32<1>(hi), s, nzs));
  o[2] = pack_bf16(fmaf(ubyte_to_f32<2>(lo), s, nzs), fmaf(ubyte_to_f32<2>(hi), s, nzs));
  o[3] = pack_bf16(fmaf(ubyte_to_f32<3>(lo), s, nzs), fmaf(ubyte_to_f32<3>(hi), s, nzs));
}
// the contract in its subtract-first form, exact for every finite scale: bf16_rne(float(u - u_z) * s)
__device__ __forceinline__ uint32_t i4_value_bits(int u, int uz, uint32_t sbits) {
  return f32_to_bf16_bits((float)(u - uz) * bf16_bits_to_f32(sbits));
}

// ---- streaming loads (weights are read once: non-temporal) ---------------------------------------------------------------
// Pointers that come out of LDS tables (the slot descriptors) have lost their address space: the loads below cast
// them back to the global address space, so that they are global_load (vmcnt only) and not flat_load instructions.
#define DSGX_GLOBAL __attribute__((address_space(1)))
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ u32x4_t ldg_stream(const void* p) {
  return __builtin_nontemporal_load((const DSGX_GLOBAL u32x4_t*)(uintptr_t)p);
}
// The software pipelines below keep D steps of loads in flight in a ring of registers: step t is computed, then the
// load of step t + D is issued into the same registers. Two empty asm statements keep the compiler from undoing that:
// pin_after() makes a load's address depend on a value the preceding compute produced, so the load is not hoisted
// above the compute (which would need a second set of registers and copies that wait for the new data); keep_whole()
// passes a loaded 16-byte value through as one register tuple, so the loop-carried value is not split into scalars
// that no longer line up with the load's destination.
__device__ __forceinline__ const uint8_t* pin_after(const uint8_t* p, float dep) {
  uint64_t a = (uint64_t)p;
  asm volatile("" : "+v"(a) : "v"(dep));
  return (const uint8_t*)a;
}
__device__ __forceinline__ u32x4_t keep_whole(u32x4_t v) {
  asm volatile("" : "+v"(v));
  return v;
}
// Wave-uniform values. The compiler cannot know that a value read from LDS or derived from the wave's index is the
// same in every lane; uni() says so (v_readfirstlane), which moves the value and all arithmetic on it (row bases,
// cursors, loop bounds, branches) to the scalar unit and lets loads use the "scalar base + lane offset" addressing.
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ uint32_t uni(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }
__device__ __forceinline__ float uni(float v) { return __uint_as_float(uni(__float_as_uint(v))); }
__device__ __forceinline__ const uint8_t* uni(const uint8_t* p) {
  const uint64_t a = (uint64_t)p;
  return (const uint8_t*)(((uint64_t)uni((uint32_t)(a >> 32)) << 32) | uni((uint32_t)a));
}
// loads at (wave-uniform base) + (32-bit lane offset)
__device__ __forceinline__ u32x4_t ldg_stream(const uint8_t* base, uint32_t voff) {
  return __builtin_nontemporal_load((const DSGX_GLOBAL u32x4_t*)((const DSGX_GLOBAL uint8_t*)(uintptr_t)base + voff));
}
__device__ __forceinline__ uint32_t ldg_u32(const uint8_t* base, uint32_t voff) {
  return *(const DSGX_GLOBAL uint32_t*)((const DSGX_GLOBAL uint8_t*)(uintptr_t)base + voff);
}
__device__ __forceinline__ uint32_t ldg_u16(const uint8_t* base, uint32_t voff) {
  return *(const DSGX_GLOBAL uint16_t*)((const DSGX_GLOBAL uint8_t*)(uintptr_t)base + voff);
}
// pin_after() for a lane offset
__device__ __forceinline__ uint32_t pin_after(uint32_t voff, float dep) {
  asm volatile("" : "+v"(voff) : "v"(dep));
  return voff;
}
__device__ __forceinline__ uint32_t ldg_u32(const void* p) { return *(const DSGX_GLOBAL uint32_t*)(uintptr_t)p; }
__device__ __forceinline__ uint32_t ldg_u16(const void* p) { return *(const DSGX_GLOBAL uint16_t*)(uintptr_t)p; }

// ---- wave64 reductions, result valid in every lane -------------------------------------------------------------------------
// Steps 1, 2, 4, 8 run inside a row of 16 lanes with DPP (quad permutes and mirrors); rows are joined with gfx950's
// v_permlane16_swap / v_permlane32_swap: with both operands v, the two results hold each lane's own half and the other
// half, so their sum (or max) is the xor-16 / xor-32 butterfly step without a trip through LDS.
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_mov(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, true);
}
template <int CTRL>
__device__ __forceinline__ float dpp_add(float v) { return v + __uint_as_float(dpp_mov<CTRL>(__float_as_uint(v))); }
__device__ __forceinline__ float wave_sum(float v) {
  v = dpp_add<0xB1>(v);   // quad_perm [1,0,3,2]
  v = dpp_add<0x4E>(v);   // quad_perm [2,3,0,1]
  v = dpp_add<0x141>(v);  // row_half_mirror
  v = dpp_add<0x140>(v);  // row_mirror: every lane of a row of 16 holds the row's sum
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// The sums over the wave of N values a lane (N a power of two up to 16) for little more than the price of one: the two
// widest butterfly steps (lane distance 32, then 16) are done as FOLDS, a lane-half swap of two values' registers
// leaving one register with the first value's pair sums in one half of the lanes and the second's in the other, so
// N registers become N / 4 before the four narrow steps (8, 4, 2, 1 within a row of 16 lanes). Every value is summed
// by the same tree whatever N is, so a result does not depend on how many others were reduced with it.
// On return v[j] holds, in lane l with l % 16 == j, the sum of value fold_var<N>(l); the other lanes of the row hold the
// same sum. fold_owner<N>(l): lane l is the one lane that keeps its value (l % 16 < registers left).
template <int N>
__device__ __forceinline__ int fold_var(uint32_t lane) {
  if (N == 1) return 0;
  if (N == 2) return lane >> 5;
  return 4 * (lane & 15) + 2 * ((lane >> 4) & 1) + (lane >> 5);
}
template <int N>
__device__ __forceinline__ bool fold_owner(uint32_t lane) {
  if (N == 1) return lane == 0;
  if (N == 2) return (lane & 31) == 0;
  return (lane & 15) < N / 4;
}
template <int N>
__device__ __forceinline__ float fold_sum(float (&v)[N], uint32_t lane) {
  static_assert(N == 1 || N == 2 || N == 4 || N == 8 || N == 16, "fold_sum: 1, 2, 4, 8 or 16 values");
  auto add32 = [](float a, float b) {
    auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
  };
  auto add16 = [](float a, float b) {
    auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
  };
  constexpr int N1 = N >= 2 ? N / 2 : 1, N2 = N >= 4 ? N / 4 : 1;
#pragma unroll
  for (int j = 0; j < N1; ++j) v[j] = N >= 2 ? add32(v[2 * j], v[2 * j + 1]) : add32(v[0], v[0]);
#pragma unroll
  for (int j = 0; j < N2; ++j) v[j] = N >= 4 ? add16(v[2 * j], v[2 * j + 1]) : add16(v[0], v[0]);
#pragma unroll
  for (int j = 0; j < N2; ++j) {
    v[j] = dpp_add<0x140>(v[j]);  // row_mirror (distance 8: both lanes' rows of eight hold different eights)
    v[j] = dpp_add<0x141>(v[j]);  // row_half_mirror
    v[j] = dpp_add<0x4E>(v[j]);   // quad_perm [2,3,0,1]
    v[j] = dpp_add<0xB1>(v[j]);   // quad_perm [1,0,3,2]
  }
  float r = v[0];
#pragma unroll
  for (int j = 1; j < N2; ++j) r = (lane & 15) == (uint32_t)j ? v[j] : r;
  return r;
}

// ---- the activation layout in LDS ---------------------------------------------------------------------------------------------
// A lane of a wavefront that streams a row holds KL consecutive k per segment of 64 * KL k (KL = 16 for FP8: one
// 16-byte load; 32 for INT4: one 16-byte load; 8, 16 or 32 for BF16: one, two or four 16-byte loads). The activations
// of row m are staged as 16-byte chunks of 8 k so that the lanes of a wavefront read consecutive chunks (no bank
// conflicts): chunk c (of KL / 8) of segment s of lane l sits at chunk index ((s * (KL / 8) + c) * 64 + l) of the row.
template <int KL>
__device__ __forceinline__ int xchunk_index(int q) {  // q: the row's chunk number in k order (k = 8 q)
  constexpr int XC = KL / 8;
  const int seg = q / (64 * XC), r = q % (64 * XC);
  return (seg * XC + r % XC) * 64 + r / XC;
}
// Stage rows x[M][ldx] (bf16, global) into lds [M][K/8 chunks] in the layout above; K a multiple of 8. Chunks past K in
// the last segment are zero-filled up to Kpad (a multiple of 64 * KL).
// COHERENT: read with device-scope coherent loads (data written by other workgroups of the same kernel).
// Eight chunks a thread are loaded before any is written to LDS, so their latencies overlap.
template <bool COHERENT>
__device__ __forceinline__ uint4 load_chunk(const uint16_t* p) {
  if (COHERENT) {
    const uint64_t* q = reinterpret_cast<const uint64_t*>(p);
    const uint64_t a = __hip_atomic_load((const DSGX_GLOBAL uint64_t*)(uintptr_t)q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint64_t b = __hip_atomic_load((const DSGX_GLOBAL uint64_t*)(uintptr_t)(q + 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return make_uint4((uint32_t)a, (uint32_t)(a >> 32), (uint32_t)b, (uint32_t)(b >> 32));
  }
  const u32x4_t v = *(const DSGX_GLOBAL u32x4_t*)(uintptr_t)p;
  return make_uint4(v.x, v.y, v.z, v.w);
}
template <int KL, bool COHERENT = false>
__device__ __forceinline__ void stage_x(uint4* lds, const uint16_t* x, size_t ldx, int M, int K, int Kpad) {
  const int nq = Kpad / 8, total = M * nq;
  constexpr int U = 8;
  for (int i0 = threadIdx.x; i0 < total; i0 += U * blockDim.x) {
    uint4 v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = i0 + u * blockDim.x;
      v[u] = make_uint4(0, 0, 0, 0);
      if (i < total) {
        const int m = i / nq, q = i % nq;
        if (8 * q < K) v[u] = load_chunk<COHERENT>(x + (size_t)m * ldx + 8 * q);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = i0 + u * blockDim.x;
      if (i < total) lds[(size_t)(i / nq) * nq + xchunk_index<KL>(i % nq)] = v[u];
    }
  }
}
// The same for `ns` consecutive slots of h (each M rows of K = ldx values) staged back to back: one pass over all of
// them, so that a chunk of slots costs one round trip and not one a slot. base(s) gives slot s's rows.
template <int KL, bool COHERENT, class Base>
__device__ __forceinline__ void stage_slots(uint4* lds, int ns, int M, int K, Base&& base) {
  const int nq = K / 8, per = M * nq, total = ns * per;
  constexpr int U = 8;
  for (int i0 = threadIdx.x; i0 < total; i0 += U * blockDim.x) {
    uint4 v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = i0 + u * blockDim.x;
      v[u] = make_uint4(0, 0, 0, 0);
      if (i < total) {
        const int s = i / per, r = i % per;
        v[u] = load_chunk<COHERENT>(base(s) + (size_t)(r / nq) * K + 8 * (r % nq));
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = i0 + u * blockDim.x;
      if (i < total) {
        const int s = i / per, r = i % per;
        lds[(size_t)s * per + (size_t)(r / nq) * nq + xchunk_index<KL>(r % nq)] = v[u];
      }
    }
  }
}

// ---- the router's row function (one wavefront a row) ------------------------------------------------------------------------------
// s = 1 / (1 + e^-l) from IEEE operations only, so the CPU and the GPU give the same bits: the reference's
// route_sigmoid (engine/experts/formats.cuh:142-163).
__device__ __forceinline__ float route_sigmoid(float l) {
  const float x = -l;
  if (x > 88.f) return 0.f;
  if (x < -87.f) return 1.f;
  const float n = rintf(x * 1.44269504f);
  float r = fmaf(-n, 0.693145751953125f, x);
  r = fmaf(-n, 1.428606765330187e-06f, r);
  float p = 1.f / 5040;
  p = fmaf(p, r, 1.f / 720);
  p = fmaf(p, r, 1.f / 120);
  p = fmaf(p, r, 1.f / 24);
  p = fmaf(p, r, 1.f / 6);
  p = fmaf(p, r, 0.5f);
  p = fmaf(p, r, 1.f);
  p = fmaf(p, r, 1.f);
  const float e = ldexpf(p, (int)n);
  return __fdiv_rn(1.f, __fadd_rn(1.f, e));
}
// softplus(l) = log1p(exp(l)) for l <= 20, again from IEEE operations only (the reference's log1pf(expf(l)),
// ds41f-4xgx10-switchless/engine/kernels/common.cuh:281, depends on the math library): exp by the sigmoid's reduction and
// polynomial; log1p(e) = log(u) e / (u - 1) with u = 1 + e; log by u = 2^k (1 + f), sqrt(1/2) < 1 + f < sqrt(2),
// s = f / (2 + f), log(1 + f) = f - f^2/2 + s (f^2/2 + R(s^2)), R the degree-7 minimax of fdlibm's e_logf.c. Every
// operation is written out and rounded on its own, so the host oracle's copy gives the same bits.
__device__ __forceinline__ float route_softplus(float l) {
  if (l < -87.f) l = -87.f;
  const float n = rintf(__fmul_rn(l, 1.44269504f));
  float r = fmaf(-n, 0.693145751953125f, l);
  r = fmaf(-n, 1.428606765330187e-06f, r);
  float p = 1.f / 5040;
  p = fmaf(p, r, 1.f / 720);
  p = fmaf(p, r, 1.f / 120);
  p = fmaf(p, r, 1.f / 24);
  p = fmaf(p, r, 1.f / 6);
  p = fmaf(p, r, 0.5f);
  p = fmaf(p, r, 1.f);
  p = fmaf(p, r, 1.f);
  const float e = ldexpf(p, (int)n);
  const float u = __fadd_rn(1.f, e);
  if (u == 1.f) return e;
  uint32_t ix = __float_as_uint(u);
  int k = (int)(ix >> 23) - 127;
  ix &= 0x007fffffu;
  const uint32_t i = (ix + (0x95f64u << 3)) & 0x800000u;
  ix |= i ^ 0x3f800000u;
  k += (int)(i >> 23);
  const float f = __fsub_rn(__uint_as_float(ix), 1.f), dk = (float)k;
  const float s_ = __fdiv_rn(f, __fadd_rn(2.f, f)), z = __fmul_rn(s_, s_), w = __fmul_rn(z, z);
  const float t1 = __fmul_rn(w, __fadd_rn(0.40000000596f, __fmul_rn(w, __fadd_rn(0.22222198546f, __fmul_rn(w, 0.15313838422f)))));
  const float t2 = __fmul_rn(z, __fadd_rn(0.66666668653f, __fmul_rn(w, __fadd_rn(0.28571429849f, __fmul_rn(w, __fadd_rn(0.18183572590f, __fmul_rn(w, 0.14798198640f)))))));
  const float R = __fadd_rn(t2, t1), hfsq = __fmul_rn(__fmul_rn(0.5f, f), f);
  const float inner = __fadd_rn(__fmul_rn(s_, __fadd_rn(hfsq, R)), __fmul_rn(dk, 9.0580006145e-06f));
  const float lg = __fsub_rn(__fmul_rn(dk, 0.69313812256f), __fsub_rn(__fsub_rn(hfsq, inner), f));
  return __fmul_rn(lg, __fdiv_rn(e, __fsub_rn(u, 1.f)));
}
__device__ __forceinline__ float route_score(float l, int score_fn) {
  if (score_fn == 0) return route_sigmoid(l);
  return sqrtf(l > 20.f ? l : route_softplus(l));  // DeepSeek's sqrt(softplus); sqrtf is the correctly rounded root (__fsqrt_rn is not)
}
// wave-wide maximum of floats (no NaNs), valid in every lane
template <int CTRL>
__device__ __forceinline__ float dpp_max(float v) { return fmaxf(v, __uint_as_float(dpp_mov<CTRL>(__float_as_uint(v)))); }
__device__ __forceinline__ float wave_max_f32(float v) {
  v = dpp_max<0xB1>(v);
  v = dpp_max<0x4E>(v);
  v = dpp_max<0x141>(v);
  v = dpp_max<0x140>(v);
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// wave-wide minimum of unsigned ints, valid in every lane
__device__ __forceinline__ uint32_t wave_min_u32(uint32_t v) {
  v = min(v, dpp_mov<0xB1>(v));
  v = min(v, dpp_mov<0x4E>(v));
  v = min(v, dpp_mov<0x141>(v));
  v = min(v, dpp_mov<0x140>(v));
  auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  v = min(r[0], r[1]);
  r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  return min(r[0], r[1]);
}

// wave-wide maximum of unsigned ints, valid in every lane
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
  v = max(v, dpp_mov<0xB1>(v));
  v = max(v, dpp_mov<0x4E>(v));
  v = max(v, dpp_mov<0x141>(v));
  v = max(v, dpp_mov<0x140>(v));
  auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  v = max(r[0], r[1]);
  r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  return max(r[0], r[1]);
}
// a float's bits as an unsigned int of the same order (no NaNs; -0 does not occur: a score is never negative zero)
__device__ __forceinline__ uint32_t f32_order_bits(float f) {
  const uint32_t b = __float_as_uint(f);
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}

// One row by one wavefront: experts e = lane + 64 j, j < NJ (E <= 64 NJ). Lane k < topk gets pick k's expert and
// weight (route_warp of the reference, engine/experts/formats.cuh:207-247, at 64 lanes): descending key (float
// compares), ties to the lower id; the sum in the butterfly order ((p0+p4)+(p2+p6))+((p1+p5)+(p3+p7)), absent places
// skipped. The code runs once a launch on a single wavefront, so its instruction count is its latency:
//  - every lane first sorts its NJ places by (key descending, j ascending) with adjacent exchanges (stable);
//  - a pick is the wave-wide maximum of the lanes' heads; the lane holding it (on a tie, rare, the lowest expert id
//    among the heads that hold it: a lane's own ties are already in id order) pops its list.
constexpr int kRouteRJ = DSGX_MAX_EXPERTS / kWave;
// a row's logits (or the bias; null: zeros) in the lanes' places; E wave-uniform
__device__ __forceinline__ void route_fetch(const float* __restrict__ row, int E, int lane, float (&v)[kRouteRJ]) {
  const int nj = (E + kWave - 1) / kWave;
#pragma unroll
  for (int j = 0; j < kRouteRJ; ++j) {
    const int e = lane + kWave * j;
    v[j] = 0.f;
    if (row && j < nj && e < E) v[j] = row[e];
  }
}
template <int NJ>
__device__ __forceinline__ void route_row_nj(const float (&logit)[kRouteRJ], const float (&bias)[kRouteRJ], int E, int topk, float scale,
                                             int score_fn, int lane, int& id_out, float& w_out) {
  // The keys are compared as unsigned ints of the floats' order (f32_order_bits): the wave-wide maximum is then one
  // instruction a step, a third of the float form's (which re-canonicalises its operands). 0 is below every key.
  constexpr uint32_t kDead = 0u;
  float s[NJ];
  uint32_t key[NJ];
  int jj[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    s[j] = 0.f, key[j] = kDead, jj[j] = j;  // an empty place never wins
    if (lane + kWave * j < E) {
      s[j] = route_score(logit[j], score_fn);
      key[j] = f32_order_bits(__fadd_rn(s[j], bias[j]));
    }
  }
  // odd-even transposition: NJ passes of adjacent exchanges, strictly-greater only (equal keys keep their j order)
#pragma unroll
  for (int pass = 0; pass < NJ; ++pass)
#pragma unroll
    for (int j = pass & 1; j + 1 < NJ; j += 2) {
      const bool sw = key[j + 1] > key[j];
      const uint32_t k0 = key[j];
      const float s0 = s[j];
      const int j0 = jj[j];
      key[j] = sw ? key[j + 1] : k0, s[j] = sw ? s[j + 1] : s0, jj[j] = sw ? jj[j + 1] : j0;
      key[j + 1] = sw ? k0 : key[j + 1], s[j + 1] = sw ? s0 : s[j + 1], jj[j + 1] = sw ? j0 : jj[j + 1];
    }
  // lane k keeps pick k; the loop is not unrolled
  float my_s = 0.f;
  int my_id = 0;
#pragma unroll 1
  for (int k = 0; k < topk; ++k) {
    const uint32_t top = wave_max_u32(key[0]);
    const uint64_t hit = __ballot(key[0] == top);
    int wl = __builtin_ctzll(hit);
    if (hit & (hit - 1)) wl = wave_min_u32(key[0] == top ? (uint32_t)(lane + kWave * jj[0]) : 0xFFFFFFFFu) & (kWave - 1);
    const int id = wl + kWave * __builtin_amdgcn_readlane(jj[0], wl);
    const float sv = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(s[0]), wl));
    if (lane == wl) {
#pragma unroll
      for (int j = 0; j + 1 < NJ; ++j) key[j] = key[j + 1], s[j] = s[j + 1], jj[j] = jj[j + 1];
      key[NJ - 1] = kDead;
    }
    if (lane == k) my_s = sv, my_id = id;
  }
  // lanes 0..7 hold p0..p7 (0 past topk: x + 0 = x): three xor steps are the reference's order of adds
  float sum = my_s;
  sum = __fadd_rn(sum, __shfl_xor(sum, 4));
  sum = __fadd_rn(sum, __shfl_xor(sum, 2));
  sum = __fadd_rn(sum, __shfl_xor(sum, 1));
  sum = __fadd_rn(sum, 1e-20f);
  id_out = my_id, w_out = lane < topk ? __fmul_rn(__fdiv_rn(my_s, sum), scale) : 0.f;
}
__device__ __forceinline__ void route_row(const float (&logit)[kRouteRJ], const float (&bias)[kRouteRJ], int E, int topk, float scale,
                                          int score_fn, int lane, int& id_out, float& w_out) {
  if (E <= 2 * kWave) route_row_nj<2>(logit, bias, E, topk, scale, score_fn, lane, id_out, w_out);
  else if (E <= 4 * kWave) route_row_nj<4>(logit, bias, E, topk, scale, score_fn, lane, id_out, w_out);
  else route_row_nj<kRouteRJ>(logit, bias, E, topk, scale, score_fn, lane, id_out, w_out);
}

__device__ __forceinline__ float bf16_lo(uint32_t p) { return __uint_as_float(p << 16); }  // the values of a packed pair
__device__ __forceinline__ float bf16_hi(uint32_t p) { return __uint_as_float(p & 0xFFFF0000u); }
// silu(g) = g / (1 + e^-g) of four values in f32, the division IEEE's: by the divisor's reciprocal and one correction step where
// |g| < 60 (the divisor is then in [1, 2^87]: no scaling; equal to the division for every f32 g there, all compared, so a gate clamped
// to a limit that is no bf16 value is in; a zero takes g's sign), by the division itself if a value of the wave lies outside.
__device__ __forceinline__ void silu4(const float (&g)[4], float (&s)[4]) {
  float d[4];
  bool far = false;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    d[i] = __fadd_rn(1.f, expf(-g[i]));
    const float r = __builtin_amdgcn_rcpf(d[i]), q = __fmul_rn(g[i], r);
    s[i] = __builtin_copysignf(fmaf(fmaf(-q, d[i], g[i]), r, q), g[i]);
    far |= !(fabsf(g[i]) < 60.f);
  }
  if (__builtin_expect(__builtin_amdgcn_ballot_w64(far) != 0, 0)) {
#pragma unroll
    for (int i = 0; i < 4; ++i) s[i] = __fdiv_rn(g[i], d[i]);
  }
}
// bf16(g / (1 + e^-g)) of a bf16 value g: where only the rounded value is used, the hardware's exponential and reciprocal do, without
// expf()'s range reduction, the correction step and the cases apart (9 vector instructions less a value). Both sides of the quotient
// are a quarter of theirs, which keeps the reciprocal normal up to the largest finite divisor, and the quarter of the divisor's 1 is one
// step above 1/4: of the 65536 bf16 values, NaN, infinities and zeros included, every one rounds to the bits that the exact sequence
// (expf, IEEE division) rounds to (all compared; with 1/4 itself 5.9375 alone does not). The prefill GEMMs' epilogues are bound by the
// vector unit (as kernels of eight waves the FP8 gate/up tile of 256 positions spent an eighth of
// its time there): FP8 gate/up at 256 rows an expert 1366 -> 1326 us, Zipf T = 8192 2919 -> 2876; INT4 at 64 rows an expert 1490 -> 1461.
__device__ __forceinline__ float silu_for_bf16(float g) {
  const float e = __builtin_amdgcn_exp2f(fmaf(g, -1.44269504088896341f, -2.f));
  return __fmul_rn(__fmul_rn(g, 0.25f), __builtin_amdgcn_rcpf(__fadd_rn(0x1.000002p-2f, e)));
}
// Four of swiglu_bits' values, packed (g, u: bf16 values). fast: the same function by the plain formula, the caller's choice: silu of four
// bf16 gates is another, one step at 5.9375 and -0 at -87.5, -88 and -88.5, whose divisor's reciprocal is not normal.
__device__ __forceinline__ uint2 swiglu4(const float (&g)[4], const float (&u)[4], bool fast) {
  float s[4];
  if (fast) {
#pragma unroll
    for (int i = 0; i < 4; ++i) s[i] = __fmul_rn(g[i], __builtin_amdgcn_rcpf(__fadd_rn(1.f, __builtin_amdgcn_exp2f(__fmul_rn(g[i], -1.44269504088896341f)))));
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) s[i] = silu_for_bf16(g[i]);
  }
  const uint32_t a = pack_bf16(s[0], s[1]), b = pack_bf16(s[2], s[3]);
  return make_uint2(pack_bf16(__fmul_rn(bf16_lo(a), u[0]), __fmul_rn(bf16_hi(a), u[1])), pack_bf16(__fmul_rn(bf16_lo(b), u[2]), __fmul_rn(bf16_hi(b), u[3])));
}
// the accumulators' four values times a matrix's scale, rounded to bf16
template <class V>
__device__ __forceinline__ void bf16_round4(const V& acc, float s2, float (&o)[4]) {
  const uint32_t a = pack_bf16(__fmul_rn(acc[0], s2), __fmul_rn(acc[1], s2)), b = pack_bf16(__fmul_rn(acc[2], s2), __fmul_rn(acc[3], s2));
  o[0] = bf16_lo(a), o[1] = bf16_hi(a), o[2] = bf16_lo(b), o[3] = bf16_hi(b);
}

// h = bf16(bf16(silu(g)) * u), g and u already bf16 values (engine/experts/decode.cu:110-113 of the reference)
__device__ __forceinline__ uint32_t swiglu_bits(float g, float u) {
  const float sl = bf16_round(__fdiv_rn(g, __fadd_rn(1.f, expf(-g))));
  return f32_to_bf16_bits(__fmul_rn(sl, u));
}

// v / d by d's reciprocal (r = rcp(d), within 1 ulp) and one correction step: the quotient rounded to nearest for every v
// and d met here (normal numbers far from the format's ends; the IEEE sequence spends twice the instructions on scaling
// for the ends). Checked against the division bit for bit in tests.
__device__ __forceinline__ float div_by(float v, float d, float r) {
  const float q = __fmul_rn(v, r);
  return fmaf(fmaf(-q, d, v), r, q);
}

// act_quant(x, 128): sixteen lanes a (row, 128-k block), eight values (one 16-byte load) a lane; the block's largest
// magnitude by four DPP steps within the row of 16 lanes
// (ds41f-4xgx10-switchless/ref/torchref/kernel.py:56-77 of the reference, scale_fmt None)
__device__ __forceinline__ void act_quant_block(const uint16_t* __restrict__ x, int T, int K, size_t blk, uint8_t* __restrict__ q, float* __restrict__ s) {
  const int KB = K / 128, l16 = threadIdx.x & 15;
  if (blk >= (size_t)T * KB) return;  // (whole rows of 16 lanes leave together)
  const size_t t = blk / KB, b = blk % KB, at = t * K + 128 * b + 8 * l16;
  const u32x4_t xv = *reinterpret_cast<const DSGX_GLOBAL u32x4_t*>((uintptr_t)(x + at));
  float v[8];
#pragma unroll
  for (int i = 0; i < 4; ++i) v[2 * i] = bf16_bits_to_f32(xv[i] & 0xFFFFu), v[2 * i + 1] = bf16_bits_to_f32(xv[i] >> 16);
  float amax = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) amax = fmaxf(amax, fabsf(v[i]));
  amax = dpp_max<0xB1>(amax);
  amax = dpp_max<0x4E>(amax);
  amax = dpp_max<0x141>(amax);
  amax = dpp_max<0x140>(amax);
  amax = fmaxf(amax, 1e-4f);
  const float sc = __fmul_rn(amax, 1.0f / 448.0f);
  if (l16 == 0) s[t * KB + b] = sc;
  float qv[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) qv[i] = fminf(448.f, fmaxf(-448.f, __fdiv_rn(v[i], sc)));
  uint32_t o[2];
  o[0] = __builtin_amdgcn_cvt_pk_fp8_f32(qv[0], qv[1], 0, false);
  o[0] = __builtin_amdgcn_cvt_pk_fp8_f32(qv[2], qv[3], o[0], true);
  o[1] = __builtin_amdgcn_cvt_pk_fp8_f32(qv[4], qv[5], 0, false);
  o[1] = __builtin_amdgcn_cvt_pk_fp8_f32(qv[6], qv[7], o[1], true);
  *reinterpret_cast<uint2*>(q + at) = make_uint2(o[0], o[1]);
}

}  // namespace dsgx
