// prefill.h — device helpers shared by the prompt-row kernels (prefill.hip,
// prefill_gemm.hip).
#pragma once

#include "common.h"
#include "uaii_hip_internal.h"

namespace uaii_hip {

typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
typedef _Float16 h4_t __attribute__((ext_vector_type(4)));
typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
typedef float f4_t __attribute__((ext_vector_type(4)));

__device__ inline h2_t as_h2(uint32_t u) { return __builtin_bit_cast(h2_t, u); }
// (v & m) | c in one v_and_or_b32. Written out because gfx9's three-operand
// encoding takes no literal constants, so the compiler splits the expression
// into v_and + v_or; here the mask sits in a scalar register and the constant
// in a vector register, both loop-invariant.
__device__ inline uint32_t and_or(uint32_t v, uint32_t m, uint32_t c) {
  uint32_t r;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(v), "s"(m), "v"(c));
  return r;
}
// bytes 0 and 2 as f16 (1024 + b)
__device__ inline uint32_t byte_pair(uint32_t v) { return and_or(v, 0x00FF00FFu, 0x64006400u); }

__device__ inline h8_t cat8(h2_t a, h2_t b, h2_t c, h2_t d) {
  return h8_t{a.x, a.y, b.x, b.y, c.x, c.y, d.x, d.y};
}

// Operands of the 16x16x32 f16 MFMA (CDNA3/CDNA4): lane l supplies row l % 16 of A
// and column l % 16 of B with k-group l / 16; D[4 (l / 16) + r][l % 16] sits in
// element r of lane l. The order of k inside a lane's group only has to agree
// between A and B.
__device__ inline f4_t mfma32(h8_t a, h8_t b, f4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// The 16x16x4 f32 MFMA: lane l supplies A[l % 16][l / 16] and B[l / 16][l % 16]; D as above.
__device__ inline f4_t mfma4(float a, float b, f4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// The sum of n K-split partials: pairs, pairs of pairs, then the groups of four in order.
// One after another, 16 or 32 roundings at the sum's own size were a third of a product's
// error (9 rows, 1024 x 14336 Q8_0, 32 splits: 1.41e-7 of the result).
template <class V, class F>
__device__ inline V split_sum(int n, F&& load) {
  V s = {};
  for (int z = 0; z < n; z += 4) {
    const int m = n - z;  // at least 1
    V a = load(z), b = {}, c = {}, d = {};
    if (m > 1) b = load(z + 1);
    if (m > 2) c = load(z + 2);
    if (m > 3) d = load(z + 3);
    s += (a + b) + (c + d);
  }
  return s;
}

__device__ inline float pow2f_i(int e) { return __uint_as_float((uint32_t)(e + 127) << 23); }

// 16 bytes per lane from a wave-uniform base (scalar registers) plus the lane's
// 32-bit byte offset into LDS at `lds` + 16 lane. The load is issued from inline
// assembly and its completion waited for with an explicit vmcnt: the compiler
// would otherwise wait for every outstanding LDS load before each LDS read. The
// LDS address goes to the asm as an M0 operand ("{m0}"), so the compiler writes M0
// itself and knows it holds that value; the s_nop gives the one wait state an LDS
// DMA needs after an M0 write.
__device__ inline void dma16s(const void* sbase, uint32_t voff, uint32_t lds) {
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"{m0}"(lds), "v"(voff), "s"(sbase)
               : "memory");
}
// The same from a per-lane address; 4 bytes per lane to `lds` + 4 lane.
__device__ inline void dma16(const void* g, uint32_t lds) {
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"{m0}"(lds), "v"(g) : "memory");
}
__device__ inline void dma4(const void* g, uint32_t lds) {
  asm volatile("s_nop 0\n\tglobal_load_lds_dword %1, off" ::"{m0}"(lds), "v"(g) : "memory");
}
// A pointer the wave holds in common, made visibly uniform so that it lives in
// scalar registers.
__device__ inline const uint8_t* uniform_ptr(const void* p) {
  const uint64_t u = (uint64_t)(uintptr_t)p;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)u);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(u >> 32));
  return reinterpret_cast<const uint8_t*>((uintptr_t)(((uint64_t)hi << 32) | lo));
}
__device__ inline uint32_t lds_addr(const void* p) {
  return __builtin_amdgcn_readfirstlane(
      (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p);
}

// silu (elementwise.cpp:73-84) and the tanh form of gelu (elementwise.cpp:56-71)
__device__ inline float pf_silu(float v) { return v / (1.0f + expf(-v)); }
__device__ inline float pf_gelu(float v) {
  const float inner = 0.7978845608f * (v + 0.044715f * v * v * v);
  return 0.5f * v * (1.0f + tanhf(inner));
}

}  // namespace uaii_hip
