// prefill_attn_f32.hip — causal attention of M prompt positions over an f32 KV
// cache (attention_kv_f32 applied to each query in turn,
// libs/uaii-kernels/src/transformer.cpp:222-433).
//
// Keys, values, queries, scores and probabilities stay f32: the contractions run
// on v_mfma_f32_16x16x4_f32, whose products and sums are f32 as the token step's
// are. That instruction does 64 multiply-adds' worth of flops per cycle and SIMD
// (157 TFLOP/s dense, a sixteenth of the f16 rate), which is still far ahead of
// what bounds a prompt: its GEMMs. 1000 positions from 0, 32/8 heads of 64: 87 us a
// layer, where token steps over the f32 cache took 1000 x 0.69 ms for all 16 layers
// (whole run of 1000 + 8 ids 691 -> 14.4 ms).
//
// Operands of 16x16x4: lane l supplies A[l % 16][l / 16] and B[l / 16][l % 16],
// D[4 (l / 16) + r][l % 16] sits in element r. With S^T = K . Q^T the lane then
// holds keys 4 g + r (g = l / 16) of query l % 16, which is exactly the B operand
// of O^T += V^T . P^T when step r of a 16-key subtile takes key 4 g + r as its
// k index g: the probabilities never leave their registers. The K operand's four
// consecutive steps take dims 16 c + 4 g + t (t = 0..3), one 16-byte read per
// lane for four instructions.
#include "common.h"
#include "uaii_hip_internal.h"

namespace uaii_hip {
namespace {

typedef float f4_t __attribute__((ext_vector_type(4)));

constexpr int PAF_TK = 32;  // keys per LDS tile: K and V double-buffered leave two blocks per CU

__device__ inline f4_t mfma4(float a, float b, f4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Block: 4 waves on one kv head; wave w takes query head w % GW of the block's GW
// heads and the 16 queries of subtile w / GW. Rows of both tiles are HD + 4 floats
// long: 4 words past a multiple of 64, so the 16 keys' K reads and the 4 x 16
// words of a V read fall into distinct banks. Query tiles run last-first: the
// last ones read the most keys and would otherwise end the launch alone.
template <int HD>
__global__ void __launch_bounds__(256, 2) k_pf_attn_f32(PfAttnArgs a) {
  constexpr int KP = HD + 4;
  constexpr int NC = HD / 16;                    // 16-dim chunks
  constexpr int PIECES = PAF_TK * (HD / 4) / 256;  // float4 pieces of a tile per thread
  __shared__ __attribute__((aligned(16))) float ks[2][PAF_TK * KP];
  __shared__ __attribute__((aligned(16))) float vs[2][PAF_TK * KP];

  const int G = a.n_heads / a.n_kv;
  const int GW = G < 4 ? G : 4;
  const int QS = 4 / GW;
  const int hb = blockIdx.y;
  const int kvh = hb / (G / GW);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, col = lane & 15, g = lane >> 4;
  const bool active = wave < GW * QS;
  const int head = kvh * G + (hb % (G / GW)) * GW + (wave % GW);
  const int64_t q0 = (int64_t)(gridDim.x - 1 - blockIdx.x) * (16 * QS);
  const int64_t qw0 = q0 + 16 * (wave / GW);
  const int64_t nkeys = a.p0 + min((int64_t)a.M, q0 + 16 * QS);  // keys the block needs (causal)
  const int64_t qrow = qw0 + col;
  const bool qvalid = active && qrow < a.M;
  const int qpos = (int)(a.p0 + qrow);
  const int64_t qpos0 = a.p0 + qw0;

  const float scale = 1.0f / sqrtf((float)HD);
  float4 q[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    q[c] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (qvalid) {
      q[c] = *reinterpret_cast<const float4*>(a.q + qrow * a.ldq + (int64_t)head * HD + 16 * c + 4 * g);
      q[c].x *= scale; q[c].y *= scale; q[c].z *= scale; q[c].w *= scale;
    }
  }
  f4_t o[NC];
#pragma unroll
  for (int d = 0; d < NC; ++d) o[d] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
  float mrun = -INFINITY, lrun = 0.0f;

  const float* kbase = reinterpret_cast<const float*>(a.kcache) + (int64_t)kvh * a.max_seq * HD;
  const float* vbase = reinterpret_cast<const float*>(a.vcache) + (int64_t)kvh * a.max_seq * HD;
  // keys past nkeys read as zeros (their scores are masked)
  float4 kreg[PIECES], vreg[PIECES];
  auto load_tile = [&](int64_t kt) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < PIECES; ++u) {
      const int c = threadIdx.x + 256 * u;
      const int key = c / (HD / 4), p = c % (HD / 4);
      kreg[u] = vreg[u] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      if (kt + key < nkeys) {
        kreg[u] = *reinterpret_cast<const float4*>(kbase + (kt + key) * HD + 4 * p);
        vreg[u] = *reinterpret_cast<const float4*>(vbase + (kt + key) * HD + 4 * p);
      }
    }
  };
  auto store_tile = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < PIECES; ++u) {
      const int c = threadIdx.x + 256 * u;
      const int key = c / (HD / 4), p = c % (HD / 4);
      *reinterpret_cast<float4*>(&ks[buf][key * KP + 4 * p]) = kreg[u];
      *reinterpret_cast<float4*>(&vs[buf][key * KP + 4 * p]) = vreg[u];
    }
  };
  auto lds_barrier = []() __attribute__((always_inline)) {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the next tile's loads stay in flight
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  auto compute = [&](int64_t kt, int buf) __attribute__((always_inline)) {
    constexpr float kLog2e = 1.4426950408889634f;
    f4_t sc[2] = {f4_t{0.0f, 0.0f, 0.0f, 0.0f}, f4_t{0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      float4 kf[2];
#pragma unroll
      for (int s = 0; s < 2; ++s)
        kf[s] = *reinterpret_cast<const float4*>(&ks[buf][(16 * s + col) * KP + 16 * c + 4 * g]);
#pragma unroll
      for (int s = 0; s < 2; ++s) sc[s] = mfma4(kf[s].x, q[c].x, sc[s]);
#pragma unroll
      for (int s = 0; s < 2; ++s) sc[s] = mfma4(kf[s].y, q[c].y, sc[s]);
#pragma unroll
      for (int s = 0; s < 2; ++s) sc[s] = mfma4(kf[s].z, q[c].z, sc[s]);
#pragma unroll
      for (int s = 0; s < 2; ++s) sc[s] = mfma4(kf[s].w, q[c].w, sc[s]);
    }
    if (kt + PAF_TK - 1 > qpos0) {  // the tile reaches past the wave's first query
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if ((int)kt + 16 * s + 4 * g + r > qpos) sc[s][r] = -INFINITY;
    }
    float tmax = -INFINITY;
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int r = 0; r < 4; ++r) tmax = fmaxf(tmax, sc[s][r]);
    tmax = fmaxf(tmax, __shfl_xor(tmax, 16, 64));
    tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
    // running max and exponentials in base 2
    const float mnew = fmaxf(mrun, tmax * kLog2e);
    const float alpha = (mrun == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f(mrun - mnew);
    const float mref = (mnew == -INFINITY) ? 0.0f : mnew;  // a fully masked row so far: p = 0
    float psum = 0.0f;
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        sc[s][r] = __builtin_amdgcn_exp2f(fmaf(sc[s][r], kLog2e, -mref));
        psum += sc[s][r];
      }
    psum += __shfl_xor(psum, 16, 64);
    psum += __shfl_xor(psum, 32, 64);
    lrun = lrun * alpha + psum;
    mrun = mnew;
    if (__any(alpha != 1.0f)) {
#pragma unroll
      for (int d = 0; d < NC; ++d) o[d] *= alpha;
    }
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float* vr = &vs[buf][(16 * s + 4 * g + r) * KP + col];
#pragma unroll
        for (int d = 0; d < NC; ++d) o[d] = mfma4(vr[16 * d], sc[s][r], o[d]);
      }
  };

  load_tile(0);
  store_tile(0);
  lds_barrier();
  int buf = 0;
  for (int64_t kt = 0; kt < nkeys; kt += PAF_TK) {
    const bool more = kt + PAF_TK < nkeys;  // block-uniform
    if (more) load_tile(kt + PAF_TK);
    // a wave whose queries all lie before the tile has nothing to add
    if (active && kt <= qpos0 + 15) compute(kt, buf);
    if (more) store_tile(buf ^ 1);
    lds_barrier();
    buf ^= 1;
  }

  if (!qvalid) return;
  const float inv = 1.0f / lrun;
  float* out = a.out + qrow * a.ldo + (int64_t)head * HD;
#pragma unroll
  for (int d = 0; d < NC; ++d)
    *reinterpret_cast<float4*>(out + 16 * d + 4 * g) =
        make_float4(o[d][0] * inv, o[d][1] * inv, o[d][2] * inv, o[d][3] * inv);
}

}  // namespace

hipError_t launch_pf_attn_f32(const PfAttnArgs& a, hipStream_t s) {
  if (a.M <= 0 || a.p0 < 0 || a.p0 + a.M > a.max_seq || a.max_seq > INT32_MAX ||
      !pf_attn_supported(a.hd, a.n_heads, a.n_kv) || a.ldq % 4 || a.ldo % 4)
    return hipErrorInvalidValue;
  const int G = a.n_heads / a.n_kv;
  const int GW = G < 4 ? G : 4;
  const int QT = 16 * (4 / GW);  // queries per block
  dim3 grid((unsigned)((a.M + QT - 1) / QT), (unsigned)(a.n_kv * (G / GW)));
  if (a.hd == 64) UAII_LAUNCH(k_pf_attn_f32<64>, grid, dim3(256), 0, s, a);
  else UAII_LAUNCH(k_pf_attn_f32<128>, grid, dim3(256), 0, s, a);
  return hipGetLastError();
}

}  // namespace uaii_hip
