// prefill.hip — the prompt path (M > 1 tokens at once) on gfx950 matrix cores.
//
// The reference prefills one token at a time through quant_gemm_f32
// (libs/uaii-quant/src/quant_gemm.cpp:22-70: per weight row, dequantise to f32
// and dot with every activation row) and attention_kv_f32
// (libs/uaii-kernels/src/transformer.cpp:222-433). Here a chunk of M prompt
// tokens runs layer by layer as dense contractions:
//
//   k_pf_prep   RMSNorm (optional) of each activation row, a power-of-two row
//               scale 2^e, and the split x * 2^e = hi + lo into two f16 values
//               (together ~22 significant bits), plus per-32 sums for formats
//               whose blocks carry a minimum.
//   k_pf_mm     the products with the packed weights (prefill_gemm.hip).
//   k_pf_qkv    Q/K/V bias, RoPE and the KV-cache append for M positions.
//   k_pf_attn   causal attention of M queries over the f16 cache on MFMA:
//               S^T = K . Q^T, online softmax, O^T += V^T . P^T, with q * scale
//               and P split into f16 hi + lo against the exact f16 keys/values.
#include "prefill.h"

namespace uaii_hip {
namespace {

// ---- activation prep ----------------------------------------------------------------

// One block of NT threads per row; rows >= M (tile padding) are written as zeros.
// Memory bound with many rows (13.4 us for 512 x 14336, 58 MB); with few it is a
// chain of round trips, shorter with a row's loads spread over more threads.
template <int NT>
__global__ void __launch_bounds__(NT) k_pf_prep(float* __restrict__ x, int64_t ldx,
                                                 int64_t M, const float* __restrict__ norm_w,
                                                 float eps, PfAct act, const float* __restrict__ part,
                                                 int nsplit) {
  extern __shared__ float row[];
  __shared__ float red[NT / 64];
  const int64_t t = blockIdx.x;
  const int tid = threadIdx.x;
  const int64_t K = act.K;
  const int nv = (int)(K / 4);
  uint2* hi2 = reinterpret_cast<uint2*>(act.hi);
  uint2* lo2 = reinterpret_cast<uint2*>(act.lo);
  // float4 i of the row: quad i % 8 of 32-block i / 8, in the order 0, 4, 1, 5, ...
  auto at = [&](int i) -> int64_t { return ((int64_t)(i >> 3) * act.mpad + t) * 8 + 2 * (i & 3) + ((i >> 2) & 1); };
  float4* raw4 = reinterpret_cast<float4*>(act.raw);
  auto raw_at = [&](int i) -> int64_t {
    return (((int64_t)((i >> 2) & 1) * (K / 32) + (i >> 3)) * act.mpad + t) * 4 + (i & 3);
  };
  if (t >= M) {
    for (int i = tid; i < nv; i += NT) {
      if (act.hi) hi2[at(i)] = lo2[at(i)] = make_uint2(0, 0);
      if (act.raw) raw4[raw_at(i)] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
    if (act.sxp) {
      for (int i = tid; i < nv / 8; i += NT)
        reinterpret_cast<uint2*>(act.sxp)[((int64_t)(i >> 3) * act.mpad + t) * 8 + (i & 7)] = make_uint2(0, 0);
    }
    if (tid == 0) act.rs[t] = 0.0f;
    return;
  }
  float4* r4 = reinterpret_cast<float4*>(row);
  float4* x4 = reinterpret_cast<float4*>(x + t * ldx);
  float ss = 0.0f, amax = 0.0f;
  for (int i = tid; i < nv; i += NT) {
    float4 v = x4[i];
    if (nsplit > 0) {
      // residual add of a K-split GEMM's partials
      const f4_t p = split_sum<f4_t>(nsplit, [&](int z) {
        return reinterpret_cast<const f4_t*>(part + ((int64_t)z * M + t) * ldx)[i];
      });
      v.x += p.x; v.y += p.y; v.z += p.z; v.w += p.w;
      x4[i] = v;
    }
    r4[i] = v;
    ss += v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
    amax = fmaxf(amax, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
  }
  if (norm_w) {
    // x * (1/sqrt(mean(x^2)+eps)) * w with two roundings (norm.cpp:122-127)
    ss = wave_sum(ss);
    if ((tid & 63) == 0) red[tid >> 6] = ss;
    __syncthreads();
    float tot = red[0];
#pragma unroll
    for (int w = 1; w < NT / 64; ++w) tot += red[w];
    const float inv = 1.0f / sqrtf(tot / (float)K + eps);
    const float4* w4 = reinterpret_cast<const float4*>(norm_w);
    amax = 0.0f;
    for (int i = tid; i < nv; i += NT) {
      float4 v = r4[i];
      const float4 w = w4[i];
      v.x = fmul_rn(fmul_rn(v.x, inv), w.x);
      v.y = fmul_rn(fmul_rn(v.y, inv), w.y);
      v.z = fmul_rn(fmul_rn(v.z, inv), w.z);
      v.w = fmul_rn(fmul_rn(v.w, inv), w.w);
      r4[i] = v;
      amax = fmaxf(amax, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
    }
    __syncthreads();  // red[] is reused below
  }
  if (act.raw) {
    for (int i = tid; i < nv; i += NT) raw4[raw_at(i)] = r4[i];
    if (!act.hi) return;
  }
  amax = wave_max(amax);
  if ((tid & 63) == 0) red[tid >> 6] = amax;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < NT / 64; ++w) amax = fmaxf(amax, red[w]);
  // scale so that max |x| * 2^e lies in [2^14, 2^15): hi keeps 11 bits of every
  // element near the top of the row and lo the next 11. The limits are where 2^e and
  // 2^-e are normal numbers and the largest finite row still fits f16.
  int e = 0;
  if (amax > 0.0f) {
    const int ex = (int)((__float_as_uint(amax) >> 23) & 0xff) - 126;  // amax in [2^(ex-1), 2^ex)
    e = min(126, max(-113, 15 - ex));
  }
  const float s = pow2f_i(e);
  if (tid == 0) act.rs[t] = pow2f_i(-e);
  for (int base = 0; base < nv; base += NT) {
    const int i = base + tid;
    float sum = 0.0f;
    if (i < nv) {
      const float4 v = r4[i];
      const float y0 = v.x * s, y1 = v.y * s, y2 = v.z * s, y3 = v.w * s;
      const _Float16 h0 = (_Float16)y0, h1 = (_Float16)y1, h2 = (_Float16)y2, h3 = (_Float16)y3;
      // an infinity is all in hi
      auto rest = [](float y, _Float16 h) { return (_Float16)(fabsf(y) == INFINITY ? 0.0f : y - (float)h); };
      const _Float16 l0 = rest(y0, h0), l1 = rest(y1, h1), l2 = rest(y2, h2), l3 = rest(y3, h3);
      // stored order (k0, k2, k1, k3)
      hi2[at(i)] = make_uint2(__builtin_bit_cast(uint32_t, h2_t{h0, h2}),
                          __builtin_bit_cast(uint32_t, h2_t{h1, h3}));
      lo2[at(i)] = make_uint2(__builtin_bit_cast(uint32_t, h2_t{l0, l2}),
                          __builtin_bit_cast(uint32_t, h2_t{l1, l3}));
      sum = (y0 + y1) + (y2 + y3);
    }
    if (act.sxp) {
      // 8 consecutive float4 = one 32-block, 64 a super-block (K % 256 == 0)
      sum += __shfl_xor(sum, 1, 64);
      sum += __shfl_xor(sum, 2, 64);
      sum += __shfl_xor(sum, 4, 64);
      if (i < nv && (i & 7) == 0) {
        _Float16* d = reinterpret_cast<_Float16*>(act.sxp) + ((int64_t)(i >> 6) * act.mpad + t) * 32 + ((i >> 3) & 7);
        float v = sum * 0.03125f;
#pragma unroll
        for (int p = 0; p < 3; ++p) {
          d[8 * p] = (_Float16)v;
          v -= (float)d[8 * p];
        }
        d[24] = (_Float16)0.0f;
      }
    }
  }
}

// ---- QKV post-processing ------------------------------------------------------------------

// One block per token: bias, RoPE of q and k pairs (host-built angle table, as
// the decode epilogue), q -> qout, k and v -> cache at position p0 + t.
__global__ void __launch_bounds__(256) k_pf_qkv(PfQkvArgs a) {
  const int64_t t = blockIdx.x;
  const int pos = a.p0 + (int)t;
  const float* row = a.qkv + t * a.ldq;
  // value x of this row: the GEMM's output, or the sum of its K-split partials
  auto val = [&](int x) -> float {
    if (a.nsplit <= 1) return row[x];
    return split_sum<float>(a.nsplit, [&](int z) { return a.part[((int64_t)z * a.M + t) * a.ldq + x]; });
  };
  const int hd = a.head_dim, half = hd / 2;
  const int npair = (a.q_dim + a.kv_dim) / 2;
  for (int u = threadIdx.x; u < npair; u += blockDim.x) {
    const bool isq = u < a.q_dim / 2;
    const int uu = isq ? u : u - a.q_dim / 2;
    const int head = uu / half, p = uu % half;
    const int r0 = head * hd + (a.rope_mode == 2 ? p : 2 * p);
    const int r1 = r0 + (a.rope_mode == 2 ? half : 1);
    const int base = isq ? 0 : a.q_dim;
    float v0 = val(base + r0), v1 = val(base + r1);
    const float* bias = isq ? a.bq : a.bk;
    if (bias) { v0 = v0 + bias[r0]; v1 = v1 + bias[r1]; }
    const float2 cs = a.rope[(int64_t)pos * half + p];
    const float n0 = v0 * cs.x - v1 * cs.y;
    const float n1 = v0 * cs.y + v1 * cs.x;
    if (isq) {
      a.qout[t * a.q_dim + r0] = n0;
      a.qout[t * a.q_dim + r1] = n1;
    } else {
      const int64_t o0 = ((int64_t)(r0 / hd) * a.max_seq + pos) * hd + (r0 % hd);
      const int64_t o1 = ((int64_t)(r1 / hd) * a.max_seq + pos) * hd + (r1 % hd);
      if (a.kv_f16) {
        reinterpret_cast<__half*>(a.kcache)[o0] = __float2half(n0);
        reinterpret_cast<__half*>(a.kcache)[o1] = __float2half(n1);
      } else {
        reinterpret_cast<float*>(a.kcache)[o0] = n0;
        reinterpret_cast<float*>(a.kcache)[o1] = n1;
      }
    }
  }
  for (int r = threadIdx.x; r < a.kv_dim; r += blockDim.x) {
    float v = val(a.q_dim + a.kv_dim + r);
    if (a.bv) v = v + a.bv[r];
    const int64_t o = ((int64_t)(r / hd) * a.max_seq + pos) * hd + (r % hd);
    if (a.kv_f16) reinterpret_cast<__half*>(a.vcache)[o] = __float2half(v);
    else reinterpret_cast<float*>(a.vcache)[o] = v;
  }
}

// ---- causal attention over the f16 cache ---------------------------------------------------

constexpr int PA_TK = 64;  // keys per LDS tile
// 16-query subtiles per wave. 2 halves the K/V staging per matrix-core op but
// needs 430 registers at head_dim 128 (one wave per SIMD): measured 1.6x slower
// than 1 on the 8B prefill.
#ifndef UAII_PA_QW
#define UAII_PA_QW 1
#endif
constexpr int PA_QW = UAII_PA_QW;

// Four f16 of the transposed 4 x 16 piece that a group of 16 lanes names (8 bytes each).
__device__ inline h4_t lds_tr4(const _Float16* p) {
  typedef short s4_t __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) s4_t* lds4;
  return __builtin_bit_cast(h4_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)p));
}

// Query tile of the xi-th of nx tiles in launch order: the longest first, and every
// other band (the tiles of one block a CU) the other way round.
__device__ inline int pf_attn_tile(int xi, int nx, int band) {
  const int b = xi / band;
  if (b & 1) xi = b * band + min(band, nx - b * band) - 1 - (xi - b * band);
  return nx - 1 - xi;
}

// Block: 4 waves on kv head hb / (G / GW); wave w takes q head
// (w % GW) of the block's GW heads and query subtiles PA_QW (w / GW) ..
// PA_QW (w / GW) + PA_QW - 1 (16 queries each). K and V tiles of 64 keys are
// double-buffered in LDS as they lie in the cache; each thread loads the next tile's
// pieces into registers while the current tile is computed.
//
// What bounds it: the softmax between the two products of a wave's tile (two waves a
// SIMD cover each other), with the hi/lo products at twice the plain matrix-core work.
// V was stored transposed, 4 bytes a lane with rows 288 words apart: 8 lanes to a bank
// on every store, as much LDS time as all fragment reads together, and 16 vector
// operations a piece to pair the keys. Stored plain and read by ds_read_b64_tr_b16
// (two reads a fragment, as before), with the probabilities' hi and lo
// halves one fused operation each: 1024 queries at 1024, 32/8 heads of 128,
// 139 -> 80 us between calls from the host, 138 -> 66 back to back with the band order
// below (25.8 GFLOP: 187 -> 391 TFLOP/s); 512 queries at 4096 210 -> 125 us, where one
// block a CU leaves the softmax uncovered; 1000 from 0 at head_dim 64 36 -> 24 us.
// Blocks are numbered head first, so that an XCD's blocks share the K/V of few heads in
// its L2, with the longest query tiles first and alternate bands reversed, which gives
// the two blocks of a CU a long and a short tile: 79.8 -> 77.6 us, 2048 from 0
// 98.2 -> 94.9 us.
template <int HD>
__global__ void __launch_bounds__(256, 2) k_pf_attn(PfAttnArgs a) {
  constexpr int KP = HD + 8;        // K tile row (halfs)
  constexpr int NC = HD / 32;       // 32-wide hd chunks (S)
  constexpr int ND = HD / 16;       // 16-row hd subtiles (O)
  constexpr int PIECES = PA_TK * (HD / 8) / 256;  // 16-byte K (and V) pieces per thread
  __shared__ _Float16 ks[2][PA_TK * KP];
  __shared__ _Float16 vs[2][PA_TK * KP];

  const int G = a.n_heads / a.n_kv;
  const int GW = G < 4 ? G : 4;
  const int QS = 4 / GW;
  const int ny = a.n_kv * (G / GW);
  const int hb = (int)blockIdx.x % ny;
  const int kvh = hb / (G / GW);
  const int hbase = kvh * G + (hb % (G / GW)) * GW;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, col = lane & 15, g = lane >> 4;
  const bool active = wave < GW * QS;
  const int head = hbase + (wave % GW);
  const int64_t q0 = (int64_t)pf_attn_tile((int)blockIdx.x / ny, (int)gridDim.x / ny, a.band) * (16 * PA_QW * QS);
  const int64_t qw0 = q0 + 16 * PA_QW * (wave / GW);   // this wave's first query
  const int64_t qend = min((int64_t)a.M, q0 + 16 * PA_QW * QS);
  const int64_t nkeys = a.p0 + qend;  // keys the block needs (causal)

  // q * scale * 2^e as f16 hi + lo per query subtile u: lane (query col, group g)
  // holds hd 32c + 8g .. +7 of chunk c. Each query row is scaled to put its largest
  // element in [2^14, 2^15): below 2^-14 f16 loses significant bits
  const float scale = 1.0f / sqrtf((float)HD);
  h8_t qhi[PA_QW][NC], qlo[PA_QW][NC];
  float qrs[PA_QW];
  bool qvalid[PA_QW];
  int64_t qpos[PA_QW];
#pragma unroll
  for (int u = 0; u < PA_QW; ++u) {
    const int64_t qrow = qw0 + 16 * u + col;
    qvalid[u] = active && qrow < a.M;
    qpos[u] = a.p0 + qrow;
    float qv[NC][8];
    float qmax = 0.0f;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      if (qvalid[u]) {
        const float4* qp = reinterpret_cast<const float4*>(a.q + qrow * a.ldq + (int64_t)head * HD + 32 * c + 8 * g);
        const float4 x0 = qp[0], x1 = qp[1];
        qv[c][0] = x0.x; qv[c][1] = x0.y; qv[c][2] = x0.z; qv[c][3] = x0.w;
        qv[c][4] = x1.x; qv[c][5] = x1.y; qv[c][6] = x1.z; qv[c][7] = x1.w;
      } else {
#pragma unroll
        for (int k = 0; k < 8; ++k) qv[c][k] = 0.0f;
      }
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        qv[c][k] = qv[c][k] * scale;
        qmax = fmaxf(qmax, fabsf(qv[c][k]));
      }
    }
    qmax = fmaxf(qmax, __shfl_xor(qmax, 16, 64));
    qmax = fmaxf(qmax, __shfl_xor(qmax, 32, 64));
    int qe = 0;
    if (qmax > 0.0f) qe = min(100, max(-100, 15 - ((int)((__float_as_uint(qmax) >> 23) & 0xff) - 126)));
    const float qs = pow2f_i(qe);
    qrs[u] = pow2f_i(-qe);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const float v = qv[c][k] * qs;
        const _Float16 h = (_Float16)v;
        qhi[u][c][k] = h;
        qlo[u][c][k] = (_Float16)(v - (float)h);
      }
    }
  }

  // scale of the raw scores into base-2 exponent units, and the causal limits
  // in 32-bit positions (a cache holds < 2^31 keys)
  float l2s[PA_QW];
  int qposi[PA_QW];
#pragma unroll
  for (int u = 0; u < PA_QW; ++u) {
    l2s[u] = qrs[u] * 1.4426950408889634f;
    qposi[u] = (int)qpos[u];
  }
  const int64_t qpos0 = a.p0 + qw0;  // the wave's first query position
  f4_t o[PA_QW][ND];
  float mrun[PA_QW], lrun[PA_QW];
#pragma unroll
  for (int u = 0; u < PA_QW; ++u) {
    mrun[u] = -INFINITY;
    lrun[u] = 0.0f;
#pragma unroll
    for (int d = 0; d < ND; ++d) o[u][d] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
  }

  const __half* kbase = reinterpret_cast<const __half*>(a.kcache) + (int64_t)kvh * a.max_seq * HD;
  const __half* vbase = reinterpret_cast<const __half*>(a.vcache) + (int64_t)kvh * a.max_seq * HD;

  // tile staging: pieces of 8 dims of a key, K and V alike; keys past nkeys read as
  // zeros. Offsets inside a tile are 32-bit and fixed per thread; only the last tile
  // checks them against nkeys.
  uint4 kreg[PIECES], vreg[PIECES];
  auto load_tile = [&](int64_t kt) __attribute__((always_inline)) {
    const __half* kt_base = reinterpret_cast<const __half*>(uniform_ptr(kbase + kt * HD));
    const __half* vt_base = reinterpret_cast<const __half*>(uniform_ptr(vbase + kt * HD));
    const bool full = kt + PA_TK <= nkeys;  // block-uniform
#pragma unroll
    for (int u = 0; u < PIECES; ++u) {
      const int c = threadIdx.x + 256 * u;
      const int key = c / (HD / 8), p = c % (HD / 8);
      kreg[u] = make_uint4(0, 0, 0, 0);
      vreg[u] = make_uint4(0, 0, 0, 0);
      if (full || kt + key < nkeys) {
        kreg[u] = *reinterpret_cast<const uint4*>(kt_base + (key * HD + 8 * p));
        vreg[u] = *reinterpret_cast<const uint4*>(vt_base + (key * HD + 8 * p));
      }
    }
  };
  auto store_tile = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < PIECES; ++u) {
      const int c = threadIdx.x + 256 * u;
      const int key = c / (HD / 8), p = c % (HD / 8);
      *reinterpret_cast<uint4*>(&ks[buf][key * KP + 8 * p]) = kreg[u];
      *reinterpret_cast<uint4*>(&vs[buf][key * KP + 8 * p]) = vreg[u];
    }
  };
  auto lds_barrier = []() __attribute__((always_inline)) {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  auto compute = [&](int64_t kt, int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < PA_QW; ++u) {
      // S^T for 4 key subtiles: lane holds keys kt + 16s + 4g + r of query col
      // raw scores (q pre-scaled by 2^qe); the running max and the exponentials
      // are in base 2: score * log2(e) = acc * l2s, p = 2^(acc * l2s - m)
      f4_t sc[4];
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4) {
        f4_t acc = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          const h8_t kf = *reinterpret_cast<const h8_t*>(&ks[buf][(16 * s4 + col) * KP + 32 * c + 8 * g]);
          acc = mfma32(kf, qhi[u][c], acc);
          acc = mfma32(kf, qlo[u][c], acc);
        }
        sc[s4] = acc;
      }
      // causal mask only on tiles that reach past the wave's first query
      // (rows past M are never stored and need none)
      if (kt + PA_TK - 1 > qpos0) {
#pragma unroll
        for (int s4 = 0; s4 < 4; ++s4)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int key = (int)kt + 16 * s4 + 4 * g + r;
            if (key > qposi[u]) sc[s4][r] = -INFINITY;
          }
      }
      float tmax = -INFINITY;
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4)
#pragma unroll
        for (int r = 0; r < 4; ++r) tmax = fmaxf(tmax, sc[s4][r]);
      tmax = fmaxf(tmax, __shfl_xor(tmax, 16, 64));
      tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
      const float mnew = fmaxf(mrun[u], tmax * l2s[u]);
      const float alpha = (mrun[u] == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f(mrun[u] - mnew);
      const float mref = (mnew == -INFINITY) ? 0.0f : mnew;  // a fully masked row so far: p = 0
      float psum = 0.0f;
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float p = __builtin_amdgcn_exp2f(fmaf(sc[s4][r], l2s[u], -mref));
          sc[s4][r] = p;
          psum += p;
        }
      psum += __shfl_xor(psum, 16, 64);
      psum += __shfl_xor(psum, 32, 64);
      lrun[u] = lrun[u] * alpha + psum;
      mrun[u] = mnew;
      if (__any(alpha != 1.0f)) {
#pragma unroll
        for (int d = 0; d < ND; ++d) o[u][d] *= alpha;
      }
      // O^T += V^T . (2^14 P)^T over two 32-key chunks (p <= 1, so 2^14 p keeps
      // hi and lo normal); lane's keys: 32c + 4g + r (r < 4), 32c + 16 + 4g + (r - 4)
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        h8_t phi, plo;
#pragma unroll
        for (int r = 0; r < 8; ++r) {
          const float p = sc[2 * c + (r >> 2)][r & 3];
          const _Float16 h = (_Float16)(p * 16384.0f);
          phi[r] = h;
          plo[r] = (_Float16)fmaf(p, 16384.0f, -(float)h);  // exact before the rounding
        }
        // V^T by transposed LDS reads: the 16 lanes of group g name 4 keys x 16 dims,
        // lane i gets dim i of the 4 keys
        h8_t vf[ND];
#pragma unroll
        for (int d = 0; d < ND; ++d) {
          const _Float16* vr = &vs[buf][(32 * c + 4 * g + (col >> 2)) * KP + 16 * d + 4 * (col & 3)];
          const h4_t v0 = lds_tr4(vr), v1 = lds_tr4(vr + 16 * KP);
          vf[d] = h8_t{v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
        }
#pragma unroll
        for (int d = 0; d < ND; ++d) o[u][d] = mfma32(vf[d], phi, o[u][d]);
#pragma unroll
        for (int d = 0; d < ND; ++d) o[u][d] = mfma32(vf[d], plo, o[u][d]);
      }
    }
  };

  load_tile(0);
  store_tile(0);
  lds_barrier();
  int buf = 0;
  for (int64_t kt = 0; kt < nkeys; kt += PA_TK) {
    const bool more = kt + PA_TK < nkeys;  // block-uniform
    if (more) load_tile(kt + PA_TK);
    if (active) compute(kt, buf);
    if (more) store_tile(buf ^ 1);
    lds_barrier();
    buf ^= 1;
  }

#pragma unroll
  for (int u = 0; u < PA_QW; ++u) {
    if (!qvalid[u]) continue;
    const int64_t qrow = qw0 + 16 * u + col;
    const float inv = (1.0f / 16384.0f) / lrun[u];
    float* out = a.out + qrow * a.ldo + (int64_t)head * HD;
#pragma unroll
    for (int d = 0; d < ND; ++d) {
      const float4 v = make_float4(o[u][d][0] * inv, o[u][d][1] * inv, o[u][d][2] * inv, o[u][d][3] * inv);
      *reinterpret_cast<float4*>(out + 16 * d + 4 * g) = v;
    }
  }
}

// ---- MoE over prompt rows ----------------------------------------------------------------

// Routing of token t on one wave from its E router logits (LDS): softmax
// (exp(l - max) * 1/sum), k rounds of the largest remaining probability (ties:
// the lower expert), weights renormalised over the chosen k
// (transformer.cpp:446-481, :565-580).
__device__ inline void moe_topk(const float* logit, int E, int k, int32_t* __restrict__ ids,
                                float* __restrict__ wout, int64_t t, int lane) {
  float p[4];
  float mx = -INFINITY;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int e = lane + 64 * j;
    p[j] = e < E ? logit[e] : -INFINITY;
    mx = fmaxf(mx, p[j]);
  }
  mx = wave_max(mx);
  float sum = 0.0f;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int e = lane + 64 * j;
    p[j] = e < E ? expf(p[j] - mx) : 0.0f;
    sum += p[j];
  }
  sum = wave_sum(sum);
  const float isum = sum > 0.0f ? 1.0f / sum : 0.0f;
#pragma unroll
  for (int j = 0; j < 4; ++j) p[j] = (lane + 64 * j < E) ? p[j] * isum : -1.0f;
  float mass = 0.0f;
  float wsel[8];
  int32_t esel[8];
  for (int q = 0; q < k; ++q) {
    float bv = -1.0f;
    int be = 0x7fffffff;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (p[j] > bv) { bv = p[j]; be = lane + 64 * j; }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const float ov = __shfl_xor(bv, o, 64);
      const int oe = __shfl_xor(be, o, 64);
      if (ov > bv || (ov == bv && oe < be)) { bv = ov; be = oe; }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (lane + 64 * j == be) p[j] = -1.0f;  // taken
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (j == q) { wsel[j] = bv; esel[j] = (be >= 0 && be < E) ? be : 0; }
    mass += bv;
  }
  if (!(mass > 0.0f)) mass = 1.0f;
  if (lane == 0) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (j < k) {
        ids[t * k + j] = esel[j];
        wout[t * k + j] = wsel[j] / mass;
      }
    }
  }
}

// One block per token: RMSNorm of x[t] (the k_pf_prep arithmetic), router
// logits against F32 / F16 rows, then the routing of k_moe_route on wave 0:
// softmax (exp(l - max) * 1/sum), k rounds of the largest remaining probability
// (ties: the lower expert), weights renormalised over the chosen k
// (transformer.cpp:446-481, :565-580).
template <int RT>
__global__ void __launch_bounds__(256) k_pf_moe_route(const float* __restrict__ x, int64_t K,
                                                      const float* __restrict__ norm_w, float eps,
                                                      DevWeight router, int E, int k,
                                                      int32_t* __restrict__ ids, float* __restrict__ wout) {
  extern __shared__ float row[];
  __shared__ float red[4];
  __shared__ float logit[256];
  const int64_t t = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int nv = (int)(K / 4);
  float4* r4 = reinterpret_cast<float4*>(row);
  const float4* x4 = reinterpret_cast<const float4*>(x + t * K);
  float ss = 0.0f;
  for (int i = tid; i < nv; i += 256) {
    const float4 v = x4[i];
    r4[i] = v;
    ss += v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
  }
  ss = wave_sum(ss);
  if (lane == 0) red[wave] = ss;
  __syncthreads();
  const float tot = red[0] + red[1] + red[2] + red[3];
  const float inv = 1.0f / sqrtf(tot / (float)K + eps);
  const float4* w4 = reinterpret_cast<const float4*>(norm_w);
  for (int i = tid; i < nv; i += 256) {
    float4 v = r4[i];
    const float4 w = w4[i];
    v.x = fmul_rn(fmul_rn(v.x, inv), w.x);
    v.y = fmul_rn(fmul_rn(v.y, inv), w.y);
    v.z = fmul_rn(fmul_rn(v.z, inv), w.z);
    v.w = fmul_rn(fmul_rn(v.w, inv), w.w);
    r4[i] = v;
  }
  __syncthreads();
  // logits: wave w takes experts w, w + 4, ...; each lane 4 consecutive inputs
  // per step, the router loads of 8 steps issued before their arithmetic (one
  // memory round trip per 8 steps, not per step)
  constexpr int RB = 8;
  for (int e = wave; e < E; e += 4) {
    float acc = 0.0f;
    const uint8_t* wr = router.a + (int64_t)e * router.a_row;
    for (int base = 0; base < nv; base += 64 * RB) {
      float4 wv[RB];
#pragma unroll
      for (int j = 0; j < RB; ++j) {
        const int i = min(base + 64 * j + lane, nv - 1);
        if constexpr (RT == T_F32) {
          wv[j] = reinterpret_cast<const float4*>(wr)[i];
        } else {
          const uint2 h = reinterpret_cast<const uint2*>(wr)[i];
          wv[j] = make_float4(h2f((uint16_t)(h.x & 0xffff)), h2f((uint16_t)(h.x >> 16)),
                              h2f((uint16_t)(h.y & 0xffff)), h2f((uint16_t)(h.y >> 16)));
        }
      }
#pragma unroll
      for (int j = 0; j < RB; ++j) {
        const int i = base + 64 * j + lane;
        if (i < nv) {
          const float4 xv = r4[i];
          acc += xv.x * wv[j].x + xv.y * wv[j].y + xv.z * wv[j].z + xv.w * wv[j].w;
        }
      }
    }
    acc = wave_sum(acc);
    if (lane == 0) logit[e] = acc;
  }
  __syncthreads();
  if (wave == 0) moe_topk(logit, E, k, ids, wout, t, lane);
}

// The same routing for one token (the decode step) on a 16-wave block: the
// router row of expert e is cut into P parts of up to 512 float4 (8 per lane),
// wave w takes the parts w, w + 16, ..., and its first part's router loads are
// issued before the RMSNorm, so the weight fetch overlaps the input's. The
// parts' sums are added in part order. dynamic LDS: K normalised inputs, then
// the E * P part sums.
template <int RT>
__global__ void __launch_bounds__(1024) k_moe_route_dec(const float* __restrict__ x, int64_t K,
                                                        const float* __restrict__ norm_w, float eps,
                                                        DevWeight router, int E, int k,
                                                        int32_t* __restrict__ ids, float* __restrict__ wout) {
  extern __shared__ float row[];
  __shared__ float red[16];
  __shared__ float logit[256];
  constexpr int RB = 8;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int nv = (int)(K / 4);
  const int P = (nv + 64 * RB - 1) / (64 * RB);
  const int items = E * P;
  float* psum = row + K;
  using Raw = typename std::conditional<RT == T_F32, float4, uint2>::type;
  auto load_item = [&](int it, Raw (&wv)[RB]) __attribute__((always_inline)) {
    const int e = it / P, part = it % P;
    const Raw* wr = reinterpret_cast<const Raw*>(router.a + (int64_t)e * router.a_row);
#pragma unroll
    for (int j = 0; j < RB; ++j) wv[j] = wr[min(part * 64 * RB + 64 * j + lane, nv - 1)];
  };
  auto dot_item = [&](int it, const Raw (&wv)[RB]) __attribute__((always_inline)) {
    const int part = it % P;
    const float4* r4 = reinterpret_cast<const float4*>(row);
    float acc = 0.0f;
#pragma unroll
    for (int j = 0; j < RB; ++j) {
      const int i = part * 64 * RB + 64 * j + lane;
      if (i < nv) {
        float4 w;
        if constexpr (RT == T_F32) {
          w = wv[j];
        } else {
          w = make_float4(h2f((uint16_t)(wv[j].x & 0xffff)), h2f((uint16_t)(wv[j].x >> 16)),
                          h2f((uint16_t)(wv[j].y & 0xffff)), h2f((uint16_t)(wv[j].y >> 16)));
        }
        const float4 xv = r4[i];
        acc += xv.x * w.x + xv.y * w.y + xv.z * w.z + xv.w * w.w;
      }
    }
    acc = wave_sum(acc);
    if (lane == 0) psum[it] = acc;
  };
  Raw w0[RB];
  if (wave < items) load_item(wave, w0);
  // RMSNorm (the k_pf_prep arithmetic) into LDS
  float4* r4 = reinterpret_cast<float4*>(row);
  const float4* x4 = reinterpret_cast<const float4*>(x);
  float ss = 0.0f;
  for (int i = tid; i < nv; i += 1024) {
    const float4 v = x4[i];
    r4[i] = v;
    ss += v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
  }
  ss = wave_sum(ss);
  if (lane == 0) red[wave] = ss;
  __syncthreads();
  float tot = 0.0f;
#pragma unroll
  for (int w = 0; w < 16; ++w) tot += red[w];
  const float inv = 1.0f / sqrtf(tot / (float)K + eps);
  const float4* n4 = reinterpret_cast<const float4*>(norm_w);
  for (int i = tid; i < nv; i += 1024) {
    float4 v = r4[i];
    const float4 w = n4[i];
    v.x = fmul_rn(fmul_rn(v.x, inv), w.x);
    v.y = fmul_rn(fmul_rn(v.y, inv), w.y);
    v.z = fmul_rn(fmul_rn(v.z, inv), w.z);
    v.w = fmul_rn(fmul_rn(v.w, inv), w.w);
    r4[i] = v;
  }
  __syncthreads();
  if (wave < items) dot_item(wave, w0);
  for (int it = wave + 16; it < items; it += 16) {
    Raw wv[RB];
    load_item(it, wv);
    dot_item(it, wv);
  }
  __syncthreads();
  if (wave != 0) return;
  for (int e = lane; e < E; e += 64) {
    float l = 0.0f;
    for (int q = 0; q < P; ++q) l += psum[e * P + q];
    logit[e] = l;
  }
  moe_topk(logit, E, k, ids, wout, 0, lane);
}

// One block lists each expert's (token, slot) entries in entry order (entry
// i = token * k + slot): counts[e], offsets[e] (exclusive prefix), list[pos] =
// token and inv[i] = pos. Wave w owns the entry range [w n / 4, (w + 1) n / 4):
// range counts by LDS atomics, then each wave walks its range 64 entries at a
// time, a lane's position within its expert being the number of same-expert
// lanes below it (ballot + popcount) past the range's running base.
__global__ void __launch_bounds__(256) k_pf_moe_lists(const int32_t* __restrict__ ids, int64_t M, int k,
                                                      int E, int32_t* counts, int32_t* offsets,
                                                      int32_t* list, int32_t* inv) {
  __shared__ int32_t cnt[4][256], base[4][256];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t n = M * k;
  const int64_t per = (n + 3) / 4;
  const int64_t r0 = min(n, (int64_t)wave * per), r1 = min(n, r0 + per);
  for (int j = tid; j < 4 * 256; j += 256) cnt[j >> 8][j & 255] = 0;
  __syncthreads();
  for (int64_t i = r0 + lane; i < r1; i += 64) atomicAdd(&cnt[wave][ids[i]], 1);
  __syncthreads();
  if (tid == 0) {
    int32_t acc = 0;
    for (int e = 0; e < E; ++e) {
      counts[e] = cnt[0][e] + cnt[1][e] + cnt[2][e] + cnt[3][e];
      offsets[e] = acc;
      for (int r = 0; r < 4; ++r) {
        base[r][e] = acc;
        acc += cnt[r][e];
      }
    }
  }
  __syncthreads();
  for (int64_t g = r0; g < r1; g += 64) {
    const int64_t i = g + lane;
    const bool act = i < r1;
    const int x = act ? ids[i] : -1;
    uint64_t pending = __ballot(act);
    while (pending) {
      const int e0 = __shfl(x, __ffsll((long long)pending) - 1, 64);  // wave-uniform
      const uint64_t m = __ballot(x == e0) & pending;
      const int32_t b = base[wave][e0];
      if (x == e0) {
        const int32_t pos = b + __popcll(m & ((1ull << lane) - 1ull));
        list[pos] = (int32_t)(i / k);
        inv[i] = pos;
      }
      if (lane == 0) base[wave][e0] = b + __popcll(m);
      pending &= ~m;
    }
  }
}

// One block per token: x[t] += w y in slot order (each slot one expert).
__global__ void __launch_bounds__(256) k_pf_moe_combine(float* __restrict__ x, int64_t D, int k,
                                                        const float* __restrict__ w,
                                                        const int32_t* __restrict__ inv,
                                                        const float* __restrict__ y) {
  const int64_t t = blockIdx.x;
  float* xr = x + t * D;
  for (int64_t i = threadIdx.x; i < D; i += 256) {
    float v = xr[i];
    for (int q = 0; q < k; ++q) v = v + w[t * k + q] * y[(int64_t)inv[t * k + q] * D + i];
    xr[i] = v;
  }
}

}  // namespace

// ---- launchers ------------------------------------------------------------------------------

bool pf_row_supported(int64_t K) { return K * 4 <= lds_limit() - 2048; }

hipError_t launch_pf_prep(float* x, int64_t ldx, int64_t M, const float* norm_w, float eps,
                          const PfAct& act, hipStream_t s, const float* part, int nsplit) {
  if (nsplit < 0 || (nsplit > 0 && !part)) return hipErrorInvalidValue;
  if (M <= 0 || M > act.mpad || act.K % 32 || act.mpad != pf_mpad(act.mpad) || ldx % 4 || (act.sxp && act.K % 256))
    return hipErrorInvalidValue;
  const size_t lds = (size_t)act.K * 4;
  if ((int64_t)lds > lds_limit()) return hipErrorInvalidValue;
  auto go = [&](auto kernel, int threads) -> hipError_t {
    if (lds > 64 * 1024) {
      const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      if (e != hipSuccess) return e;
    }
    UAII_LAUNCH(kernel, dim3((unsigned)act.mpad), dim3(threads), lds, s, x, ldx, M, norm_w, eps, act, part, nsplit);
    return hipGetLastError();
  };
  // Up to a block per two CUs the row's own latency is the launch's: whole products of 9
  // to 100 rows take 3-4 % less with 1024 threads (six formats, K of 1408 to 14336), of
  // 300 and 500 rows 0.5 %, at K = 512 up to 3 % more.
  return act.mpad <= 128 && act.K >= 1024 ? go(&k_pf_prep<1024>, 1024) : go(&k_pf_prep<256>, 256);
}

hipError_t launch_pf_qkv(const PfQkvArgs& a, hipStream_t s) {
  if (a.M <= 0 || a.head_dim <= 0 || a.head_dim % 2 || a.q_dim % a.head_dim ||
      a.kv_dim % a.head_dim || a.p0 < 0 || a.p0 + a.M > a.max_seq)
    return hipErrorInvalidValue;
  UAII_LAUNCH(k_pf_qkv, dim3((unsigned)a.M), dim3(256), 0, s, a);
  return hipGetLastError();
}

bool pf_attn_supported(int head_dim, int n_heads, int n_kv) {
  if (head_dim != 64 && head_dim != 128) return false;
  if (n_kv <= 0 || n_heads % n_kv) return false;
  const int G = n_heads / n_kv;
  const int GW = G < 4 ? G : 4;
  return G % GW == 0;
}

hipError_t launch_pf_attn(const PfAttnArgs& a, hipStream_t s) {
  if (a.M <= 0 || a.p0 < 0 || a.p0 + a.M > a.max_seq || !pf_attn_supported(a.hd, a.n_heads, a.n_kv) ||
      a.ldq % 4 || a.ldo % 4)
    return hipErrorInvalidValue;
  const int G = a.n_heads / a.n_kv;
  const int GW = G < 4 ? G : 4;
  const int QS = 4 / GW;
  const int QT = 16 * PA_QW * QS;  // queries per block
  const int ny = a.n_kv * (G / GW);
  const int64_t blocks = (int64_t)((a.M + QT - 1) / QT) * ny;
  if (blocks > INT32_MAX) return hipErrorInvalidValue;
  PfAttnArgs b = a;
  b.band = std::max(1, device_cus() / ny);  // query tiles that give every CU one block
  const dim3 grid((unsigned)blocks);
  if (a.hd == 64) UAII_LAUNCH(k_pf_attn<64>, grid, dim3(256), 0, s, b);
  else UAII_LAUNCH(k_pf_attn<128>, grid, dim3(256), 0, s, b);
  return hipGetLastError();
}

bool pf_router_supported(int type) { return type == T_F32 || type == T_F16; }

hipError_t launch_pf_moe_route(const float* x, int64_t M, int64_t K, const float* norm_w, float eps,
                               const DevWeight& router, int E, int k, int32_t* ids, float* w,
                               hipStream_t s) {
  if (M <= 0 || K % 4 || !norm_w || E < 1 || E > 256 || k < 1 || k > 8 || k > E ||
      router.rows < E || router.cols != K || !pf_router_supported(router.type))
    return hipErrorInvalidValue;
  if (M == 1) {
    // the decode step: the 16-wave kernel
    const int64_t P = (K / 4 + 511) / 512;
    const size_t lds1 = (size_t)(K + E * P) * 4;
    if ((int64_t)lds1 > lds_limit()) return hipErrorInvalidValue;
    const void* fn = router.type == T_F32 ? reinterpret_cast<const void*>(&k_moe_route_dec<T_F32>)
                                          : reinterpret_cast<const void*>(&k_moe_route_dec<T_F16>);
    if (lds1 > 64 * 1024) {
      const hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds1);
      if (e != hipSuccess) return e;
    }
    if (router.type == T_F32)
      UAII_LAUNCH(k_moe_route_dec<T_F32>, dim3(1), dim3(1024), lds1, s, x, K, norm_w, eps, router, E, k, ids, w);
    else
      UAII_LAUNCH(k_moe_route_dec<T_F16>, dim3(1), dim3(1024), lds1, s, x, K, norm_w, eps, router, E, k, ids, w);
    return hipGetLastError();
  }
  const size_t lds = (size_t)K * 4;
  if ((int64_t)lds > lds_limit()) return hipErrorInvalidValue;
  if (router.type == T_F32) {
    if (lds > 64 * 1024) {
      const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_pf_moe_route<T_F32>),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      if (e != hipSuccess) return e;
    }
    UAII_LAUNCH(k_pf_moe_route<T_F32>, dim3((unsigned)M), dim3(256), lds, s, x, K, norm_w, eps, router, E,
                k, ids, w);
  } else {
    if (lds > 64 * 1024) {
      const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_pf_moe_route<T_F16>),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      if (e != hipSuccess) return e;
    }
    UAII_LAUNCH(k_pf_moe_route<T_F16>, dim3((unsigned)M), dim3(256), lds, s, x, K, norm_w, eps, router, E,
                k, ids, w);
  }
  return hipGetLastError();
}

hipError_t launch_pf_moe_lists(const int32_t* ids, int64_t M, int k, int E, int32_t* counts,
                               int32_t* offsets, int32_t* list, int32_t* inv, hipStream_t s) {
  if (M <= 0 || k < 1 || k > 8 || E < 1 || E > 256) return hipErrorInvalidValue;
  UAII_LAUNCH(k_pf_moe_lists, dim3(1), dim3(256), 0, s, ids, M, k, E, counts, offsets, list, inv);
  return hipGetLastError();
}

hipError_t launch_pf_moe_combine(float* x, int64_t M, int64_t D, int k, const float* w,
                                 const int32_t* inv, const float* y, hipStream_t s) {
  if (M <= 0 || D <= 0 || k < 1 || k > 8) return hipErrorInvalidValue;
  UAII_LAUNCH(k_pf_moe_combine, dim3((unsigned)M), dim3(256), 0, s, x, D, k, w, inv, y);
  return hipGetLastError();
}

}  // namespace uaii_hip
