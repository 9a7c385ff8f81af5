// prefill_gemm.hip — C[M][N] = A . W^T for prompt rows (M > 1) on gfx950 matrix
// cores (quant_gemm_f32, libs/uaii-quant/src/quant_gemm.cpp:22-70: per weight row,
// dequantise to f32 and dot with every activation row).
//
// For the quantised formats the activations come from k_pf_prep as f16 pairs hi + lo
// (about 22 significant bits), the weights as small integers that f16 holds exactly,
// decoded in registers from their split GGUF layout; v_mfma_f32_16x16x32_f16 multiplies
// the integers with hi and with lo and sums in f32.
//
// F16 weights take the f32 rows and v_mfma_f32_16x16x4_f32 (157 TFLOP/s dense, a
// sixteenth of the f16 rate). As f16 pairs their products, whose exponents spread, lost
// more to the f16 op's sums than one GEMV per row does (1.05e-7 of the result against
// 0.83e-7 at K = 512; 1.5e-6 against 0.85e-7 with subnormal weights), and infinities met
// zeros. Now eight products make a sum, four sums are added in pairs, and the running sum
// carries what it lost to rounding beside it: 0.72e-7 at every K up to 14336 and
// 0.77e-7 .. 0.99e-7 with K splits, where the GEMV has 0.83e-7 .. 1.07e-7. 1024 rows of
// 4096 x 4096 104 -> 359 us, 9 rows 16.4 -> 19.5 (one row at a time 7.0 ms and 64 us); the
// matrix ops and the sums' vector work beside them bound it (95 TFLOP/s; 112 with one
// sum a block and plain additions, whose error was 1.0e-7).
//
// What bounds it. With many rows, vector and LDS work beside the matrix ops: a probe
// of f16 matrix ops (two waves per SIMD, nothing loaded from memory) sustained 1.9
// PFLOP/s bare, 1.40 with three vector ops per matrix op, 1.18 with those and an A
// read (16 bytes a lane) for every four matrix ops, 1.05 with one for every two. A
// 16-row subtile of A is read once per 32 k as hi and once as lo and serves the NT
// column subtiles of the wave, so NT = 4 halves the reads of the 64 x 32 wave tile
// used before; the integers' hi and lo products count twice, so 1.1 PFLOP/s of matrix
// ops are 0.55 of the product's. Measured on 1024 rows, 28672 x 4096 (TFLOP/s, before
// and now): Q4_0 453, 481; Q8_0 386, 430; Q4_K 266, 455; Q6_K 186, 347; on Q5_K 400,
// which ran one row at a time. With few rows the launch is a chain of
// round trips to memory; a K split and smaller blocks shorten it: 9 rows, 4096 x 4096,
// with the preparation and the fold (us): Q4_0 47, 17; Q8_0 52, 19; Q4_K 88, 17;
// Q6_K 120, 20.
//
// Block: 4 waves side by side along N, 16 MT rows x 64 NT columns. K runs in
// stages of 64 (two 32-blocks) through two LDS buffers in turn, four in blocks of up to
// 32 rows (see buffers): everything a stage needs travels global -> LDS
// (global_load_lds_dwordx4) while the stages before it are computed, the block's A rows
// and each wave's own weight rows, so no registers hold data in transit (held there,
// they spilled beside the accumulators). Lane group
// g = lane / 16 takes word g (4 bytes) of each 16-byte chunk of its row; with
// 32-value blocks of two such halves that makes its eight k of a block the quads
// 4 g .. and 16 + 4 g .., the order in which k_pf_prep stores A (see PfAct), for
// every block format.
//
// Scales. Q4_0 and Q8_0 blocks each have an f16 scale of their own, applied to the
// block's f32 product. In Q4_K and Q5_K the 6-bit sub-block scale folds into the
// integer: sc q <= 63 * 31 < 2048 is exact in f16 (one packed FMA from the (64 + q)
// form that the decode gives anyway), so the super-block's 256 k
// accumulate in the matrix core and only d is applied to the sum. Their minimums
// are one more matrix op per super-block: the eight sub-block sums of A, each as
// three f16 parts (all of its 24 bits), times the eight 6-bit minimums, then dmin.
// Q6_K folds its int8 sub-block scale too: sc (q - 32) is an integer of up to 12
// bits, held as an f16 pair (the remainder is 0 or +-1).
#include <type_traits>

#include "prefill.h"

namespace uaii_hip {
namespace {

constexpr int GW = 4;  // waves side by side along N

// Q8_0 with the K sums' rounding error carried along (PfGemmArgs::carry): the prompt rows
// of sessions that ran them one token a step. Plain, the sums of 256 k were added one
// after another, 16 to 56 of them, and the error grew past the step kernel's 1.09e-7 ..
// 1.18e-7 of the result (1000 rows: 1.19e-7 at 14336 x 4096, 1.38e-7 at 4096 x 14336).
// The carry takes the registers of half the columns, so its waves are 32 wide.
// Carried: 0.93e-7 .. 1.10e-7 at every size, below the step kernel's there; 1000 rows
// 303 -> 324 us at 14336 x 4096, 317 -> 334 at 4096 x 14336, 100 -> 103 at 4096 x 4096.
constexpr int Q8_0_CARRY = 256 + T_Q8_0;
template <int FMT>
__device__ constexpr bool is_q8() { return FMT == T_Q8_0 || FMT == Q8_0_CARRY; }

// Ties what computes v (or is computed from it) to this place: instruction selection
// orders a block's pure arithmetic as it likes, and left to itself decodes several
// subtiles ahead or leaves sums waiting, until registers spill (Q4_K, MT = 4: 168).
__device__ inline void pin(uint32_t& v) { asm volatile("" : "+v"(v)); }
__device__ inline void pin(f4_t& v) { asm volatile("" : "+v"(v)); }
__device__ inline void pin(uint4& q) { pin(q.x); pin(q.y); pin(q.z); pin(q.w); }

__device__ inline h2_t pk_fma(h2_t a, h2_t b, h2_t c) { return __builtin_elementwise_fma(a, b, c); }
__device__ inline h2_t h2_of(float v) { return h2_t{(_Float16)v, (_Float16)v}; }

// ---- weight bytes -------------------------------------------------------------------

// Formats whose scale is applied per 256 k (and whose rows are whole super-blocks).
template <int FMT>
__device__ constexpr bool is_k() { return FMT == T_Q4_K || FMT == T_Q5_K || FMT == T_Q6_K; }
// Formats with a minimum per sub-block.
template <int FMT>
__device__ constexpr bool has_min() { return FMT == T_Q4_K || FMT == T_Q5_K; }

// Q6_K's d is read as it is needed; its pointers name their address space (they would
// be flat otherwise, whose loads also hold up the LDS counter).
typedef const __attribute__((address_space(1))) uint8_t* gptr;
template <class T>
__device__ inline T ldg(gptr p, uint32_t o) {
  return *(const __attribute__((address_space(1))) T*)(p + o);
}

// Bytes of a weight row in LDS. Per stage: the payload (PB bytes; Q6_K's stages take
// the runs s and s + 2 of a 128-value half, whose low bits are the two nibbles of the
// same 32 bytes) and a dword of scales (Q4_0, Q8_0). Per two stages: Q6_K's high bits
// of the half. Per four: a super-block's scales (16 bytes, and Q5_K's high bits).
template <int FMT>
constexpr int payload() { return FMT == T_F16 ? 128 : is_q8<FMT>() ? 64 : 32; }
template <int FMT>
constexpr bool has_dword() { return FMT == T_Q4_0 || is_q8<FMT>(); }

// A super-block's scales of the lane's column, decoded from its 16 bytes.
template <int FMT> struct Unit {};
template <> struct Unit<T_Q4_K> { uint32_t sc[2]; float d; };
template <> struct Unit<T_Q5_K> { uint32_t sc[2]; float d; uint32_t h[2]; };
template <> struct Unit<T_Q6_K> { uint32_t sc[4]; float d; };

// The words of one block of the lane's row (F16: two quads; Q6_K: with the high bits).
template <int FMT>
constexpr int words() { return FMT == T_F16 || FMT == T_Q6_K ? 4 : FMT == T_Q4_0 ? 1 : 2; }
template <int FMT> struct Words { uint32_t w[words<FMT>()]; uint32_t d; };

template <int FMT>
__device__ inline void pin_unit(Unit<FMT>& u) {
  if constexpr (has_min<FMT>()) { pin(u.sc[0]); pin(u.sc[1]); }
  if constexpr (FMT == T_Q5_K) { pin(u.h[0]); pin(u.h[1]); }
  if constexpr (FMT == T_Q6_K) { pin(u.sc[0]); pin(u.sc[1]); pin(u.sc[2]); pin(u.sc[3]); }
}

// Slot of 16-byte part p of row r (PARTS parts): the permutations that measured free
// of bank conflicts for 32- and 64-byte rows; 128-byte rows take the 64-byte one.
template <int PARTS>
__device__ inline int wslot(int r, int p) { return PARTS == 2 ? p ^ ((r >> 3) & 1) : p ^ ((r >> 2) & 3); }

// What the unsigned values of Q4_K and Q5_K are centred on: their sums then stay
// small, and the rounding of the accumulators with them (K = 14336: 4.7e-7 of the
// result without, see k_pf_mm).
template <int FMT>
constexpr int center() { return FMT == T_Q4_K ? 8 : 16; }

// B operand of block t (0, 1) of stage h (0..3) of its 256 k: the block's integers
// (Q6_K: with their remainder in blo).
template <int FMT>
__device__ inline void decode_block(const Words<FMT>& r, const Unit<FMT>& u, int h, int t, h8_t& b, h8_t& blo) {
  const uint32_t kLo = 0x000F000Fu, kHi = 0x00F000F0u;
  if constexpr (FMT == T_Q4_0) {
    const uint32_t w = r.w[0], w8 = w >> 8;
    const h2_t c = h2_of(-1032.0f), s = h2_of(0.0625f), e = h2_of(-72.0f);
    b = cat8(as_h2(and_or(w, kLo, 0x64006400u)) + c, as_h2(and_or(w8, kLo, 0x64006400u)) + c,
             pk_fma(as_h2(and_or(w, kHi, 0x64006400u)), s, e), pk_fma(as_h2(and_or(w8, kHi, 0x64006400u)), s, e));
  } else if constexpr (is_q8<FMT>()) {
    const uint32_t v0 = r.w[0] ^ 0x80808080u, v1 = r.w[1] ^ 0x80808080u;
    const h2_t c = h2_of(-1152.0f);
    b = cat8(as_h2(byte_pair(v0)) + c, as_h2(byte_pair(v0 >> 8)) + c, as_h2(byte_pair(v1)) + c,
             as_h2(byte_pair(v1 >> 8)) + c);
  } else if constexpr (FMT == T_F16) {
    // the f32 values of quad g (b) and quad 4 + g (blo)
    auto quad = [&](uint32_t u, uint32_t v) __attribute__((always_inline)) {
      const h2_t p = as_h2(u), q = as_h2(v);
      return __builtin_bit_cast(h8_t, f4_t{(float)p.x, (float)p.y, (float)q.x, (float)q.y});
    };
    b = quad(r.w[0], r.w[1]);
    blo = quad(r.w[2], r.w[3]);
  } else if constexpr (FMT == T_Q4_K || FMT == T_Q5_K) {
    const int j = 2 * h + t;  // sub-block: the stage's low (t = 0) or high nibbles
    const uint32_t w0 = r.w[0], w1 = r.w[1];
    // The value's bits at bits 4.. of an f16 with 64's exponent read 64 + q; one
    // packed FMA gives sc (64 + q) - sc (64 + c) = sc (q - c), every term exact.
    const uint32_t k64 = 0x54005400u;
    const uint32_t sel = 0x04000400u + 0x00010001u * (uint32_t)(j & 3);
    const h2_t sc = as_h2(__builtin_amdgcn_perm(0x64646464u, u.sc[j >> 2], sel)) + h2_of(-1024.0f);
    const h2_t off = sc * h2_of(-64.0f - (float)center<FMT>());
    uint32_t v[4];
    if constexpr (FMT == T_Q4_K) {
      const uint32_t e0 = t ? w0 : w0 << 4, o0 = t ? w0 >> 8 : w0 >> 4;
      const uint32_t e1 = t ? w1 : w1 << 4, o1 = t ? w1 >> 8 : w1 >> 4;
      v[0] = and_or(e0, kHi, k64); v[1] = and_or(o0, kHi, k64);
      v[2] = and_or(e1, kHi, k64); v[3] = and_or(o1, kHi, k64);
    } else {
      const int sh = 4 - j;  // sub-block j's bit of each qh byte to bit 4
      const uint32_t h0 = sh >= 0 ? u.h[0] << sh : u.h[0] >> -sh, h1 = sh >= 0 ? u.h[1] << sh : u.h[1] >> -sh;
      const uint32_t v0 = ((w0 >> (4 * t)) & 0x0F0F0F0Fu) | (h0 & 0x10101010u);
      const uint32_t v1 = ((w1 >> (4 * t)) & 0x0F0F0F0Fu) | (h1 & 0x10101010u);
      v[0] = and_or(v0 << 4, 0x01F001F0u, k64); v[1] = and_or(v0 >> 4, 0x01F001F0u, k64);
      v[2] = and_or(v1 << 4, 0x01F001F0u, k64); v[3] = and_or(v1 >> 4, 0x01F001F0u, k64);
    }
    b = cat8(pk_fma(as_h2(v[0]), sc, off), pk_fma(as_h2(v[1]), sc, off), pk_fma(as_h2(v[2]), sc, off),
             pk_fma(as_h2(v[3]), sc, off));
  } else if constexpr (FMT == T_Q6_K) {
    // run q = h % 2 + 2 t of half h / 2: low (t = 0) or high nibbles, qh bits 2 q; its
    // two 16-element sub-blocks have int8 scales 8 (h / 2) + 2 q and + 1
    const int q = (h & 1) + 2 * t;
    h2_t hi[4], lo[4];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const uint32_t hq = q < 2 ? r.w[2 + e] << (4 - 2 * q) : r.w[2 + e] >> (2 * q - 4);
      const uint32_t q6 = ((r.w[e] >> (4 * t)) & 0x0F0F0F0Fu) | (hq & 0x30303030u);
      const int si = 8 * (h >> 1) + 2 * q + e;
      const _Float16 s = (_Float16)(float)(int8_t)((u.sc[si >> 2] >> (8 * (si & 3))) & 0xff);
      const h2_t sc = {s, s}, c = h2_of(-1056.0f);
      const h2_t p0 = as_h2(byte_pair(q6)) + c, p1 = as_h2(byte_pair(q6 >> 8)) + c;
      hi[2 * e] = p0 * sc;
      lo[2 * e] = pk_fma(p0, sc, -hi[2 * e]);
      hi[2 * e + 1] = p1 * sc;
      lo[2 * e + 1] = pk_fma(p1, sc, -hi[2 * e + 1]);
    }
    b = cat8(hi[0], hi[1], hi[2], hi[3]);
    blo = cat8(lo[0], lo[1], lo[2], lo[3]);
  }
}
// f16 scale of block t (Q4_0, Q8_0)
template <int FMT>
__device__ inline float block_scale(const Words<FMT>& r, int t) {
  if constexpr (has_dword<FMT>()) return h2f((uint16_t)(r.d >> (16 * t)));
  else return 1.0f;
}

// ---- the kernel ---------------------------------------------------------------------

// Column subtiles per wave. F16's 128 bytes per row and stage leave LDS for two
// blocks per CU only with two (it has no decode to pay for, so its LDS reads may).
template <int FMT>
constexpr int nt_of() { return FMT == T_F16 || FMT == Q8_0_CARRY ? 2 : 4; }

// LDS: A stages [NB][block 2][hi/lo 2][BM rows][64 B], then per wave the payload
// stages [NB][rows][payload], and for the formats that have them the dwords
// [NB][rows][4], the super-blocks' 16 bytes [2][rows][16], the high bits
// [NH][rows][32], and for the block the sub-block sums [2][BM][64].
// Buffers of a stage: a stage is requested NB - 1 stages ahead. Two are enough where
// a stage's matrix ops last longer than a round trip to memory; blocks of up to 32
// rows are bound by that trip and take four.
template <int MT>
constexpr int buffers() { return MT <= 2 ? 4 : 2; }
template <int FMT, int MT>
struct Lds {
  static constexpr int BM = 16 * MT, NR = 16 * nt_of<FMT>();
  static constexpr int A = 4 * BM * 64;
  static constexpr int W = NR * payload<FMT>();
  static constexpr int D = has_dword<FMT>() ? 256 : 0;
  static constexpr int S = is_k<FMT>() ? NR * 16 : 0;
  static constexpr int H = FMT == T_Q5_K || FMT == T_Q6_K ? NR * 32 : 0;
  static constexpr int X = has_min<FMT>() ? BM * 64 : 0;
  // the high bits' buffers: by unit (Q5_K), by half and, requested further ahead, unit
  static constexpr int NB = buffers<MT>(), NH = FMT == T_Q6_K && NB > 2 ? 4 : 2;
  static constexpr int wave = NB * (W + D) + 2 * S + NH * H;
  static constexpr int oW = NB * A, oD = NB * W, oS = oD + NB * D, oH = oS + 2 * S;
  static constexpr int oX = oW + GW * wave, total = oX + 2 * X;
};

// Output rows [m0, mend) of this grid row and the first weight row of its expert
// (0 without grouping).
struct Range { int64_t m0, mend, mfirst, wrow0; };

template <int N, class F>
__device__ inline __attribute__((always_inline)) void for_n(F&& f) {
  if constexpr (N > 0) {
    for_n<N - 1>(f);
    f(std::integral_constant<int, N - 1>{});
  }
}
// KH = 2: a block holds two such groups of waves, each on its own half of the block's
// K range with its own LDS buffers; the second group hands its sums over through LDS.
// That fills a CU where the grid gives it one block only, without the partials in
// memory that a split of K over blocks costs (500 x 6144 x 4096, two groups, one, and one
// with the K split doubled: Q8_0 87.5, 95.4, 90.4 us; Q4_0 76.3, 85.6, 82.9).
template <int FMT, int EPI, int MT, int KH>
__global__ void __launch_bounds__(GW * 64 * KH, 2 / KH) k_pf_mm(PfGemmArgs a) {
  constexpr int NT = nt_of<FMT>();
  constexpr bool F32 = FMT == T_F16;          // f32 operands
  constexpr bool CARRY = F32 || FMT == Q8_0_CARRY;
  constexpr bool BLOCK_SCALE = !is_k<FMT>() && !F32;  // f32 sums per 32-block
  constexpr bool TWO = FMT != T_Q4_0 && !F32;  // sums per 256 k, then over K
  using L = Lds<FMT, MT>;
  constexpr int BM = 16 * MT;
  constexpr int NQ = (EPI == EPI_SWIGLU) ? NT / 2 : NT;  // distinct row subtiles
  constexpr int NR = 16 * NT;
  constexpr bool MIN = has_min<FMT>();
  extern __shared__ __attribute__((aligned(16))) uint8_t lds_all[];

  // Grid position. Blocks go to the XCDs round-robin in dispatch order; with the
  // column-tile count a multiple of 8, XCD x takes the column tiles 8 c + x, row
  // tile fastest, so that the blocks resident on one XCD share weights in its L2.
  int tile = blockIdx.x, gy = blockIdx.y;
  if ((gridDim.x & 7) == 0) {
    const int id = blockIdx.y * gridDim.x + blockIdx.x;
    const int loc = id >> 3;
    gy = loc % gridDim.y;
    tile = (loc / gridDim.y) * 8 + (id & 7);
  }
  int si = 0;
  for (int k = 1; k < a.nseg; ++k) if (tile >= a.seg[k].tile0) si = k;
  const PfSeg& seg = a.seg[si];
  const int wave = __builtin_amdgcn_readfirstlane((threadIdx.x >> 6) & (GW - 1));
  const int kg = KH == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);  // the wave's group
  uint8_t* lds = lds_all + kg * L::total;
  const int lane = threadIdx.x & 63, col = lane & 15, g = lane >> 4;
  const int64_t n0 = ((int64_t)(tile - seg.tile0) * GW + wave) * (16 * NQ);
  Range mr;
  if (a.gtab) {
    const int32_t* e = a.gtab + 3 * gy;
    mr = Range{e[1], e[2], e[1], (int64_t)e[0] * seg.rows};
  } else {
    mr = Range{(int64_t)gy * BM, a.M, 0, 0};
  }
  // Activation row of output row t. Rows past the range read its first row (the
  // map's first entry without grouping) and their results are dropped; unmapped,
  // ungrouped rows below mpad are read as they are.
  auto arow = [&](int64_t t) __attribute__((always_inline)) -> int64_t {
    if (!a.arow && !a.gtab) return t;
    const int64_t tc = t < mr.mend ? t : mr.mfirst;
    return a.arow ? (int64_t)a.arow[tc] : tc;
  };
  // this block's stages: units of 256 k (four stages), split evenly along grid z
  const int nst = (int)(a.K / 64), nun = (nst + 3) / 4;
  const uint32_t parts = (uint32_t)a.ksplit * KH, part0 = blockIdx.z * KH;  // nun < 2^23, parts <= 128
  const auto first = [&](uint32_t q) { return 4 * (int)((uint32_t)nun * q / parts); };
  const int sbeg = first(part0 + kg), send = min(nst, first(part0 + kg + 1));
  // every group of the block goes through as many stages (and barriers) as the longest
  int count = (send - sbeg + 3) / 4 * 4;
  if constexpr (KH == 2) {
    const int o = kg ^ 1;
    count = max(count, (min(nst, first(part0 + o + 1)) - first(part0 + o) + 3) / 4 * 4);
  }

  // A copies: wave w takes hi or lo (w & 1) of the stage's block w / 2, one
  // instruction per 16 rows, lane -> (row, slot); piece p of row r sits in slot
  // p ^ ((r >> 1) & 3), which keeps the fragment reads free of bank conflicts.
  uint32_t aoff[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int r = 16 * i + (lane >> 2);
    aoff[i] = (uint32_t)(arow(mr.m0 + r) * 64) + 16 * ((lane & 3) ^ ((r >> 1) & 3));
  }
  const uint8_t* abase = uniform_ptr((wave & 1) ? a.alo : a.ahi);
  const int64_t bstride = a.act_ld * 64;  // bytes of one 32-block of all rows
  const uint8_t* xbase = uniform_ptr(a.sxp);

  // Weight rows: subtile j's 16 rows start at n0 + 16 j, moved back where the
  // segment ends sooner; the columns it then shares with the subtile before it are
  // not stored twice. Row r of the wave's NR rows: subtile r / 16.
  int64_t nb[NQ];
#pragma unroll
  for (int j = 0; j < NQ; ++j) nb[j] = max((int64_t)0, min(n0 + 16 * j, seg.rows - 16));
  auto wrow = [&](int r, const DevWeight** w) __attribute__((always_inline)) -> int64_t {
    const int j = r >> 4;
    *w = (EPI == EPI_SWIGLU && j >= NQ) ? &seg.w2 : &seg.w;
    const int64_t first = max((int64_t)0, min(n0 + 16 * (j % NQ), seg.rows - 16));
    return mr.wrow0 + min(first + (r & 15), seg.rows - 1);
  };
  constexpr int WP = payload<FMT>() / 16, NW = NR * WP / 64, RW = 64 / WP;  // parts, copies, rows per copy
  const uint8_t* wsrc[NW];
#pragma unroll
  for (int u = 0; u < NW; ++u) {
    const DevWeight* w;
    const int r = RW * u + lane / WP;
    const int64_t row = wrow(r, &w);
    wsrc[u] = w->a + row * w->a_row + 16 * wslot<WP>(r, lane % WP);
  }
  const uint8_t *dsrc = nullptr, *ssrc = nullptr, *hsrc[2] = {nullptr, nullptr};
  gptr d6[NT];
  if constexpr (has_dword<FMT>() || is_k<FMT>()) {
    const DevWeight* w;
    const int64_t row = wrow(lane & (NR - 1), &w);
    if constexpr (has_dword<FMT>()) dsrc = w->b + row * w->b_row;
    if constexpr (MIN) ssrc = w->b + row * w->b_row;
    if constexpr (FMT == T_Q6_K) ssrc = w->c + row * w->c_row;
  }
  if constexpr (L::H > 0) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const DevWeight* w;
      const int r = 32 * u + (lane >> 1);
      const int64_t row = wrow(r, &w);
      hsrc[u] = (FMT == T_Q5_K ? w->c + row * w->c_row : w->b + row * w->b_row) + 16 * wslot<2>(r, lane & 1);
    }
  }
  if constexpr (FMT == T_Q6_K) {
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const DevWeight* w;
      const int64_t row = wrow(16 * j + col, &w);
      d6[j] = (gptr)(uintptr_t)(w->d + row * w->d_row);
    }
  }

  // requests that every wave makes for a stage h (some make more: the sums), and the
  // s_waitcnt operand for at most n outstanding (lgkmcnt 0)
  constexpr auto requests = [](int h) {
    h &= 3;
    return MT + NW + (has_dword<FMT>() ? 1 : 0) + (is_k<FMT>() && h == 0 ? 1 : 0) +
           ((FMT == T_Q5_K && h == 0) || (FMT == T_Q6_K && (h & 1) == 0) ? 2 : 0);
  };
  constexpr auto vm_wait = [](int n) { return 0x0070 | (n & 15) | ((n >> 4) << 14); };
  static_assert(requests(0) + requests(2) < 64, "vmcnt");
  const uint32_t lbase = lds_addr(lds);
  const uint32_t wbase = lbase + L::oW + wave * L::wave;
  // stage st, h = st % 4, into buffer h % NB (unit data: the unit's parity)
  auto issue = [&](auto h_c, int st) __attribute__((always_inline)) {
    constexpr int h = decltype(h_c)::value, buf = h % L::NB;
    const int ub = (st >> 2) & 1;
    {
      // Q6_K: stage h takes the runs h % 2 and h % 2 + 2 of its half
      const int blk = FMT == T_Q6_K ? 4 * (st >> 1) + (h & 1) + 2 * (wave >> 1) : 2 * st + (wave >> 1);
      const uint8_t* src = uniform_ptr(abase + blk * bstride);
#pragma unroll
      for (int i = 0; i < MT; ++i) dma16s(src, aoff[i], lbase + buf * L::A + (wave * BM + 16 * i) * 64);
    }
#pragma unroll
    for (int u = 0; u < NW; ++u) dma16(wsrc[u] + (int64_t)st * payload<FMT>(), wbase + buf * L::W + 1024 * u);
    if constexpr (has_dword<FMT>()) dma4(dsrc + (int64_t)st * 4, wbase + L::oD + buf * L::D);
    if constexpr (is_k<FMT>() && h == 0) {
      dma16(ssrc + (int64_t)(st >> 2) * 16, wbase + L::oS + ub * L::S);
      if constexpr (MIN) {
        const uint8_t* src = uniform_ptr(xbase + (st >> 2) * bstride);
#pragma unroll
        for (int i = 0; i < MT; ++i)
          if ((i & 3) == wave) dma16s(src, aoff[i], lbase + L::oX + ub * L::X + 16 * i * 64);
      }
    }
    if constexpr ((FMT == T_Q5_K && h == 0) || (FMT == T_Q6_K && (h & 1) == 0)) {
      const int hb = FMT == T_Q5_K ? ub : (h >> 1) + (L::NH == 4 ? 2 * ub : 0);
#pragma unroll
      for (int u = 0; u < 2; ++u)
        dma16(hsrc[u] + (int64_t)(FMT == T_Q5_K ? st >> 2 : st >> 1) * 32, wbase + L::oH + hb * L::H + 1024 * u);
    }
  };

  const f4_t zero = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
  f4_t acc[MT][NT], part[MT][NT];
  f4_t lost[CARRY ? MT : 1][NT];  // what acc lost to rounding
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      acc[i][j] = part[i][j] = zero;
      if constexpr (CARRY) lost[i][j] = zero;
    }

  Unit<FMT> unit[NT];

  // fragment of 16-row subtile i, block t, hi (0) or lo (1) in buffer `buf`
  const int fragoff = col * 64 + 16 * (g ^ ((col >> 1) & 3));
  auto frag = [&](int buf, int t, int hl, int i) __attribute__((always_inline)) -> h8_t {
    return *reinterpret_cast<const h8_t*>(lds + fragoff + (buf * L::A + ((t * 2 + hl) * BM + 16 * i) * 64));
  };
  // the lane's words: parts of row 16 j + col sit in the same slots for every j
  const uint8_t* wl = lds + L::oW + wave * L::wave;
  uint32_t poff[4];
#pragma unroll
  for (int p = 0; p < 4; ++p)
    poff[p] = col * payload<FMT>() + 16 * (p < WP ? wslot<WP>(col, p) : 0) + (FMT == T_F16 ? 8 * (g & 1) : 4 * g);
  // F16: quad g and quad 4 + g of a 64-byte block, quads 2 p and 2 p + 1 in part p
  uint32_t foff[2];
#pragma unroll
  for (int e = 0; e < 2; ++e) foff[e] = col * 128 + 16 * wslot<4>(col, (g >> 1) + 2 * e) + 8 * (g & 1);
  uint32_t hoff[2];
#pragma unroll
  for (int p = 0; p < 2; ++p) hoff[p] = col * 32 + 16 * wslot<2>(col, p) + 4 * g;
  auto lw = [&](uint32_t o) __attribute__((always_inline)) { return *reinterpret_cast<const uint32_t*>(wl + o); };
  auto read_words = [&](auto h_c, int ub, int t, int j, Words<FMT>& r) __attribute__((always_inline)) {
    constexpr int h = decltype(h_c)::value, buf = h % L::NB;
    const uint32_t o = buf * L::W + 16 * j * payload<FMT>();
    if constexpr (FMT == T_Q4_0) {
      r.w[0] = lw(o + poff[t]);
    } else if constexpr (is_q8<FMT>()) {
      r.w[0] = lw(o + poff[2 * t]);
      r.w[1] = lw(o + poff[2 * t + 1]);
    } else if constexpr (FMT == T_F16) {
      // quads g (part g / 2 of the block's four) and 4 + g
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const uint2 v = *reinterpret_cast<const uint2*>(wl + o + 64 * t + foff[e]);
        r.w[2 * e] = v.x;
        r.w[2 * e + 1] = v.y;
      }
    } else {
      r.w[0] = lw(o + poff[0]);
      r.w[1] = lw(o + poff[1]);
    }
    if constexpr (FMT == T_Q6_K) {
      const uint32_t ho = L::oH + ((h >> 1) + (L::NH == 4 ? 2 * ub : 0)) * L::H + 16 * j * 32;
      r.w[2] = lw(ho + hoff[0]);
      r.w[3] = lw(ho + hoff[1]);
    }
    if constexpr (has_dword<FMT>()) r.d = lw(L::oD + buf * L::D + 4 * (16 * j + col));
  };
  float d6n[NT];  // Q6_K: the next unit's d
  auto load_d6 = [&](int st) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < NT; ++j) d6n[j] = h2f(ldg<uint16_t>(d6[j], (uint32_t)(st >> 2) * 2));
  };

  // A block runs column subtile by column subtile: the A fragments of all MT row
  // subtiles stay in registers, subtile j + 1's weights decode beside the matrix ops
  // of subtile j (their words were read one subtile earlier still), and the last
  // subtile's ops are followed by the next block's fragment reads. The scheduling
  // fence between subtiles bounds what is live at MT = 4; with fewer rows registers are
  // plenty and the subtiles may overlap.
  h8_t fa[MT][2], bc, bcl;
  float sc;
  auto stage = [&](auto h_c, int st) __attribute__((always_inline)) {
    constexpr int h = decltype(h_c)::value, buf = h % L::NB;
    const int ub = (st >> 2) & 1;
    // Stage st complete in LDS (at most the requests of the stages after it that were
    // made outstanding), and every wave past its reads of the buffer taken next.
    if constexpr (L::NB == 2) {
      __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0)
    } else {
      constexpr int n1 = requests(h + 1), n2 = n1 + requests(h + 2);
      if (st + 2 < send) __builtin_amdgcn_s_waitcnt(vm_wait(n2));
      else if (st + 1 < send) __builtin_amdgcn_s_waitcnt(vm_wait(n1));
      else __builtin_amdgcn_s_waitcnt(0x0070);
    }
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (st >= send) return;  // the other group is longer
    Words<FMT> wd[2];
    read_words(h_c, ub, 0, 0, wd[0]);
    read_words(h_c, ub, 0, 1, wd[1]);
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      fa[i][0] = frag(buf, 0, 0, i);
      fa[i][1] = frag(buf, 0, 1, i);
    }
    constexpr int ahead = L::NB - 1;
    if (st + ahead < send) issue(std::integral_constant<int, (h + ahead) & 3>{}, st + ahead);
    if constexpr (h == 0 && is_k<FMT>()) {
      h8_t xs[MT];
      if constexpr (MIN) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
          xs[i] = *reinterpret_cast<const h8_t*>(lds + L::oX + ub * L::X + 16 * i * 64 + fragoff);
      }
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const uint4 m = *reinterpret_cast<const uint4*>(wl + L::oS + ub * L::S + 16 * (16 * j + col));
        if constexpr (FMT == T_Q6_K) {
          unit[j].sc[0] = m.x; unit[j].sc[1] = m.y; unit[j].sc[2] = m.z; unit[j].sc[3] = m.w;
          unit[j].d = d6n[j];
        }
        if constexpr (MIN) {
          // 6-bit (scale, min) pairs of the 12-byte field (gguf_dequant.cpp:107-115),
          // four to a word
          unit[j].sc[0] = m.y & 0x3F3F3F3Fu;
          unit[j].sc[1] = (m.w & 0x0F0F0F0Fu) | ((m.y >> 2) & 0x30303030u);
          unit[j].d = h2f((uint16_t)(m.x & 0xffff));
          if constexpr (FMT == T_Q5_K) {
            unit[j].h[0] = lw(L::oH + ub * L::H + 16 * j * 32 + hoff[0]);
            unit[j].h[1] = lw(L::oH + ub * L::H + 16 * j * 32 + hoff[1]);
          }
          // acc += d c (sums . sc) - dmin (sums . mn): what the centring takes off
          // the values, and the minimums. 32 x the 6-bit numbers (the sums are
          // stored times 1/32).
          auto six = [&](uint32_t w0, uint32_t w1) __attribute__((always_inline)) {
            const h2_t c = h2_of(-32768.0f), s = h2_of(32.0f);
            auto pr = [&](uint32_t w, uint32_t sel) __attribute__((always_inline)) {
              return pk_fma(as_h2(__builtin_amdgcn_perm(0x64646464u, w, sel)), s, c);
            };
            return cat8(pr(w0, 0x04010400u), pr(w0, 0x04030402u), pr(w1, 0x04010400u), pr(w1, 0x04030402u));
          };
          const h8_t s6 = six(unit[j].sc[0], unit[j].sc[1]);
          const h8_t m6 = six(m.z & 0x3F3F3F3Fu, ((m.w >> 4) & 0x0F0F0F0Fu) | ((m.z >> 2) & 0x30303030u));
          const float dc = unit[j].d * (float)center<FMT>(), dmin = h2f((uint16_t)(m.x >> 16));
#pragma unroll
          for (int i = 0; i < MT; ++i) {
            const f4_t ps = mfma32(xs[i], s6, zero), pm = mfma32(xs[i], m6, zero);
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][j][r] += fmaf(dc, ps[r], -(dmin * pm[r]));
            pin(acc[i][j]);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
    if constexpr (h == 3 && FMT == T_Q6_K) load_d6(min(st + 1, send - 1));
    f4_t p[2][MT];
    float psc = 0.0f;
    auto decode = [&](int t, int j, Words<FMT>& w, h8_t& b, h8_t& bl, float& s) __attribute__((always_inline)) {
#pragma unroll
      for (int e = 0; e < words<FMT>(); ++e) pin(w.w[e]);
      if constexpr (is_k<FMT>()) pin_unit<FMT>(unit[j]);
      decode_block<FMT>(w, unit[j], h, t, b, bl);
      s = block_scale<FMT>(w, t);
    };
    auto phase = [&](auto q_c) __attribute__((always_inline)) {
      constexpr int q = decltype(q_c)::value, t = q / NT, j = q % NT;  // block, subtile
      constexpr bool last = j + 1 == NT, more = t < 1;
      h8_t bn, bnl;
      float sn = 0.0f;
      if constexpr (q + 1 < 2 * NT) decode((q + 1) / NT, (q + 1) % NT, wd[(q + 1) & 1], bn, bnl, sn);
      if constexpr (q + 2 < 2 * NT) read_words(h_c, ub, (q + 2) / NT, (q + 2) % NT, wd[q & 1]);
      // Of the block's last subtile the fragments are free once their products are
      // issued; the fences keep the next block's reads from moving ahead of that,
      // where they would need registers of their own.
      auto next_frags = [&](int hl) __attribute__((always_inline)) {
        if constexpr (last && more) {
          if constexpr (MT == 4) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int i = 0; i < MT; ++i) fa[i][hl] = frag(buf, t + 1, hl, i);
        }
      };
      if constexpr (BLOCK_SCALE) {
        constexpr int cur = q & 1;
#pragma unroll
        for (int i = 0; i < MT; ++i) p[cur][i] = mfma32(fa[i][0], bc, zero);
        next_frags(0);
#pragma unroll
        for (int i = 0; i < MT; ++i) p[cur][i] = mfma32(fa[i][1], bc, p[cur][i]);
        next_frags(1);
        // the scale of the subtile before, while this one's products run
        if constexpr (q > 0) {
          constexpr int pj = (j + NT - 1) % NT, pt = j > 0 ? t : t - 1;
#pragma unroll
          for (int i = 0; i < MT; ++i) {
            if constexpr (!TWO) acc[i][pj] += psc * p[cur ^ 1][i];
            else if constexpr (h == 0 && pt == 0) part[i][pj] = psc * p[cur ^ 1][i];
            else part[i][pj] += psc * p[cur ^ 1][i];
            if constexpr (TWO) pin(part[i][pj]);
            else pin(acc[i][pj]);
          }
        }
        psc = sc;
      } else if constexpr (F32) {
        // four sums of 8 values (two matrix ops each), added in pairs
        const f4_t bq[2] = {__builtin_bit_cast(f4_t, bc), __builtin_bit_cast(f4_t, bcl)};
        f4_t s8[4][MT];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
#pragma unroll
          for (int i = 0; i < MT; ++i)
            s8[e >> 1][i] = mfma4(__builtin_bit_cast(f4_t, fa[i][e >> 2])[e & 3], bq[e >> 2][e & 3],
                                  (e & 1) == 0 ? zero : s8[e >> 1][i]);
          if (e == 3) next_frags(0);
        }
        next_frags(1);
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          const f4_t add = (s8[0][i] + s8[1][i]) + (s8[2][i] + s8[3][i]), to = acc[i][j] + add;
          lost[i][j] += add - (to - acc[i][j]);
          acc[i][j] = to;
          pin(acc[i][j]);
          pin(lost[i][j]);
        }
      } else {
        constexpr bool first = h == 0 && t == 0;  // of the unit
#pragma unroll
        for (int i = 0; i < MT; ++i) part[i][j] = mfma32(fa[i][1], bc, first ? zero : part[i][j]);
        next_frags(1);
        if constexpr (FMT == T_Q6_K) {
#pragma unroll
          for (int i = 0; i < MT; ++i) part[i][j] = mfma32(fa[i][0], bcl, part[i][j]);  // (lo, remainder): 2^-21
        }
#pragma unroll
        for (int i = 0; i < MT; ++i) part[i][j] = mfma32(fa[i][0], bc, part[i][j]);
        next_frags(0);
      }
      bc = bn;
      bcl = bnl;
      sc = sn;
      if constexpr (MT == 4) __builtin_amdgcn_sched_barrier(0);
    };
    decode(0, 0, wd[0], bc, bcl, sc);
    for_n<2 * NT>(phase);
    if constexpr (BLOCK_SCALE) {
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        if constexpr (TWO) part[i][NT - 1] += psc * p[1][i];
        else acc[i][NT - 1] += psc * p[1][i];
      }
    }
  };

  if (KH == 1 || sbeg < send) issue(std::integral_constant<int, 0>{}, sbeg);
  if constexpr (L::NB > 2) {
    if (sbeg + 1 < send) issue(std::integral_constant<int, 1>{}, sbeg + 1);
    if (sbeg + 2 < send) issue(std::integral_constant<int, 2>{}, sbeg + 2);
  }
  if constexpr (FMT == T_Q6_K) load_d6(min(sbeg, nst - 1));
  for (int st = sbeg; st < sbeg + count; st += 4) {
    stage(std::integral_constant<int, 0>{}, st);
    stage(std::integral_constant<int, 1>{}, st + 1);
    stage(std::integral_constant<int, 2>{}, st + 2);
    stage(std::integral_constant<int, 3>{}, st + 3);
    // the unit's sums into the accumulators
    if (TWO && st < send) {
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          if constexpr (is_k<FMT>()) {
            acc[i][j] += unit[j].d * part[i][j];
          } else if constexpr (CARRY) {
            const f4_t to = acc[i][j] + part[i][j];
            lost[i][j] += part[i][j] - (to - acc[i][j]);
            acc[i][j] = to;
            pin(lost[i][j]);
          } else {
            acc[i][j] += part[i][j];
          }
          pin(acc[i][j]);
        }
    }
  }

  if constexpr (CARRY) {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r)  // an infinite sum has nothing beside it
          if (isfinite(acc[i][j][r])) acc[i][j][r] += lost[i][j][r];
  }

  if constexpr (KH == 2) {
    __builtin_amdgcn_s_waitcnt(0x0070);
    __syncthreads();
    f4_t* x = reinterpret_cast<f4_t*>(lds_all);
    if (kg == 1) {
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) x[((i * NT + j) * GW + wave) * 64 + lane] = acc[i][j];
    }
    __syncthreads();
    if (kg == 1) return;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) acc[i][j] += x[((i * NT + j) * GW + wave) * 64 + lane];
  }

  // epilogue: lane holds rows m0 + 16 i + 4 g + r of column nb[j] + col
  const bool split = a.ksplit > 1;
#pragma unroll
  for (int i = 0; i < MT; ++i) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int64_t t = mr.m0 + 16 * i + 4 * g + r;
      if (t >= mr.mend) continue;
      const float rs = F32 ? 1.0f : a.rs[arow(t)];
      float* yrow = a.y + t * a.ldy + seg.col0;
      float* prw = split ? a.part + ((int64_t)blockIdx.z * a.M + t) * a.ldp + seg.col0 : nullptr;
#pragma unroll
      for (int j = 0; j < NQ; ++j) {
        const int64_t n = nb[j] + col;
        if (n < n0 + 16 * j || n >= seg.rows) continue;
        const float v = acc[i][j][r] * rs;
        if (split) {
          prw[n] = v;
          if constexpr (EPI == EPI_SWIGLU) prw[seg.rows + n] = acc[i][j + NQ][r] * rs;
          continue;
        }
        if constexpr (EPI == EPI_STORE) {
          yrow[n] = v;
        } else if constexpr (EPI == EPI_ADD) {
          yrow[n] = yrow[n] + v;
        } else if constexpr (EPI == EPI_SWIGLU) {
          yrow[n] = pf_silu(v) * (acc[i][j + NQ][r] * rs);
        } else if constexpr (EPI == EPI_GELU) {
          yrow[n] = pf_gelu(v);
        }
      }
    }
  }
}

// The partials of a K-split launch, added up (split_sum), and the epilogue:
// y [M][ldy] from part [ksplit][M][ldp]; SwiGLU's gate and up sums side by side.
// Block: 256 V-wide pieces of row blockIdx.y.
template <int EPI, int V>
__global__ void __launch_bounds__(256) k_pf_fold(const float* __restrict__ part, int ksplit, int64_t M, int64_t N,
                                                 int64_t ldp, float* __restrict__ y, int64_t ldy) {
  typedef float vec __attribute__((ext_vector_type(V)));
  const int64_t n = ((int64_t)blockIdx.x * 256 + threadIdx.x) * V, t = blockIdx.y;
  if (n >= N) return;
  const float* p = part + t * ldp + n;
  const int64_t zs = M * ldp;
  const auto at = [&](int64_t o) { return *reinterpret_cast<const vec*>(p + o); };
  vec v = split_sum<vec>(ksplit, [&](int z) { return at(z * zs); }), u;
  if constexpr (EPI == EPI_SWIGLU) u = split_sum<vec>(ksplit, [&](int z) { return at(z * zs + N); });
  vec* o = reinterpret_cast<vec*>(y + t * ldy + n);
  if constexpr (EPI == EPI_ADD) v += *o;
#pragma unroll
  for (int e = 0; e < V; ++e) {
    if constexpr (EPI == EPI_GELU) v[e] = pf_gelu(v[e]);
    if constexpr (EPI == EPI_SWIGLU) v[e] = pf_silu(v[e]) * u[e];
  }
  *o = v;
}

template <int FMT, int EPI, int MT, int KH>
hipError_t go(PfGemmArgs a, hipStream_t s) {
  const int per_tile = GW * 16 * (EPI == EPI_SWIGLU ? nt_of<FMT>() / 2 : nt_of<FMT>());
  int ntiles = 0;
  for (int k = 0; k < a.nseg; ++k) {
    a.seg[k].tile0 = ntiles;
    ntiles += (int)((a.seg[k].rows + per_tile - 1) / per_tile);
  }
  constexpr int lds = KH * Lds<FMT, MT>::total;
  static_assert(KH == 1 || lds >= MT * nt_of<FMT>() * GW * 64 * 16, "the groups' exchange");
  static_assert(lds <= 160 * 1024, "LDS of a CU");
  if (lds > lds_limit()) return hipErrorInvalidValue;
  if (lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_pf_mm<FMT, EPI, MT, KH>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return e;
  }
  dim3 grid((unsigned)ntiles, (unsigned)(a.gtab ? a.ntab : a.mpad / (16 * MT)), (unsigned)a.ksplit);
  UAII_LAUNCH((k_pf_mm<FMT, EPI, MT, KH>), grid, dim3(GW * 64 * KH), lds, s, a);
  return hipGetLastError();
}

// The kernel's format.
int kernel_fmt(const PfGemmArgs& a) {
  const int type = a.seg[0].w.type;
  return a.carry && type == T_Q8_0 ? Q8_0_CARRY : type;
}

// Column tiles of a launch.
int64_t col_tiles(const PfGemmArgs& a) {
  const int fmt = kernel_fmt(a);
  const int per = GW * 16 * (fmt == T_F16 || fmt == Q8_0_CARRY ? 2 : 4) / (a.epi == EPI_SWIGLU ? 2 : 1);
  int64_t n = 0;
  for (int k = 0; k < a.nseg; ++k) n += (a.seg[k].rows + per - 1) / per;
  return n;
}

// Row subtiles per block, at most what the rows fill (the expert tables are built
// for 64-row groups).
int row_tiles(const PfGemmArgs& a) {
  if (a.gtab) return 4;
  // Few blocks leave the chip to the latency of each one, which grows with its rows; but
  // blocks of fewer rows read the weights more often, and leave less of the chip to split
  // K over. So the line is one of blocks and of the K that they go through (b1, blocks at
  // 16 rows, times K). Microseconds at 16, 32, 64 rows a block, whole calls:
  //                        b1  b1 K / 2^18   Q8_0          Q4_K          Q6_K
  //   100 x 1536 x 512     48  0.1          14  17  22    14  17  22    15  18  23
  //   300 x 1408 x 512 +  220  0.4          15  20  24    16  20  24    18  21  25
  //   500 x 1408 x 512 +  352  0.7          24  19  26    20  20  27    30  22  27
  //   200 x 2048 x 2048   128  1            25  26  32    28  28  32    32  29  33
  //   100 x 4096 x 4096   128  2            34  30  32    40  33  32    48  36  35
  //   100 x 2048 x 8192    64  2            36  33  36    42  35  35    50  38  38
  //   60 x 4096 x 14336    64  3.5          50  43  46    61  47  45    74  51  53
  //   300 x 4096 x 4096   320  5            94  66  51    78  75  49   150  84  57
  //   300 x 4096 x 14336  320  18          297 203 118   247 234 112   477 267 134
  // (+ SwiGLU.) Q4_0 and Q5_K fall as Q8_0 and Q4_K do. F16's column tiles are half as
  // wide: 100 x 4096 x 4096 74, 69, 60; 300 x 4096 x 14336 581, 818, 654.
  // Q6_K, with half as many matrix ops again to a block, leaves 16 rows at half the line.
  const int64_t b1 = col_tiles(a) * (a.mpad / 16), w = b1 * a.K;
  if (a.mpad == 16 || (b1 <= 256 && w <= (1 << (a.seg[0].w.type == T_Q6_K ? 17 : 18)))) return 1;
  return a.mpad == 32 || (b1 <= 384 && w <= (1 << 19)) ? 2 : 4;
}

// Wave groups per block: two where the grid has no more blocks than the chip has CUs.
int k_groups(const PfGemmArgs& a, int cus) {
  if (row_tiles(a) != 4) return 1;
  const int64_t blocks = col_tiles(a) * (a.gtab ? a.ntab : a.mpad / 64) * a.ksplit;
  return blocks <= cus && (a.K + 255) / 256 >= 2 * a.ksplit ? 2 : 1;
}

template <int FMT, int EPI>
hipError_t go_rows(const PfGemmArgs& a, hipStream_t s) {
  switch (row_tiles(a)) {
    case 1: return go<FMT, EPI, 1, 1>(a, s);
    case 2: return go<FMT, EPI, 2, 1>(a, s);
    default: return k_groups(a, device_cus()) == 2 ? go<FMT, EPI, 4, 2>(a, s) : go<FMT, EPI, 4, 1>(a, s);
  }
}

template <int FMT>
hipError_t go_epi(const PfGemmArgs& a, hipStream_t s) {
  switch (a.epi) {
    case EPI_STORE: return go_rows<FMT, EPI_STORE>(a, s);
    case EPI_ADD: return go_rows<FMT, EPI_ADD>(a, s);
    case EPI_SWIGLU: return go_rows<FMT, EPI_SWIGLU>(a, s);
    case EPI_GELU: return go_rows<FMT, EPI_GELU>(a, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

bool pf_supported(int type) {
  return type == T_Q4_0 || type == T_Q8_0 || type == T_F16 || type == T_Q4_K || type == T_Q5_K || type == T_Q6_K;
}

bool pf_required(int type) { return type == T_Q4_0 || type == T_Q8_0 || type == T_Q4_K || type == T_Q6_K; }

int pf_device_cus() { return device_cus(); }

bool pf_k_quant(int type) { return type == T_Q4_K || type == T_Q5_K || type == T_Q6_K; }

int64_t pf_mpad(int64_t m) { return m <= 16 ? 16 : m <= 32 ? 32 : (m + 63) / 64 * 64; }

int pf_gemm_group_rows(int type) { return 64; }

int pf_gemm_ksplit(const PfGemmArgs& a, int cus, int64_t part_floats) {
  if (a.gtab || a.nseg < 1 || a.M > 65535 || !pf_supported(a.seg[0].w.type)) return 1;
  int64_t rows = 0;
  for (int k = 0; k < a.nseg; ++k) rows += a.seg[k].rows;
  if (a.epi == EPI_SWIGLU) rows *= 2;
  const int64_t tiles = std::max<int64_t>(1, col_tiles(a) * (a.mpad / (16 * row_tiles(a))));
  const int64_t units = (a.K + 255) / 256;
  // one block per CU (of two wave groups each where the rows make for 64-row blocks)
  int64_t ks = std::min<int64_t>(std::min<int64_t>(units, 32), cus / tiles);
  if (a.M * rows > 0) ks = std::min<int64_t>(ks, part_floats / (a.M * rows));
  return (int)std::max<int64_t>(ks, 1);
}

template <int EPI>
static hipError_t fold(const PfGemmArgs& a, hipStream_t s) {
  const int64_t N = a.seg[0].rows;
  // four columns a thread where every row of the partials and of y starts on 16 bytes
  if (N % 4 == 0 && a.ldp % 4 == 0 && a.ldy % 4 == 0 && (uintptr_t)a.y % 16 == 0 && (uintptr_t)a.part % 16 == 0) {
    UAII_LAUNCH((k_pf_fold<EPI, 4>), dim3((unsigned)((N + 1023) / 1024), (unsigned)a.M), dim3(256), 0, s, a.part,
                a.ksplit, a.M, N, a.ldp, a.y, a.ldy);
  } else {
    UAII_LAUNCH((k_pf_fold<EPI, 1>), dim3((unsigned)((N + 255) / 256), (unsigned)a.M), dim3(256), 0, s, a.part,
                a.ksplit, a.M, N, a.ldp, a.y, a.ldy);
  }
  return hipGetLastError();
}

hipError_t launch_pf_fold(const PfGemmArgs& a, hipStream_t s) {
  if (a.ksplit < 2 || a.nseg != 1 || a.seg[0].col0 != 0 || a.M > 65535) return hipErrorInvalidValue;
  switch (a.epi) {
    case EPI_STORE: return fold<EPI_STORE>(a, s);
    case EPI_ADD: return fold<EPI_ADD>(a, s);
    case EPI_GELU: return fold<EPI_GELU>(a, s);
    case EPI_SWIGLU: return fold<EPI_SWIGLU>(a, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_pf_gemm(PfGemmArgs a, hipStream_t s) {
  if (a.ksplit < 1) a.ksplit = 1;
  if (a.act_ld <= 0) a.act_ld = a.mpad;
  if (!a.arow && !a.gtab && a.act_ld != a.mpad) return hipErrorInvalidValue;
  if (a.nseg < 1 || a.nseg > 3 || a.M <= 0 || a.M > a.mpad || a.mpad != pf_mpad(a.mpad) || a.K % 64)
    return hipErrorInvalidValue;
  if (a.gtab) {
    // every table entry lies inside [0, M) and names an expert below ngroups (the
    // caller builds it on the host); here the launch itself is checked
    if (a.ntab < 1 || a.ngroups < 1 || a.ksplit != 1 || a.nseg != 1 ||
        a.gbm != pf_gemm_group_rows(a.seg[0].w.type) || (!a.arow && a.act_ld < a.mpad))
      return hipErrorInvalidValue;
    const PfSeg& sg = a.seg[0];
    if (sg.rows * a.ngroups > sg.w.rows || (a.epi == EPI_SWIGLU && sg.rows * a.ngroups > sg.w2.rows))
      return hipErrorInvalidValue;
  }
  const int type = a.seg[0].w.type;
  if (!pf_supported(type) || (pf_k_quant(type) && a.K % 256)) return hipErrorInvalidValue;
  if ((type == T_Q4_K || type == T_Q5_K) && !a.sxp) return hipErrorInvalidValue;
  // Rows are addressed by 32-bit byte offsets inside a 32-block; the Q4_0 and Q8_0
  // bound is that of the entry points' contract.
  if (a.act_ld * 64 >= (int64_t(1) << 31) || a.K >= (int64_t(1) << 31)) return hipErrorInvalidValue;
  if ((type == T_Q4_0 || type == T_Q8_0) && a.act_ld * a.K * 2 >= (int64_t(1) << 31)) return hipErrorInvalidValue;
  if (a.ksplit > 1 && (!a.part || a.ksplit > (a.K + 255) / 256 || a.ksplit > 64)) return hipErrorInvalidValue;
  if (a.epi == EPI_SWIGLU && a.nseg != 1) return hipErrorInvalidValue;
  for (int k = 0; k < a.nseg; ++k) {
    const PfSeg& sg = a.seg[k];
    if (sg.w.type != type || sg.w.cols != a.K || sg.rows <= 0 || sg.rows > sg.w.rows)
      return hipErrorInvalidValue;
    if (a.epi == EPI_SWIGLU && (sg.w2.type != type || sg.w2.cols != a.K || sg.rows > sg.w2.rows))
      return hipErrorInvalidValue;
  }
  switch (kernel_fmt(a)) {
    case T_Q4_0: return go_epi<T_Q4_0>(a, s);
    case T_Q8_0: return go_epi<T_Q8_0>(a, s);
    case Q8_0_CARRY: return go_epi<Q8_0_CARRY>(a, s);
    case T_F16: return go_epi<T_F16>(a, s);
    case T_Q4_K: return go_epi<T_Q4_K>(a, s);
    case T_Q5_K: return go_epi<T_Q5_K>(a, s);
    case T_Q6_K: return go_epi<T_Q6_K>(a, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace uaii_hip
