// kh_pair.h — prompt GEMMs on the fp16 matrix cores with both operands kept to 32-bit accuracy (.bin models; the
// reference multiplies the prompt one token at a time: cpu/matmul_kernel.cpp:5-41, cuda/matmul_kernel.cu:56-87).
//
//   C[rows, T] = W[rows, K] . X[T, K]^T      every number v of X and of fp32 weights travels as a PAIR of halves
//       hi = fp16(s v),  lo = fp16(s v - hi)          s a power of two
// hi + lo is s v to at most one unit in the last place of fp32 (11 + 11 bits and the sign of lo) for |s v| from 2^-2 to 2^15
// and to 2^-25 absolutely below that, where lo is a subnormal.  A product takes three matrix instructions (hi hi, hi lo,
// lo hi; lo lo is 2^-22 of it at most) of v_mfma_f32_16x16x32_f16 into fp32 accumulators.  int8 weights are exact in
// fp16 and take two; their group scale is applied in fp32 to the sum of each 64-column group.
// Against v_mfma_f32_16x16x4_f32 the unit is 16 times as fast, so 5.3 (8) times the work per cycle is left, and a sum is
// rounded once per 32 columns and product instead of once per 4 columns.
//
// Scales bring the largest number that they cover to [2^14, 2^15): numbers down to 2^-16 of it keep the accuracy of fp32,
// smaller ones have an error of 2^-39 of it.  Normed rows have one per token (k_pair_rmsnorm).  Attention outputs and the
// gated unit have one per token and 64 columns, found where they are made (passes of few tokens: 32, see kPairTiles): a few
// columns may be far above the others there, and a bound from the weights would have to hold for all of them (one row each
// of w1 and w3 at 2^12 of its usual size, undone by w2: K/V rows 2.5e-2 from 64 bits instead of 4e-7).  A row of fp32 weights
// has one in every workgroup that reads it, from its first 32 columns, which it brings to [2^9, 2^10).  Where a number
// behind them is too large for a half (2^6 times as large at least), the sums are no longer finite, and the wave starts
// again with scales from all columns; a row that begins with zeros is read through at once.  (Following the largest number
// in the loop instead made w1 + w3 of Llama-3.2-1B 5 % slower at 512 tokens.)  Nothing is kept from one pass to the next:
// weights may be written between two calls.
// Where every wave starts again (one such number in 1 % of the rows), a prompt takes 2.2 / 1.9 / 1.95 times as long at 128 /
// 512 / 1900 tokens as without, 1.8 / 0.95 / 0.7 times as long as on the fp32 matrix cores.  (With one request in flight in
// the second way and in the search for the scales: 3.5 / 3.3 / 3.2 times as long as without.  The workgroup once more through
// its ring, decided by a vote: 2.35 / 2.0 / 1.95, and 1 % slower where nothing overflows.)
// Where the last token of a prompt is in the pass (pair_takes_last), logits come from it: see `product`.
// K/V rows of models of eight layers and 400 tokens, rms against 64 bits: 4.3e-7 (int8), 5.6e-7 (fp32); on the fp32 matrix
// cores 1.2e-6 and 1.3e-6.  That needs numbers that weigh alike in a result to lie within about 2^12 of one another where
// they share a scale.
//
// Kernel: the stage ring of kh_lgemm.h.  A workgroup owns BM tokens x BN weight rows; a stage of 32 (int8: 64) columns
// is moved to LDS by global_load_lds_dwordx4 in 128-byte rows (pairs: 32 hi | 32 lo; fp32 weights as they lie in the
// file; int8 64-byte rows), swizzled so that the 16 rows of a fragment touch all banks.  fp32 weights are split in
// registers behind the LDS read: two numbers take two multiplications, two v_cvt_pk_f16_f32 and two v_fma_mix_f32.
// (v_fma_mixlo / mixhi would be fewer, but they run at half the rate: w1 + w3 of Llama-3.2-1B at 2048 tokens took 462 us
// with them against 389.)  Weights are the first MFMA operand, so a lane ends with four consecutive rows of one token.
#pragma once
#include <type_traits>

#include "kh_gemm.h"
#include "kh_q8ring.h"

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

// Chunk c (16 bytes) of a 128-byte LDS row r lies in slot c ^ pair_swz(r).  ds_read_b128 serves 16 lanes at a time - 0-3,
// 12-15, 20-27 and 4-11, 16-19, 28-31 of each half wave (found by fitting SQ_LDS_BANK_CONFLICT of four layouts) - and
// 64 banks hold two rows: with this table every fragment read of the kernel (16 rows; chunk h, 2 h or 2 (h & 1) by lane
// group h) is free of conflicts, with r & 7 a third of the LDS cycles were.
__device__ __forceinline__ int pair_swz(int r) { return ((r & 2) << 1) | ((r & 4) ? 3 : 0); }
#define KH_PAIR_STAGE(Q) ((Q) ? 64 : 32)  // columns of a stage
#define KH_PAIR_TOP 15  // a bound is scaled to less than 2^15: a factor of two below the largest fp16

struct KhPairArgs {
  KhLin w[3];          // QKV: wq, wk, wv; RESID: w[0]; SWIGLU: w1, w3
  const char* X;       // pair slab: [T][K / 32][32 hi | 32 lo]
  const float* xs;     // QKV, SWIGLU: 1 / its scales, one per token
  const unsigned char* xe;  // RESID: 1 / its scales, one per token and stage of columns, at pair_exp_at
  int xe_ld;
  int fine;            // RESID, fp32: the two stages of 64 columns may differ in scale
  int keep;            // the last token's result goes into logits: its sums are kept longer
  float* out;          // QKV: Q [T][ldo]; RESID: X [T][ldo] (+=)
  char* pairs;         // SWIGLU: pair slab of the gated unit, [T][ldo / 32]
  unsigned char* out_e;  // SWIGLU: 1 / its scales
  float* kc;           // QKV: K / V cache rows of this layer, row (pos0 + t) * rows1
  float* vc;
  float* part;         // RESID with gridDim.y > 1: partial rows [z][tcap][ldo], added by the k_pair_rmsnorm that follows
  int rows0, rows1;    // QKV: rows of wq, of wk = wv; else rows0 = rows of one matrix
  int N;               // rows of all matrices together
  int ldo, K, T, pos0, tcap, tiles_t, tiles_f;
  int rope, head_size; // QKV: KH_PG_ROPE_* in the epilogue
  const float* sin_cache;
  const float* cos_cache;
};

__device__ __forceinline__ f32x4 mfma_pair(const f16x8& a, const f16x8& b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}
// two floats to two halves, round to nearest even (v_cvt_pk_f16_f32)
__device__ __forceinline__ f16x2 pair_cvt(float a, float b) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  return __builtin_convertvector((f32x2{a, b}), f16x2);
}
// byte offset of the hi half of column k of a row of pairs; the lo half lies 64 bytes further
__host__ __device__ __forceinline__ size_t pair_at(int k) { return (size_t)(k >> 5) * 128 + (k & 31) * 2; }
__device__ __forceinline__ void pair_store4(char* row, int k, const f32x4& v, float s) {
  f16x4 hi, lo;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    hi[i] = (_Float16)(v[i] * s);
    lo[i] = (_Float16)__builtin_fmaf(v[i], s, -(float)hi[i]);
  }
  *(f16x4*)(row + pair_at(k)) = hi;
  *(f16x4*)(row + pair_at(k) + 64) = lo;
}
__device__ __forceinline__ float pair_top4(const f32x4& v) {
  return fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)));
}
// power of two that brings `bound` to [2^(top - 1), 2^top), 2^100 at most (the smallest one for infinities and NaN)
__device__ __forceinline__ float pair_scale_to(float bound, int top) {
  const int e = (int)((__float_as_uint(bound) >> 23) & 255) - 126;  // |bound| < 2^e
  int k = top - e;
  k = k < -114 ? -114 : (k > 100 ? 100 : k);
  return __uint_as_float((unsigned)(k + 127) << 23);
}
__device__ __forceinline__ float pair_scale(float bound) { return bound == 0.f ? 1.0f : pair_scale_to(bound, KH_PAIR_TOP); }
__device__ __forceinline__ float pair_inv(float s) { return __uint_as_float(0x7f000000u - __float_as_uint(s)); }  // 1 / s
// 1 / s as its exponent, and where that of a token and a stage lies: 16 stages of a token side by side
__device__ __forceinline__ unsigned char pair_exp(float s) { return (unsigned char)(254u - (__float_as_uint(s) >> 23)); }
__device__ __forceinline__ size_t pair_exp_at(int stage, int t, int ld) { return ((size_t)(stage >> 4) * ld + t) * 16 + (stage & 15); }
__host__ __device__ __forceinline__ size_t pair_exp_bytes(int K, bool q, int tokens) {
  return (size_t)((K / KH_PAIR_STAGE(q) + 15) / 16) * 16 * tokens;
}
// eight int8, times sgn = +-1 -> fp16, exact: 0x6400 + u is 1024 + u, u = q + 128
__device__ __forceinline__ f16x8 pair_q8(unsigned a, unsigned b, float sgn) {
  const f16x2 one = {(_Float16)sgn, (_Float16)sgn}, bias = {(_Float16)(-1152.0f * sgn), (_Float16)(-1152.0f * sgn)};
  union { f16x8 v; f16x2 p[4]; } r;
  const unsigned src[2] = {a ^ 0x80808080u, b ^ 0x80808080u};
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    union { unsigned u; f16x2 h; } lo, hi;
    lo.u = __builtin_amdgcn_perm(0x64646464u, src[i], 0x04010400u);
    hi.u = __builtin_amdgcn_perm(0x64646464u, src[i], 0x04030402u);
    r.p[2 * i] = __builtin_elementwise_fma(lo.h, one, bias);
    r.p[2 * i + 1] = __builtin_elementwise_fma(hi.h, one, bias);
  }
  return r.v;
}

// GROUP: whether X has a scale per group of columns
template <bool Q, bool GROUP, int TM, int TN, int WM, int WN, int NST>
struct PairCfg {
  static constexpr int BM = 16 * TM * WM, BN = 16 * TN * WN, NW = WM * WN;
  static constexpr int XB = Q ? 2 : 1;                     // 128-byte blocks of a token per stage
  static constexpr int XR = BM * XB / 8;                   // 1-KiB requests: activations
  static constexpr int WR = Q ? BN / 16 : BN / 8;          // weights
  static constexpr int SR = Q ? BN / 64 : 0;               // 256-byte requests: group scales of int8 weights
  static constexpr int EX = GROUP ? (BM + 63) / 64 : 0;    // 1-KiB requests: scales of 16 stages, by the first waves
  static constexpr int STAGE = (XR + WR) * 1024 + SR * 256;
  static constexpr int NL = XR / NW + WR / NW + (Q ? 1 : 0);  // requests of a wave per stage
  static constexpr int LDS = NST * STAGE + 2 * EX * 1024;
  static_assert(NW % 2 == 0 && XR % NW == 0 && WR % NW == 0, "every wave issues the same number of requests");
};

// blockIdx.x -> (row tile, token tile): every XCD (blocks go round them) takes an eighth of the tiles, row tile by row tile, so the
// token tiles of a row tile run on one XCD, or on two, and its weights cross HBM once or twice.  (Whole row tiles an XCD leave some
// with one more than others: 20 of them by 25 token tiles, wq + wk + wv of TinyLlama at 777 tokens, 72.8 -> 48.1 us.)  blockIdx.y = K
// slice (RESID).
template <bool Q, int EPI, int TM, int TN, int WM, int WN, int NST>
__global__ __launch_bounds__(64 * WM * WN, 2) void k_pair_gemm(const KhPairArgs a) {
  constexpr bool GROUP = EPI == KH_PG_RESID;
  typedef PairCfg<Q, GROUP, TM, TN, WM, WN, NST> C;
  extern __shared__ __attribute__((aligned(1024))) char smem_raw[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int xcd = (int)blockIdx.x & 7, all = a.tiles_f * a.tiles_t, tile = (xcd * all >> 3) + ((int)blockIdx.x >> 3);
  if (tile >= (xcd + 1) * all >> 3) return;  // uniform: the grid is rounded up
  const int ft = tile / a.tiles_t, tt = tile % a.tiles_t;
  const int t0 = tt * C::BM, f0 = ft * C::BN;
  const int K = a.K;
  // place f of the stacked rows -> matrix, row.  Runs of 16 places are runs of 16 rows: SWIGLU takes 16 rows of w1, the
  // same 16 of w3, ...; half-mode RoPE takes 16 rows of a head, then their 16 partners half a head further.
  auto place = [&](int f, int& mat, int& row) __attribute__((always_inline)) {
    mat = 0;
    row = f;
    if (EPI == KH_PG_SWIGLU) {
      mat = (f >> 4) & 1;
      row = (f >> 5) * 16 + (f & 15);
    } else if (EPI == KH_PG_QKV) {
      if (f >= a.rows0 + a.rows1) {
        mat = 2;
        row = f - a.rows0 - a.rows1;
      } else if (f >= a.rows0) {
        mat = 1;
        row = f - a.rows0;
      }
      if (a.rope == KH_PG_ROPE_TILES) {
        const int head = row / a.head_size, q = row - head * a.head_size;
        row = head * a.head_size + (q >> 5) * 16 + (q & 15) + ((q & 16) ? a.head_size >> 1 : 0);
      }
    }
  };
  // The tile with the token that logits come from: its 16-row tiles turn within a wave until that token lies in the last of
  // them, whose sums are kept longer (fold).
  constexpr bool KEEPS = Q || EPI != KH_PG_QKV;
  const bool keep = KEEPS && a.keep && t0 + C::BM >= a.T;  // uniform
  const int turn = keep ? ((a.T - 1 - t0) >> 4) + 1 : 0;
  auto token_of = [&](int r) __attribute__((always_inline)) {
    const int m = r >> 4;
    return t0 + ((m / TM * TM + (m + turn) % TM) << 4) + (r & 15);
  };
  // ---- staging addresses
  static_assert(TN % 2 == 0, "both tiles of a SWIGLU or half-mode RoPE pair lie in one wave");
  constexpr int NX = C::XR / C::NW, NWR = C::WR / C::NW;
  unsigned xoff[NX], woff;  // per lane; the rows of a wave's weight requests differ by their bases
  const char* wbase[NWR];
  const char* sbase = nullptr;
  const int sub = lane >> 3, ch8 = (lane & 7) ^ pair_swz(sub);
  const int groups = (K + 63) >> 6, stages = K >> (Q ? 6 : 5);  // slices begin at a multiple of 64 columns
  const int z0 = (int)((long)blockIdx.y * groups / gridDim.y) * (Q ? 1 : 2);
  int z1 = (int)((long)(blockIdx.y + 1) * groups / gridDim.y) * (Q ? 1 : 2);
  z1 = z1 < stages ? z1 : stages;
#pragma unroll
  for (int j = 0; j < NX; ++j) {
    const int r = 8 * (j * C::NW + wave) + sub;  // LDS row: block-major for int8
    int t = token_of(Q ? r % C::BM : r);
    t = t < a.T ? t : a.T - 1;
    xoff[j] = (unsigned)t * (unsigned)(4 * K) + (Q ? (unsigned)(r / C::BM) * 128u : 0u) + 16u * ch8 + (unsigned)z0 * (128u * C::XB);
  }
#pragma unroll
  for (int j = 0; j < NWR; ++j) {
    const int run = Q ? 16 : 8;
    int f = f0 + run * (j * C::NW + wave);
    f = f < a.N - run ? f : a.N - run;
    int mat, row;
    place(f, mat, row);
    wbase[j] = (const char*)a.w[mat].w + ((size_t)(unsigned)row * (unsigned)K + (unsigned)z0 * (Q ? 64u : 32u)) * (Q ? 1 : 4);
  }
  if (Q) {
    const int rr = lane >> 2, ch = (lane & 3) ^ ((rr & 4) >> 1);
    woff = (unsigned)rr * (unsigned)K + 16u * ch;
  } else {
    woff = (unsigned)sub * (unsigned)(4 * K) + 16u * ch8;
  }
  if (Q) {  // scales of 64 places: one dword a lane (SWIGLU and RoPE runs of 16 may lie in two matrices: 64-bit addresses)
    int f = f0 + 64 * (wave % (C::SR ? C::SR : 1)) + lane;
    f = f < a.N ? f : a.N - 1;
    int mat, row;
    place(f, mat, row);
    sbase = (const char*)(mat == 0 ? a.w[0].scales : (mat == 1 ? a.w[1].scales : a.w[2].scales)) +
            ((size_t)row * (K >> 6) + z0) * 4;
  }
  const unsigned lds0 = (unsigned)__builtin_amdgcn_readfirstlane((int)kh_lds_addr(smem_raw)) + 1024u * wave;
  auto issue = [&](int slot) __attribute__((always_inline)) {
    const unsigned d = lds0 + (unsigned)(slot * C::STAGE);
#pragma unroll
    for (int j = 0; j < NWR; ++j) {
      dma_x4_keep(wbase[j], woff, d + (unsigned)(C::XR * 1024 + j * C::NW * 1024));
      wbase[j] += Q ? 64 : 128;
    }
#pragma unroll
    for (int j = 0; j < NX; ++j) {
      dma_x4_keep(a.X, xoff[j], d + (unsigned)(j * C::NW * 1024));
      xoff[j] += 128 * C::XB;
    }
    if (Q) {
      const unsigned sd = lds0 - 1024u * wave + (unsigned)(slot * C::STAGE + (C::XR + C::WR) * 1024) +
                          256u * (unsigned)(wave % (C::SR ? C::SR : 1));
      dma_x1_keep(sbase, sd);
      sbase += 4;
    }
  };
  // The scales of 16 stages: 16 bytes a token.  A request per stage (four bytes a token) made these GEMMs 5 % slower.
  auto issue_exps = [&](int c) __attribute__((always_inline)) {
    if (!GROUP || wave >= C::EX) return;
    int r = 64 * wave + lane;
    asm volatile("" : "+v"(r));  // or the offset takes a register throughout the loop
    const int t = token_of(r);
    const unsigned eoff = 16u * (unsigned)(t < a.T ? t : a.T - 1);
    dma_x4_keep(a.xe + (size_t)c * a.xe_ld * 16, eoff, lds0 + (unsigned)(NST * C::STAGE + (c & 1) * C::EX * 1024));
  };
  const int nk = z1 - z0;
  f32x4 acc[TN][TM];
  const int wm = wave % WM, wn = wave / WM;
  const int fr = lane & 15, fh = lane >> 4;
  float wsc[TN];  // fp32 weights: the scale of row fr of every tile, with the sign of the present sum
#pragma unroll
  for (int n = 0; n < TN; ++n)
#pragma unroll
    for (int m = 0; m < TM; ++m) acc[n][m] = f32x4{0.f, 0.f, 0.f, 0.f};
  // Scales are requested 16 stages ahead of their first use, those of a slice's second 16 with the first: a slice may begin at
  // the end of 16 stages, and stage k only waits for what was requested NST - 2 stages before it.
  static_assert(NST - 2 < 16, "scales have landed when they are read");
  issue_exps(z0 >> 4);
  if (((z0 >> 4) + 1) * 16 < z1) issue_exps((z0 >> 4) + 1);
#pragma unroll
  for (int s = 0; s < NST - 1; ++s)
    if (s < nk) issue(s);
  int slot = 0, fill = NST - 1;
  f32x4 grp[Q ? 1 : TN][Q ? 1 : TM];  // fp32 weights: the sums of two stages
  // The matrix unit rounds its sums down: a bias that the mean over many cached rows keeps while it averages everything else
  // (logits behind 1900 prompt tokens: 1.7e-6 from 64 bits instead of 1.3e-6 on fp32 fma chains).  Every other group takes
  // its weights with the sign turned and is subtracted, which cancels it: 1.1e-6.
  float sgn = 1.0f, xinv[TM];
  unsigned xe[TM];
  auto row_top = [&](float v) __attribute__((always_inline)) {  // over the four lanes of row fr
    v = fmaxf(v, __shfl_xor(v, 16));
    return fmaxf(v, __shfl_xor(v, 32));
  };
  auto row_at = [&](int n) __attribute__((always_inline)) {
    int f = f0, mat, row;
    asm volatile("" : "+s"(f));  // or the addresses are kept in registers throughout the loop
    f += (wn * TN + n) * 16;
    f = f < a.N - 16 ? f : a.N - 16;
    place(f, mat, row);
    return (const float*)a.w[mat].w + (size_t)(row + fr) * K;
  };
  auto row_scale = [&](int n) __attribute__((always_inline)) {  // from all columns of the slice
    const float* w = row_at(n);
    float t = 0.f;
#pragma unroll 8
    for (int k = z0 * 32 + 4 * fh; k < z1 * 32; k += 16) t = fmaxf(t, pair_top4(*(const f32x4*)(w + k)));
    return pair_scale(row_top(t));
  };
  auto split = [&](const f32x4 (&wv)[2], float sc, f16x8& wh, f16x8& wl) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
      const float v0 = wv[e >> 2][e & 3], v1 = wv[e >> 2][(e & 3) + 1];
      const f16x2 hi = pair_cvt(v0 * sc, v1 * sc);
      const f16x2 lo = pair_cvt(__builtin_fmaf(v0, sc, -(float)hi.x), __builtin_fmaf(v1, sc, -(float)hi.y));
      wh[e] = hi.x; wh[e + 1] = hi.y;
      wl[e] = lo.x; wl[e + 1] = lo.y;
    }
  };
  // Every group's sum is folded into the accumulators with one rounding of them, the largest error of a long dot product.  The
  // rows of a prompt's tokens are averaged over by those that attend to them, but logits come from the last one's.  Its tile of
  // 16 tokens (m = TM - 1) runs a loop of its own, in which what a fold rounds off is summed and added at the end (lost), and,
  // with fp32 weights, every stage's sum starts from zero and has the product lo lo as well; the other tiles of the workgroup
  // are as ever, and a pass without the last token has no such workgroup.  wq + wk + wv of fp32 do without: their errors stay
  // where they are.  Logits from 64 bits (mean of 4 to 16 models), the token as a step of its own on fp32 fma chains / in the
  // pass with the sums of all others / with its own:
  //   Qwen2.5-0.5B 41, 300 tokens 7.1 7.3e-7 / - - / 6.9 7.0; TinyLlama 700, 1900 1.13 1.09e-6 / - - / 0.98 0.92; Llama-3.2-1B
  //   150, 512 1.17 1.08e-6 / 1.36 1.23 / 1.08 0.86; Llama-2-7B int8 60, 225, 777 3.8 3.7 3.0e-6 / 3.6 3.6 - / 3.2 3.3 2.75;
  //   stories15M 60, 200 2.53 2.49e-7 / - - / 2.56 2.54 (40 models, deviation of a mean 0.04).
  // Prompts without it: 1 to 4 % faster (Llama-2-7B int8 777 tokens 25.9 ms instead of 26.8, Qwen 41 1.84 instead of 1.91).
  auto product = [&](auto kept) __attribute__((always_inline)) {
    constexpr bool KEEP = decltype(kept)::value;
    f32x4 lost[KEEP ? TN : 1];
#pragma unroll
    for (int n = 0; n < (KEEP ? TN : 1); ++n) lost[n] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto fold = [&](int n, int m, int i, float f, float g) __attribute__((always_inline)) {
      const float s = __builtin_fmaf(f, g, acc[n][m][i]);
      if constexpr (KEEP)
        if (m == TM - 1) lost[n][i] += __builtin_fmaf(f, g, acc[n][m][i] - s);
      acc[n][m][i] = s;
    };
    // (of a sum that has overflowed, what was lost is the opposite infinity, then NaN)
    auto settle = [&]() __attribute__((always_inline)) {
      if constexpr (KEEP) {
#pragma unroll
        for (int n = 0; n < TN; ++n)
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[n][TM - 1][i] += fabsf(lost[n][i]) < INFINITY ? lost[n][i] : 0.f;
      }
    };
    auto stage = [&](int k, auto open) __attribute__((always_inline)) {
      constexpr bool OPEN = decltype(open)::value;  // fp32: first stage of a sum
      // stage k has landed when at most the requests of the stages behind it are outstanding
      // (and with it the scales, which were requested before those)
      if (NST > 2 && k + NST - 2 < nk) wait_vm<(NST - 2) * C::NL>();
      else wait_vm<0>();
      __syncthreads();
      const int at = z0 + k;
      if (GROUP && k > 0 && (at & 15) == 0 && ((at >> 4) + 1) * 16 < z1) issue_exps((at >> 4) + 1);
      const unsigned char* exps = (const unsigned char*)smem_raw + NST * C::STAGE + ((at >> 4) & 1) * C::EX * 1024 + (at & 15);
      if (k + NST - 1 < nk) issue(fill);
      const char* st = smem_raw + slot * C::STAGE;
      const char* wst = st + C::XR * 1024;
      if constexpr (!Q) {
        f16x8 xh[TM], xl[TM];
        f32x4 wv[TN][2];
#pragma unroll
        for (int n = 0; n < TN; ++n) {
          const int r = (wn * TN + n) * 16 + fr;
          wv[n][0] = *(const f32x4*)(wst + r * 128 + (((2 * fh) ^ pair_swz(r)) << 4));
          wv[n][1] = *(const f32x4*)(wst + r * 128 + (((2 * fh + 1) ^ pair_swz(r)) << 4));
        }
#pragma unroll
        for (int m = 0; m < TM; ++m) {
          const int r = (wm * TM + m) * 16 + fr;
          xh[m] = *(const f16x8*)(st + r * 128 + ((fh ^ pair_swz(r)) << 4));
          xl[m] = *(const f16x8*)(st + r * 128 + (((4 + fh) ^ pair_swz(r)) << 4));
        }
        if constexpr (GROUP) {
#pragma unroll
          for (int m = 0; m < TM; ++m) xe[m] = exps[((wm * TM + m) * 16 + fr) * 16];
        }
        if (OPEN && k == 0) {
#pragma unroll
          for (int n = 0; n < TN; ++n) {
            const float t = row_top(fmaxf(pair_top4(wv[n][0]), pair_top4(wv[n][1])));
            wsc[n] = pair_scale_to(t, 10);
            if (__builtin_amdgcn_ballot_w64(t == 0.f)) wsc[n] = row_scale(n);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int n = 0; n < TN; ++n) {
          f16x8 wh, wl;
          split(wv[n], wsc[n], wh, wl);
          constexpr int PM = KEEP ? TM - 1 : TM;
#pragma unroll
          for (int m = 0; m < PM; ++m) grp[n][m] = mfma_pair(wl, xh[m], OPEN ? f4_zero() : grp[n][m]);
#pragma unroll
          for (int m = 0; m < PM; ++m) grp[n][m] = mfma_pair(wh, xl[m], grp[n][m]);
#pragma unroll
          for (int m = 0; m < PM; ++m) grp[n][m] = mfma_pair(wh, xh[m], grp[n][m]);
          if constexpr (KEEP) {
            constexpr int m = TM - 1;
            f32x4 g = mfma_pair(wl, xl[m], f4_zero());
            g = mfma_pair(wh, xh[m], mfma_pair(wh, xl[m], mfma_pair(wl, xh[m], g)));
            if (OPEN) grp[n][m] = g;
            else grp[n][m] += g;
          }
        }
      } else {
        // lane (i, h) takes columns 16 h .. + 15 of its 64-column group; either product takes eight of them
        constexpr bool LATE = KEEP && GROUP && TM > 4;  // the scales of the weights behind the products, or it spills
        f16x8 xh[TM][2], xl[TM][2];
        i32x4 qv[TN];
        f32x4 sc[TN];
#pragma unroll
        for (int n = 0; n < TN; ++n) {
          const int r = (wn * TN + n) * 16 + fr;
          qv[n] = *(const i32x4*)(wst + r * 64 + ((fh ^ ((r & 4) >> 1)) << 4));
          if (!LATE) sc[n] = *(const f32x4*)(wst + C::WR * 1024 + ((wn * TN + n) * 16 + 4 * fh) * 4);
        }
#pragma unroll
        for (int m = 0; m < TM; ++m) {
          const int r = (wm * TM + m) * 16 + fr;
          const char* row = st + ((fh >> 1) * C::BM + r) * 128;
#pragma unroll
          for (int b = 0; b < 2; ++b) {
            const int c = 2 * (fh & 1) + b;
            xh[m][b] = *(const f16x8*)(row + ((c ^ pair_swz(r)) << 4));
            xl[m][b] = *(const f16x8*)(row + (((4 + c) ^ pair_swz(r)) << 4));
          }
        }
        if constexpr (GROUP) {
#pragma unroll
          for (int m = 0; m < TM; ++m) xe[m] = exps[((wm * TM + m) * 16 + fr) * 16];
        }
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int m = 0; m < TM; ++m)
          if (GROUP) xinv[m] = sgn * __uint_as_float(xe[m] << 23);
#pragma unroll
        for (int n = 0; n < TN; ++n) {
          const f16x8 w0 = pair_q8((unsigned)qv[n].x, (unsigned)qv[n].y, sgn), w1 = pair_q8((unsigned)qv[n].z, (unsigned)qv[n].w, sgn);
          f32x4 g[TM];
#pragma unroll
          for (int m = 0; m < TM; ++m) g[m] = mfma_pair(w0, xl[m][0], f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
          for (int m = 0; m < TM; ++m) g[m] = mfma_pair(w1, xl[m][1], g[m]);
#pragma unroll
          for (int m = 0; m < TM; ++m) g[m] = mfma_pair(w0, xh[m][0], g[m]);
#pragma unroll
          for (int m = 0; m < TM; ++m) g[m] = mfma_pair(w1, xh[m][1], g[m]);
          if constexpr (LATE) {
            __builtin_amdgcn_sched_barrier(0);
            sc[n] = *(const f32x4*)(wst + C::WR * 1024 + ((wn * TN + n) * 16 + 4 * fh) * 4);
          }
          const f32x4 sg = {sc[n].x * sgn, sc[n].y * sgn, sc[n].z * sgn, sc[n].w * sgn};
#pragma unroll
          for (int m = 0; m < TM; ++m)
#pragma unroll
            for (int i = 0; i < 4; ++i) fold(n, m, i, GROUP ? sc[n][i] * xinv[m] : sg[i], g[m][i]);
        }
      }
      __builtin_amdgcn_s_setprio(0);
      slot = slot + 1 == NST ? 0 : slot + 1;
      fill = fill + 1 == NST ? 0 : fill + 1;
    };
    auto close = [&]() __attribute__((always_inline)) {
      if constexpr (!Q) {
#pragma unroll
        for (int m = 0; m < TM; ++m) xinv[m] = GROUP ? sgn * __uint_as_float(xe[m] << 23) : sgn;
#pragma unroll
        for (int n = 0; n < TN; ++n) {
#pragma unroll
          for (int m = 0; m < TM; ++m)
#pragma unroll
            for (int i = 0; i < 4; ++i) fold(n, m, i, xinv[m], grp[n][m][i]);
          wsc[n] = -wsc[n];
        }
      }
      sgn = -sgn;
    };
    // The wave's tiles once more, from memory, with scales from all columns (x * 0 above: also where the inputs are not finite).
    auto again = [&]() __attribute__((always_inline)) {
      const float* w[TN];
      sgn = 1.0f;
#pragma unroll
      for (int n = 0; n < TN; ++n) {
        wsc[n] = row_scale(n);
        w[n] = row_at(n) + 8 * fh;
        if constexpr (KEEP) lost[n] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int m = 0; m < TM; ++m) acc[n][m] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
      constexpr int PART = GROUP && TM > 4 ? 4 : TM;  // token tiles requested at once (eight with their scales spill)
#pragma nounroll
      for (int k = z0; k < z1; ++k) {
        f32x4 wv[TN][2];
#pragma unroll
        for (int n = 0; n < TN; ++n) {
          wv[n][0] = *(const f32x4*)(w[n] + 32 * k);
          wv[n][1] = *(const f32x4*)(w[n] + 32 * k + 4);
        }
        f16x8 wh[TN], wl[TN];
#pragma unroll
        for (int m0 = 0; m0 < TM; m0 += PART) {
          f16x8 xh[PART], xl[PART];
          unsigned e[PART];
#pragma unroll
          for (int m = 0; m < PART; ++m) {
            int t = token_of((wm * TM + m0 + m) * 16 + fr);
            t = t < a.T ? t : a.T - 1;
            const char* x = a.X + ((unsigned)t * (unsigned)(4 * K) + 128u * k + 16u * fh);
            xh[m] = *(const f16x8*)x;
            xl[m] = *(const f16x8*)(x + 64);
            e[m] = GROUP ? a.xe[pair_exp_at(k, t, a.xe_ld)] : 127u;
          }
          __builtin_amdgcn_sched_barrier(0);  // requests in front of products
          if (m0 == 0) {
#pragma unroll
            for (int n = 0; n < TN; ++n) split(wv[n], sgn * wsc[n], wh[n], wl[n]);
          }
#pragma unroll
          for (int m = 0; m < PART; ++m) {
            const float f = sgn * __uint_as_float(e[m] << 23);
#pragma unroll
            for (int n = 0; n < TN; ++n) {
              const f32x4 g = mfma_pair(wh[n], xh[m], mfma_pair(wh[n], xl[m], mfma_pair(wl[n], xh[m], f4_zero())));
#pragma unroll
              for (int i = 0; i < 4; ++i) fold(n, m0 + m, i, f, g[i]);
            }
          }
        }
        sgn = -sgn;
      }
      settle();
    };
    const std::true_type first{};
    const std::false_type second{};
    if constexpr (Q) {
      for (int k = 0; k < nk; ++k) {
        stage(k, first);
        close();
      }
    } else {
      int k = 0;
      for (; k + 1 < nk; k += 2) {
        stage(k, first);
        if (GROUP && a.fine) {  // uniform
          close();
#pragma unroll
          for (int n = 0; n < TN; ++n)
#pragma unroll
            for (int m = 0; m < TM; ++m) grp[n][m] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        stage(k + 1, second);
        close();
      }
      if (k < nk) {
        stage(k, first);
        close();
      }
    }
    settle();
    if constexpr (!Q) {
      // a half that has overflowed has left infinities or NaN in its row
      float all = 0.f;
#pragma unroll
      for (int n = 0; n < TN; ++n)
#pragma unroll
        for (int m = 0; m < TM; ++m)
#pragma unroll
          for (int i = 0; i < 4; ++i) all = __builtin_fmaf(acc[n][m][i], 0.f, all);
      if (__builtin_amdgcn_ballot_w64(all != 0.f)) again();
    }
  };
  if constexpr (KEEPS) {
    if (keep) product(std::true_type());
    else product(std::false_type());
  } else {
    product(std::false_type());
  }
  // ---- epilogue: lane (fr, fh) of tile (n, m) holds rows 4 fh .. + 3 of the tile for token t0 + .. + fr
  f32x4 wi[TN];
  if constexpr (!Q) {
#pragma unroll
    for (int n = 0; n < TN; ++n)
#pragma unroll
      for (int i = 0; i < 4; ++i) wi[n][i] = pair_inv(__shfl(fabsf(wsc[n]), 4 * fh + i));
  }
  float xi[TM];
#pragma unroll
  for (int m = 0; m < TM; ++m) {
    const int tok = token_of((wm * TM + m) * 16 + fr);
    xi[m] = GROUP ? 1.0f : a.xs[tok < a.T ? tok : a.T - 1];
  }
  auto value = [&](int n, int m) __attribute__((always_inline)) {
    f32x4 v = acc[n][m];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (!GROUP) v[i] *= xi[m];
      if (!Q) v[i] *= wi[n][i];
    }
    return v;
  };
  if constexpr (EPI == KH_PG_SWIGLU) {
    // a wave holds 8 TN columns of the gated unit; 64 columns, those of `per` waves, share a scale, or the 32 of a workgroup
    constexpr int per = WN * TN < 8 ? WN : 8 / TN, sub = KH_PAIR_STAGE(Q) / (8 * TN);  // sub: waves of a stage
    static_assert(sub > 0 && per % sub == 0 && WN % per == 0, "whole stages in a workgroup");
    float* tops = (float*)smem_raw;  // [WN][BM]
    f32x4 o[TM][TN / 2];
    __syncthreads();  // the last stage has been read
#pragma unroll
    for (int m = 0; m < TM; ++m) {
      float top = 0.f;
#pragma unroll
      for (int n = 0; n < TN; n += 2) {
        const int f = f0 + (wn * TN + n) * 16;
        o[m][n / 2] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (f >= a.N) continue;
        const f32x4 g = value(n, m), u = value(n + 1, m);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          o[m][n / 2][i] = swiglu1(g[i], u[i]);
          top = fmaxf(top, fabsf(o[m][n / 2][i]));
        }
      }
      top = fmaxf(top, __shfl_xor(top, 16));
      top = fmaxf(top, __shfl_xor(top, 32));
      if (fh == 0) tops[wn * C::BM + (wm * TM + m) * 16 + fr] = top;
    }
    __syncthreads();
    const int stage = (f0 >> 1) / KH_PAIR_STAGE(Q) + wn / sub;
#pragma unroll
    for (int m = 0; m < TM; ++m) {
      const int at = (wm * TM + m) * 16 + fr, tok = token_of(at);
      if (tok >= a.T) continue;
      float top = 0.f;
#pragma unroll
      for (int w = 0; w < per; ++w) top = fmaxf(top, tops[(wn / per * per + w) * C::BM + at]);
      const float s = pair_scale(top);
      if (fh == 0 && wn % sub == 0 && stage * 2 * KH_PAIR_STAGE(Q) < a.N) a.out_e[pair_exp_at(stage, tok, a.xe_ld)] = pair_exp(s);
#pragma unroll
      for (int n = 0; n < TN; n += 2) {
        const int f = f0 + (wn * TN + n) * 16;
        if (f < a.N) pair_store4(a.pairs + (size_t)tok * a.ldo * 4, (f >> 5) * 16 + 4 * fh, o[m][n / 2], s);
      }
    }
    return;
  }
#pragma unroll
  for (int m = 0; m < TM; ++m) {
    const int tok = token_of((wm * TM + m) * 16 + fr);
    if (tok >= a.T) continue;
#pragma unroll
    for (int n = 0; n < TN; ++n) {
      const int f = f0 + (wn * TN + n) * 16;
      if (f >= a.N) continue;
      int mat, row;
      place(f, mat, row);
      row += 4 * fh;
      if (EPI == KH_PG_RESID) {
        const f32x4 v = value(n, m);
        if (gridDim.y > 1) {
          *(f32x4*)(a.part + ((size_t)blockIdx.y * a.tcap + tok) * a.ldo + row) = v;
        } else {  // residual add (llama3.cpp:686,719)
          f32x4* dst = (f32x4*)(a.out + (size_t)tok * a.ldo + row);
          f32x4 x = *dst;
#pragma unroll
          for (int i = 0; i < 4; ++i) x[i] += v[i];
          *dst = x;
        }
      } else {
        auto biased = [&](f32x4 v, int r) __attribute__((always_inline)) {  // before RoPE (matmul.cpp:74-77)
          if (a.w[mat].bias) {
            const f32x4 b = *(const f32x4*)(a.w[mat].bias + r);
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] += b[i];
          }
          return v;
        };
        float* dst = mat == 0 ? a.out + (size_t)tok * a.ldo : (mat == 1 ? a.kc : a.vc) + (size_t)(a.pos0 + tok) * a.rows1;
        const int hs = a.head_size;
        const float* sn = a.sin_cache + (size_t)(a.pos0 + tok) * hs;
        const float* cs = a.cos_cache + (size_t)(a.pos0 + tok) * hs;
        if (a.rope == KH_PG_ROPE_TILES) {
          if (n & 1) continue;
          // tile n + 1 holds the partners, half a head further; cache column 2 j (cpu/rope_kernel.cpp:18-42)
          const f32x4 lo = biased(value(n, m), row), hi = biased(value(n + 1, m), row + (hs >> 1));
          f32x4 olo = lo, ohi = hi;
          if (mat < 2) {
            const int j = row % hs;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const float s = sn[2 * (j + i)], c = cs[2 * (j + i)];
              olo[i] = lo[i] * c - hi[i] * s;
              ohi[i] = lo[i] * s + hi[i] * c;
            }
          }
          *(f32x4*)(dst + row) = olo;
          *(f32x4*)(dst + row + (hs >> 1)) = ohi;
        } else {
          f32x4 v = biased(value(n, m), row);
          if (mat < 2 && a.rope == KH_PG_ROPE_PAIRS) {  // pairs (row, row + 1) (cpu/rope_kernel.cpp:98-121)
            const int c = row % hs;
            const float s0 = sn[c], c0 = cs[c], s1 = sn[c + 2], c1 = cs[c + 2];
            v = f32x4{v.x * c0 - v.y * s0, v.x * s0 + v.y * c0, v.z * c1 - v.w * s1, v.z * s1 + v.w * c1};
          }
          *(f32x4*)(dst + row) = v;
        }
      }
    }
  }
}

// ---- the per-token kernels between the GEMMs ------------------------------------------------------------------------
// Chunk k (four columns) of token t with a scale per 64 columns, whose chunks lie in 16 neighbouring lanes; chunks from n4 on
// are zeros.  chunks: those of a stage (8 or 16), every stage gets the scale.
__device__ __forceinline__ void pair_emit(char* row, unsigned char* exps, int ld, int t, int k, int n4, int chunks, const f32x4& v) {
  float top = pair_top4(v);
#pragma unroll
  for (int o = 8; o; o >>= 1) top = fmaxf(top, __shfl_xor(top, o));
  if (k >= n4) return;
  const float s = pair_scale(top);
  pair_store4(row, 4 * k, v, s);
  if ((k & (chunks - 1)) == 0) exps[pair_exp_at(k / chunks, t, ld)] = pair_exp(s);
}
// k_pg_rmsnorm (kh_gemm.h) with a row of pairs as its output; one workgroup per token
static __global__ __launch_bounds__(KH_WG) void k_pair_rmsnorm(float* __restrict__ X, const float* __restrict__ w, char* __restrict__ out,
                                                               float* __restrict__ inv, int dim, float eps, int tcap,
                                                               const float* __restrict__ part, int kz) {
  __shared__ float red[KH_WG / KH_WAVE], tops[KH_WG / KH_WAVE];
  const int t = blockIdx.x;
  f32x4* x4 = (f32x4*)(X + (size_t)t * dim);
  const f32x4* w4 = (const f32x4*)w;
  const int n4 = dim >> 2;
  constexpr int KEEP = 4;  // the row stays in registers between the two passes for dim <= 4096
  f32x4 keep[KEEP];
  float ss = 0.f, top = 0.f;
  auto load = [&](int k) __attribute__((always_inline)) {
    f32x4 v = x4[k];
    if (kz > 0) {  // the residual GEMM in front split K: its partial rows, in fixed order
      f32x4 s = f4_zero();
      for (int z = 0; z < kz; ++z) {
        const f32x4 p = *(const f32x4*)(part + ((size_t)z * tcap + t) * dim + 4 * k);
        s.x += p.x; s.y += p.y; s.z += p.z; s.w += p.w;
      }
      v.x += s.x; v.y += s.y; v.z += s.z; v.w += s.w;  // the residual, the largest of them, is rounded once
      x4[k] = v;
    }
    const f32x4 g = w4[k];
    ss = fma4(v, v, ss);
    top = fmaxf(top, pair_top4(f32x4{g.x * v.x, g.y * v.y, g.z * v.z, g.w * v.w}));
    return v;
  };
#pragma unroll
  for (int i = 0; i < KEEP; ++i) {
    const int k = (int)threadIdx.x + i * KH_WG;
    if (k < n4) keep[i] = load(k);
  }
  for (int k = (int)threadIdx.x + KEEP * KH_WG; k < n4; k += KH_WG) (void)load(k);  // (re-read by this same thread below)
  // the row's scale: the largest |g x|, found with the sum of squares
  ss = wave_sum(ss);
  for (int o = 32; o; o >>= 1) top = fmaxf(top, __shfl_xor(top, o));
  if ((threadIdx.x & 63) == 0) {
    red[threadIdx.x >> 6] = ss;
    tops[threadIdx.x >> 6] = top;
  }
  __syncthreads();
  ss = red[0];
  top = tops[0];
#pragma unroll
  for (int i = 1; i < KH_WG / KH_WAVE; ++i) {
    ss += red[i];
    top = fmaxf(top, tops[i]);
  }
  const float rs = 1.0f / sqrtf(ss / (float)dim + eps), s = pair_scale(rs * top);
  if (threadIdx.x == 0) inv[t] = pair_inv(s);
  auto emit = [&](int k, const f32x4& v) __attribute__((always_inline)) {
    const f32x4 g = w4[k];
    pair_store4(out + (size_t)t * dim * 4, 4 * k, f32x4{g.x * (rs * v.x), g.y * (rs * v.y), g.z * (rs * v.z), g.w * (rs * v.w)}, s);
  };
#pragma unroll
  for (int i = 0; i < KEEP; ++i) {
    const int k = (int)threadIdx.x + i * KH_WG;
    if (k < n4) emit(k, keep[i]);
  }
  for (int k = (int)threadIdx.x + KEEP * KH_WG; k < n4; k += KH_WG) emit(k, x4[k]);
}
// rows of pairs and their scales from rows of fp32; one workgroup per token
static __global__ __launch_bounds__(KH_WG) void k_pair_convert(const float* __restrict__ A, char* __restrict__ out,
                                                               unsigned char* __restrict__ exps, int dim, int tcap, int chunks) {
  const int t = blockIdx.x, n4 = dim >> 2;
  const f32x4* a4 = (const f32x4*)(A + (size_t)t * dim);
  for (int k0 = 0; k0 < n4; k0 += KH_WG) {
    const int k = k0 + (int)threadIdx.x;
    pair_emit(out + (size_t)t * dim * 4, exps, tcap, t, k, n4, chunks, k < n4 ? a4[k] : f4_zero());
  }
}
