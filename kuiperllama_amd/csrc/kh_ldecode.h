// kh_ldecode.h — fused decode step of the layer-list models: B sequences (1, 2 or 4), one token each.
//
// Per layer   mixer mamba1: 4 launches      latent attention: 6      attention over heads: 3, or 5
//   k_ld_in   norms -> LDS ; every projection that reads them: mixer input (+ bias), router (+ shared gate row), dense
//             or shared feed-forward's gate / up ; mamba x rows go through the convolution and silu in the epilogue
//   k_ld_mid  router choice, chosen experts' gate / up ; mamba: W_x ; latent: W_uq behind its RMS norm, cache row ;
//             heads: cache row, attention (kh_ldheads.h)
//   mamba     k_ld_scan   dt projection, softplus, one step of the selective scan, gate
//   latent    k_ld_absorb W_uk^T q per head, rotation ; k_latent_attn (time splits) ; k_ld_values merge + W_uv per head
//   heads     of more than 128 elements or over more keys than kh_ldheads.h takes: k_heads_attn (time splits) ; k_ld_merge merge
//             and output gate
//   k_ld_out  W_o . v (+ bias) + experts' down + shared down + identity experts, times the residual multiplier, +
//             residual: one dot product per row over a concatenation of weight rows
// A loop that enters through a matrix: k_ld_enter in front of each pass.  Then k_ld_head (final norm, head, soft cap,
// argmax partials) and the sampler of kh_fused.h.
//
// GEMV core: a wave owns R rows.  A row is cut into BLOCKS of 64 x 16 bytes; U blocks of R rows are requested together
// (non-temporal), and the first tile of a wave is requested before the input vectors are staged.  Vectors lie in LDS
// as fp32, block by block, split into planes of four so that a lane's reads are consecutive 16-byte slots; their tails
// are zeros, so the clamped weight loads of a tail lane contribute nothing.  Accumulation is fp32.
#pragma once
#include "kh_heads.h"
#include "kh_hybrid.h"
#include "kh_ldheads.h"

namespace khm {

template <class T>
struct Ld {
  static constexpr int E = Tile<T>::N;     // elements of a 16-byte load
  static constexpr int P = E / 4;          // float4 planes of a block
  static constexpr int BE = 64 * E;        // elements of a block
  static __host__ __device__ __forceinline__ int blocks(int n) { return (n + BE - 1) / BE; }
  static __host__ __device__ __forceinline__ size_t vec_bytes(int n) { return (size_t)blocks(n) * BE * 4; }
  // place (in floats) of element i of a staged vector
  static __device__ __forceinline__ int place(int i) {
    const int b = i / BE, r = i - b * BE, l = r / E, e = r - l * E;
    return b * BE + ((e >> 2) * 64 + l) * 4 + (e & 3);
  }
};

// float4 group i (elements 4 i ..) of a staged vector: its 16-byte slot
template <class T>
__device__ __forceinline__ int ld_slot(int i) {
  constexpr int B4 = Ld<T>::BE / 4, P = Ld<T>::P;
  const int b = i / B4, r = i - b * B4;
  return b * B4 + (r % P) * 64 + r / P;
}
// n4 valid float4 of src -> slots [0, total4), zeros behind them; times g
template <class T, int NT>
__device__ __forceinline__ void ld_stage(f32x4* xs, const float* src, int n4, int total4, float g, int tid) {
  for (int i0 = tid; i0 < total4; i0 += 4 * NT) {
    f32x4 v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int i = i0 + j * NT;
      v[j] = i < n4 ? ((const f32x4*)src)[i] : f4_zero();
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (i0 + j * NT < total4) xs[ld_slot<T>(i0 + j * NT)] = v[j] * g;
  }
}
// Sums over the wave of R B values per lane, value n = R q + r for row r and vector q.  Two values share each exchange: halves of
// the wave, then rows of 16 lanes, then four steps within a row - 4 + 4 + 2 + 2 + 16 instructions for 16 values where a
// sum of its own for each takes twelve times 16, on vector units that four products per weight keep busy (k_ld_in, k_ld_head).
// The order of a value's additions does not depend on R and B.  Lane l ends with value ld_own(l).n, if it is one's owner.
__device__ __forceinline__ float ld_fold32(float a, float b) {  // lanes 0 .. 31: of a, 32 .. 63: of b
  const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(int, a), __builtin_bit_cast(int, b), false, false);
  return __builtin_bit_cast(float, (int)r[0]) + __builtin_bit_cast(float, (int)r[1]);
}
__device__ __forceinline__ float ld_fold16(float a, float b) {  // even rows: of a, odd rows: of b
  const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(int, a), __builtin_bit_cast(int, b), false, false);
  return __builtin_bit_cast(float, (int)r[0]) + __builtin_bit_cast(float, (int)r[1]);
}
template <int N>
__device__ __forceinline__ float ld_fold(const float (&v)[N], int lane) {
  static_assert(N == 2 || N == 4 || N == 8 || N == 16 || N == 32, "values");
  if constexpr (N == 2) {
    return group_sum<16>(xor16_sum(ld_fold32(v[0], v[1])));
  } else {
    float s[N / 4], x = 0.f;
#pragma unroll
    for (int i = 0; i < N / 4; ++i) s[i] = group_sum<16>(ld_fold16(ld_fold32(v[4 * i], v[4 * i + 1]), ld_fold32(v[4 * i + 2], v[4 * i + 3])));
#pragma unroll
    for (int i = 0; i < N / 4; ++i) x = (lane & 15) == i ? s[i] : x;
    return x;
  }
}
struct LdOwn {
  int n, r, q;
  bool on;
};
template <int R, int B>
__device__ __forceinline__ LdOwn ld_own(int lane) {
  constexpr int N = R * B;
  const int k = lane & 15, g = lane >> 4;
  const int n = N == 2 ? lane >> 5 : 4 * k + ((g & 1) << 1 | g >> 1);
  return {n, n % R, n / R, N == 2 ? (lane & 31) == 0 : k < N / 4};
}
template <int R, int B>
__device__ __forceinline__ float ld_sums(const float (&acc)[R][B], int lane) {
  float v[R * B];
#pragma unroll
  for (int q = 0; q < B; ++q)
#pragma unroll
    for (int r = 0; r < R; ++r) v[q * R + r] = acc[r][q];
  return ld_fold(v, lane);
}
// Rows 0, 1 of four are gates, rows 2, 3 their ups: an owner of row r < 2 gets the other's value in u (and its own in g).
__device__ __forceinline__ void ld_gate_up(float v, float& g, float& u) { KH_SWAP16(v, g, u); }

// Layer norm (rms: RMS norm, shift 0) of Q rows (NT threads, NV float4 of a row each, rows padded with zeros to ld) into LDS
// slots, rows xstride4 slots apart.  v: the rows in registers; the normalised values also go to `out` (ldo4 apart) when given.
// Mean and variance come from ONE workgroup reduction of (x - shift) and (x - shift)^2 for all rows, shift = an element of the
// row: no cancellation beyond the distance of that element from the mean.  Every wave finishes the statistics for itself, those of
// all rows at once in its lanes.  red: 64 floats.  Waves behind the first NT threads only meet the barrier.
template <class T, int NT, int NV, int Q>
__device__ __forceinline__ void ld_norm(const f32x4 (&v)[Q][NV], const f32x4 (&w)[NV], const f32x4 (&b)[NV], const float (&shift)[Q],
                                        bool rms, int W, int n4, int total4, float eps, float* red, f32x4* xs, int xstride4,
                                        f32x4* out, int ldo4) {
  static_assert(NT == 512 && Q <= 4, "eight waves of eight values are the lanes of one");
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (wave >= NT / 64) {  // uniform
    __syncthreads();
    return;
  }
  float s[2 * Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    s[2 * q] = s[2 * q + 1] = 0.f;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int i = threadIdx.x + NT * j;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float d = 4 * i + k < W ? v[q][j][k] - shift[q] : 0.f;
        s[2 * q] += d;
        s[2 * q + 1] = __builtin_fmaf(d, d, s[2 * q + 1]);
      }
    }
  }
  {
    const float x = ld_fold(s, lane);
    const LdOwn o = ld_own<2, Q>(lane);
    if (o.on) red[8 * wave + o.n] = x;
  }
  __syncthreads();
  const int c = lane & 7;  // value c = 2 q (+ 1) of wave lane / 8
  float x = c < 2 * Q ? red[lane] : 0.f;
  x += __shfl_xor(x, 8, 64);
  x = xor32_sum(xor16_sum(x));
  const float y = dpp_f32<KH_DPP_XOR1>(x), s1 = c & 1 ? y : x, s2 = c & 1 ? x : y;
  const float m = rms ? 0.f : s1 / (float)W;
  const float var = fmaxf(s2 / (float)W - m * m, 0.f);
  const float rs = 1.0f / sqrtf(var + eps);
  auto of_row = [&](float z, int q) __attribute__((always_inline)) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, z), 2 * q));
  };
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const float mean = rms ? 0.f : shift[q] + of_row(m, q), rstd = of_row(rs, q);
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int i = threadIdx.x + NT * j;
      f32x4 y;
#pragma unroll
      for (int k = 0; k < 4; ++k) y[k] = (v[q][j][k] - mean) * rstd * w[j][k] + b[j][k];  // pads: zero weight and bias
      if (i < total4) xs[(size_t)q * xstride4 + ld_slot<T>(i)] = i < n4 ? y : f4_zero();
      if (out && i < n4) out[(size_t)q * ldo4 + i] = y;
    }
  }
}
// The rows of how many of B sequences are requested at once and normed behind one reduction: all, where the registers hold them.
// (One after the other they are a load and a reduction each.)
constexpr int ld_rows_at_once(int B, int NV) { return B * NV <= 8 ? B : 1; }

template <class T, int R, int U>
struct LdTile {
  typename Tile<T>::frag v[R][U];
};
// one row set: base address of row r (wave-uniform), valid 16-byte chunks per row
template <class T, int R, int U>
__device__ __forceinline__ void ld_load(LdTile<T, R, U>& t, const T* const (&row)[R], int b0, int nblk, int nch, int lane) {
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int b = b0 + u;
    if (b < nblk) {  // uniform
      int c = b * 64 + lane;
      c = c < nch ? c : nch - 1;
#pragma unroll
      for (int r = 0; r < R; ++r) t.v[r][u] = ld_nt((const typename Tile<T>::frag*)row[r] + c);
    }
  }
}
template <class T>
__device__ __forceinline__ float ld_dot(const typename Tile<T>::frag& w, const f32x4* x /* plane stride 64 */, float acc) {
#pragma unroll
  for (int p = 0; p < Ld<T>::P; ++p) {
    const f32x4 v = x[p * 64];
#pragma unroll
    for (int i = 0; i < 4; ++i) acc = __builtin_fmaf((float)w[4 * p + i], v[i], acc);
  }
  return acc;
}
// xs: LDS vectors, xstride floats apart; b0: the tile's first block
template <class T, int R, int U, int B>
__device__ __forceinline__ void ld_fma(const LdTile<T, R, U>& t, const float* xs, int xstride, int b0, int nblk, int lane,
                                       float (&acc)[R][B]) {
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int b = b0 + u;
    if (b < nblk) {
#pragma unroll
      for (int q = 0; q < B; ++q) {
        const f32x4* x = (const f32x4*)(xs + (size_t)q * xstride + (size_t)b * Ld<T>::BE) + lane;
#pragma unroll
        for (int r = 0; r < R; ++r) acc[r][q] = ld_dot<T>(t.v[r][u], x, acc[r][q]);
      }
    }
  }
}
// the rest of a row set behind its first tile
template <class T, int R, int U, int B>
__device__ __forceinline__ void ld_rows(LdTile<T, R, U>& t, const T* const (&row)[R], int nblk, int nch, const float* xs,
                                        int xstride, int lane, float (&acc)[R][B]) {
  for (int b0 = 0; b0 < nblk; b0 += U) {
    if (b0) ld_load<T, R, U>(t, row, b0, nblk, nch, lane);
    ld_fma<T, R, U, B>(t, xs, xstride, b0, nblk, lane, acc);
  }
}
// A wave's items, `step` apart.  A tile is requested again as soon as its products are done; sixteen waves a CU keep requests in
// flight meanwhile.  set_rows(item, row) gives an item's rows, early(item) requests what done(item, sum) needs beside the sums
// (ld_sums).  ld_items_begin requests the first tile and may come long before.
template <class T, int R, int U, class S>
__device__ __forceinline__ void ld_items_begin(LdTile<T, R, U>& t, int item, int items, int nblk, int nch, int lane, S&& set_rows) {
  if (item >= items) return;
  const T* row[R];
  set_rows(item, row);
  ld_load<T, R, U>(t, row, 0, nblk, nch, lane);
}
template <int B, class T, int R, int U, class S, class E, class D>
__device__ __forceinline__ void ld_items(LdTile<T, R, U>& t, int item, int step, int items, int nblk, int nch, const float* xs, int xstride,
                                         int lane, S&& set_rows, E&& early, D&& done) {
  if (item >= items) return;
  float acc[R][B] = {};
  int b = 0;
  early(item);
  for (;;) {
    ld_fma<T, R, U, B>(t, xs, xstride, b, nblk, lane, acc);
    const bool last = b + U >= nblk;
    const int it2 = last ? item + step : item;
    b = last ? 0 : b + U;
    if (it2 < items) {
      const T* row[R];
      set_rows(it2, row);
      ld_load<T, R, U>(t, row, b, nblk, nch, lane);
    }
    if (!last) continue;
    done(item, ld_sums(acc, lane));
    if (it2 >= items) return;
    item = it2;
    early(item);
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int q = 0; q < B; ++q) acc[r][q] = 0.f;
  }
}

struct LdTabs {
  const int32_t *tok, *pos, *slot;  // [B]
};

// The embedding output of a token: scale * embed[token] + pos_emb[position] (pos_emb nullptr: none), rows of ld elements
struct LdEmbed {
  const void *embed, *pos_emb;
  float scale;
};
template <class T>
__device__ __forceinline__ f32x4 ld_embed(const LdEmbed& e, int tok, int pos, int ld, int i4) {
  f32x4 v = quad_f((const T*)e.embed + (size_t)tok * ld + 4 * i4) * e.scale;
  if (e.pos_emb) v += quad_f((const T*)e.pos_emb + (size_t)pos * ld + 4 * i4);
  return v;
}

// ---- k_ld_in -----------------------------------------------------------------------------------------------------
enum LdInKind { LDI_PLAIN = 0, LDI_CONV = 1, LDI_GATED = 2 };
struct LdInSeg {
  const void* w;
  float* out;      // [B][ldo]
  const float* bias;  // LDI_PLAIN: one per row, or nullptr
  int rows, ldo, kind, norm2;  // rows: weight rows (GATED: output columns); norm2: input is the second norm
  int wg0, nwg;
};
struct LdInArgs {
  LdInSeg seg[3];
  int nseg;
  const float* x_in;   // [B][ld]
  float* x_cur;        // written by workgroup 0 when the input is modified
  LdEmbed emb;
  const float* step;
  const float *w1, *b1, *w2, *b2;  // b: nullptr with rms
  float* xn2;          // [B][ld], written by the router's first workgroup xn2_wg (nullptr: nobody reads it)
  int xn2_wg;
  int W, ld, from_embed, add_x0, rms;
  float eps;
  GateAct act;
  LdTabs t;
  // LDI_CONV
  const float *conv_w, *conv_b;
  float *conv_st, *xc;  // state + slot * slot_stride ; convolved inputs [B][xc_ld]
  size_t slot_stride;
  int inner, taps, xc_ld;
};

// k_ld_in and k_ld_head: one workgroup of sixteen waves per CU, which stages the rows once.  The first eight request the rows and
// norm them, the others meanwhile weights: a wave that has requested more than the memory pipe takes (32 KB a CU are in
// flight) is held up where it is, and the norm was done 5 ... 10 us into the launch where every wave asked for weights first.
// As workgroups of four waves, up to four per CU and one CU with twice the items of another (us, before / now): k_ld_in of 2048
// columns in bf16, four sequences, 50 and 26 MB 20.8 / 16.3 and 13.9 / 11.5; in fp32, one sequence, 100 and 51 MB 21.9 / 19.1 and
// 17.5 / 11.9; 1024 columns, 10 and 6 MB 6.5 / 5.3 and 5.8 / 4.7.  k_ld_head, 131 MB: four sequences 35.2 / 28.6 (one
// in fp32, 262 MB: 42.8 / 44.4).
// (Four rows of more than 4096 columns, NV = 4: eight waves; sixteen would have too few registers.)
constexpr int kLdNorm = 512;
constexpr int ld_in_wg(int B, int NV) { return B * NV >= 16 ? kLdNorm : 1024; }
// blocks of a tile: 128 registers a wave hold them beside the rows (more than 4096 columns: NV = 4).  One vector: all of a row of
// 2048 at once, a launch of two items a CU is one round trip (k_ld_in of 1024 columns in fp32, 6 and 10 MB: 6.9 and 7.2 us with
// two, 4.7 and 5.3 with four).
constexpr int ld_in_tile(int B, int NV) { return B == 1 && NV < 4 ? 4 : 2; }
template <class T, int B, int NV>
__global__ __launch_bounds__(ld_in_wg(B, NV)) void k_ld_in(const LdInArgs a) {
  constexpr int R = 4, U = ld_in_tile(B, NV), NT = kLdNorm, NW = ld_in_wg(B, NV) / 64;
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  float* xs = (float*)smem_raw;
  __shared__ float red[64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wg = blockIdx.x;
  int si = 0;
  if (a.nseg > 1 && wg >= a.seg[1].wg0) si = 1;
  if (a.nseg > 2 && wg >= a.seg[2].wg0) si = 2;
  // values, not references: a selected address of a kernel argument would force the arguments into scratch memory
  const T* w = (const T*)(si == 0 ? a.seg[0].w : si == 1 ? a.seg[1].w : a.seg[2].w);
  float* out = si == 0 ? a.seg[0].out : si == 1 ? a.seg[1].out : a.seg[2].out;
  const int rows = si == 0 ? a.seg[0].rows : si == 1 ? a.seg[1].rows : a.seg[2].rows;
  const int ldo = si == 0 ? a.seg[0].ldo : si == 1 ? a.seg[1].ldo : a.seg[2].ldo;
  const int kind = si == 0 ? a.seg[0].kind : si == 1 ? a.seg[1].kind : a.seg[2].kind;
  const int norm2 = si == 0 ? a.seg[0].norm2 : si == 1 ? a.seg[1].norm2 : a.seg[2].norm2;
  const int wg0 = si == 0 ? a.seg[0].wg0 : si == 1 ? a.seg[1].wg0 : a.seg[2].wg0;
  const int nwg = si == 0 ? a.seg[0].nwg : si == 1 ? a.seg[1].nwg : a.seg[2].nwg;
  const float* bias = si == 0 ? a.seg[0].bias : si == 1 ? a.seg[1].bias : a.seg[2].bias;
  const int nblk = Ld<T>::blocks(a.ld), nch = a.ld / Ld<T>::E;
  const int per = kind == LDI_GATED ? R / 2 : R;  // outputs per item
  const int items = (rows + per - 1) / per;
  // dealt over the workgroups in turn: every CU draws the same number of them, give or take one; first those of the waves that
  // do not norm
  const int item = ((wave + NW / 2) % NW) * nwg + (wg - wg0), step = NW * nwg;
  auto set_rows = [&](int it, const T* (&row)[R]) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      int i;
      if (kind == LDI_GATED) {
        int j = it * 2 + (r & 1);
        j = j < rows ? j : rows - 1;
        i = (j >> 4) * 32 + (j & 15) + (r >> 1) * 16;
      } else {
        i = it * R + r;
        i = i < rows ? i : rows - 1;
      }
      row[r] = w + (size_t)i * a.ld;
    }
  };
  // ---- the rows
  constexpr int Q = ld_rows_at_once(B, NV);
  const int xstride = nblk * Ld<T>::BE, n4 = a.ld >> 2, total4 = xstride >> 2;
  f32x4 nw[NV], nb[NV], v[Q][NV];
  float shift[Q];
  auto get = [&](int q, f32x4 (&x)[NV], float& sh) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int i = threadIdx.x + NT * j;
      x[j] = f4_zero();
      if (i < n4) {
        x[j] = a.from_embed ? ld_embed<T>(a.emb, a.t.tok[q], a.t.pos[q], a.ld, i) : ((const f32x4*)(a.x_in + (size_t)q * a.ld))[i];
        if (a.add_x0) x[j] += ld_embed<T>(a.emb, a.t.tok[q], a.t.pos[q], a.ld, i);
        if (a.step) x[j] += ((const f32x4*)a.step)[i];
      }
    }
    sh = 0.f;
    if (!a.rms) sh = a.from_embed ? (float)((const T*)a.emb.embed)[(size_t)a.t.tok[q] * a.ld] : a.x_in[(size_t)q * a.ld];
  };
  auto weights = [&]() __attribute__((always_inline)) {
    const f32x4 *wp = (const f32x4*)(norm2 ? a.w2 : a.w1), *bp = (const f32x4*)(norm2 ? a.b2 : a.b1);
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int i = threadIdx.x + NT * j;
      nw[j] = i < n4 ? wp[i] : f4_zero();
      nb[j] = bp && i < n4 ? bp[i] : f4_zero();
    }
  };
  const bool norms = wave < NT / 64;
  if (norms && Q == B) {
#pragma unroll
    for (int q = 0; q < Q; ++q) get(q, v[q], shift[q]);
    weights();
  }
  LdTile<T, R, U> t;
  if (!norms) ld_items_begin(t, item, items, nblk, nch, lane, set_rows);
  // ---- layer norm of B rows
#pragma unroll 1
  for (int q0 = 0; q0 < B; q0 += Q) {
    if (Q < B) {
      if (norms) {
        get(q0, v[0], shift[0]);  // Q = 1
        __builtin_amdgcn_sched_barrier(0);
        weights();  // behind what get() adds up: the registers do not hold both
      }
      if (q0) __syncthreads();  // red is free again
    }
    if (a.x_cur && wg == 0 && norms) {
#pragma unroll
      for (int q = 0; q < Q; ++q)
#pragma unroll
        for (int j = 0; j < NV; ++j)
          if ((int)threadIdx.x + NT * j < n4) ((f32x4*)(a.x_cur + (size_t)(q0 + q) * a.ld))[threadIdx.x + NT * j] = v[q][j];
    }
    // the router's first workgroup leaves the second norm for the launches that follow
    f32x4* keep = a.xn2 && wg == a.xn2_wg ? (f32x4*)(a.xn2 + (size_t)q0 * a.ld) : nullptr;
    int W = a.W, m4 = n4, t4 = total4;
    if (Q < B) asm volatile("" : "+s"(W), "+s"(m4), "+s"(t4));  // or the lane masks of all pieces are kept over the rows: scratch
    ld_norm<T, NT, NV, Q>(v, nw, nb, shift, a.rms, W, m4, t4, a.eps, red, (f32x4*)(xs + (size_t)q0 * xstride), total4, keep, n4);
  }
  if (norms) ld_items_begin(t, item, items, nblk, nch, lane, set_rows);
  __syncthreads();
  // the owner of sum (r, q) finishes output r of sequence q: operands of a convolution of up to CT taps are requested early
  constexpr int CT = 4;
  const LdOwn own = ld_own<R, B>(lane);
  const int lr = own.r, lq = own.q;
  const bool conv_pre = kind == LDI_CONV && a.taps <= CT;
  float cw[CT], cs[CT], cb = 0.f, bi = 0.f;
  bool fresh = false;
  float* st0 = nullptr;
  if (kind == LDI_CONV && own.on) {
    fresh = a.t.pos[lq] == 0;
    st0 = a.conv_st + (size_t)a.t.slot[lq] * a.slot_stride;
  }
  auto early = [&](int it) __attribute__((always_inline)) {
    if (!own.on) return;
    const int i = it * R + lr;
    if (bias) bi = bias[i < rows ? i : rows - 1];
    if (conv_pre && i < a.inner) {
      cb = a.conv_b[i];
#pragma unroll
      for (int k = 0; k < CT; ++k) {
        cw[k] = k < a.taps ? a.conv_w[(size_t)i * a.taps + k] : 0.f;
        cs[k] = k + 1 < a.taps && !fresh ? st0[(size_t)k * a.inner + i] : 0.f;
      }
    }
  };
  auto done = [&](int it, float v) __attribute__((always_inline)) {
    if (kind == LDI_GATED) {
      float g, u;
      ld_gate_up(v, g, u);
      const int j = it * 2 + lr;
      if (own.on && lr < 2 && j < rows) out[(size_t)lq * ldo + j] = gated1(a.act, g, u);
      return;
    }
    const int i = it * R + lr;
    if (!own.on || i >= rows) return;
    if (kind != LDI_CONV || i >= a.inner) {
      out[(size_t)lq * ldo + i] = v + bi;
      return;
    }
    float* st = st0 + i;
    float c;
    if (conv_pre) {
      c = cb;
#pragma unroll
      for (int k = 0; k < CT; ++k) {
        if (k + 1 < a.taps) {
          c = __builtin_fmaf(cw[k], cs[k], c);
          if (k) st[(size_t)(k - 1) * a.inner] = cs[k];
        } else if (k + 1 == a.taps) {
          c = __builtin_fmaf(cw[k], v, c);
        }
      }
    } else {
      const float* w1 = a.conv_w + (size_t)i * a.taps;
      c = a.conv_b[i];
      for (int k = 0; k + 1 < a.taps; ++k) {
        const float in = fresh ? 0.f : st[(size_t)k * a.inner];
        c = __builtin_fmaf(w1[k], in, c);
        if (k) st[(size_t)(k - 1) * a.inner] = in;
      }
      c = __builtin_fmaf(w1[a.taps - 1], v, c);
    }
    if (a.taps > 1) st[(size_t)(a.taps - 2) * a.inner] = v;
    a.xc[(size_t)lq * a.xc_ld + i] = silu1(c);
  };
  ld_items<B>(t, item, step, items, nblk, nch, xs, xstride, lane, set_rows, early, done);
}

// ---- k_ld_mid ----------------------------------------------------------------------------------------------------
struct LdMidArgs {
  // experts: workgroups [0, B top nwg_e), behind those of attention over heads
  const float* z;        // [B][ldz]
  const float *corr, *xn2;
  const void* gu;        // experts [2 ffp][ldw]
  float* he;             // [B][top][ffp], weighted
  int32_t* ids;          // [B][top] (-1: identity), written for k_ld_out
  float *id_w, *sh_g;    // [B]
  int nwg_e, top, n_out, n_expert, shared, ffp, ldz, W, ldw, over_chosen;
  GateAct act;
  // mixer: workgroups [.., + nwg_m)
  const void* wm;        // rows x ld
  const float* v;        // [B][ldv] input vectors (n valid entries)
  const float* vnorm;    // RMS norm weight (nullptr: none)
  float* om;             // [B][ldo]
  int nwg_m, rows, ldm, n, n4, ldv, ldo;  // n4: float4 of a row that may be read (no norm)
  // cache rows: the last workgroups (latent attention: one per sequence; heads: one wave per key / value head)
  int latent;
  HeadRow hr;
  LdHeads att;           // attention over heads: the first workgroups (none: it has launches of its own)
  const float* raw;      // [B][ldv]: q latent, kv latent, rotated part
  const float* kvn;
  const float2* rope;
  void* cache;
  size_t slot_elems;
  int qr, R, dr, Rp, row, dims;
  float eps;
  LdTabs t;
};
// Steps of B sequences: are the experts that several of them chose read once (k_ld_mid<.., SHARE>)?  That takes the LDS of B
// vectors and a barrier in front of the first weight, so it has to save something: with even routing, one choice in sixteen is
// also an earlier sequence's.  us a step of four mamba layers of 1024 columns with few choices alike, each sequence's own / read
// once, two and four sequences: 4 of 128 132 / 140 and 168 / 175, 8 of 256 148 / 151 and 195 / 199, 8 of 512 with 128 columns
// 141 / 147 and 177 / 187; with many (6 of 36 outputs) see k_ld_mid.
static inline bool ld_shares(int B, int top, int n_out) {
  const double p = (double)top / n_out;
  double none = 1.0;  // that no one of B chose an expert
  for (int q = 0; q < B; ++q) none *= 1.0 - p;
  return 1.0 - (1.0 - none) / (B * p) >= 1.0 / 16;
}
// HEADS: the layer's mixer is attention over heads (its workgroups' registers, 151 in bf16 and 175 in fp32, would take a fourth
// workgroup per CU from the other mixers')
template <class T, int B, int NV, int RP, bool SHARE, bool HEADS>
__global__ __launch_bounds__(256, B > 1 && sizeof(T) == 2 ? 3 : 1) void k_ld_mid(const LdMidArgs a) {
  constexpr int R = 4, U = B > 1 ? 2 : 4, SB = SHARE ? B : 1;  // (three blocks spill, and so do four workgroups per CU: 35 and 40 us for 30.5)
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  float* xs = (float*)smem_raw;
  __shared__ float red[KH_WAVES_MAX];
  __shared__ int32_t rid[SB][KH_MOE_MAX_TOP];
  __shared__ float rwt[SB][KH_MOE_MAX_TOP];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int wg = blockIdx.x;
  if constexpr (HEADS) {
    if (wg < a.att.nwg) {  // ---- attention over heads, a chain of round trips: in front
      ld_heads<T>(a.att, a.hr, a.raw, a.ldv, (const T*)a.cache, a.slot_elems, a.t.pos, a.t.slot, wg, smem_raw);
      return;
    }
    wg -= a.att.nwg;
  }
  LdTile<T, R, U> t;
  const T* row[R];
  const int ne = B * a.top * a.nwg_e;
  if (wg < ne) {  // ---- one chosen expert of one sequence (SHARE: and of those behind it that chose it too)
    const int pair = wg / a.nwg_e, part = wg - pair * a.nwg_e, q = pair / a.top, k = pair - q * a.top;
    const int nblk = Ld<T>::blocks(a.ldw), nch = a.ldw / Ld<T>::E;
    const int n4 = a.ldw >> 2, total4 = nblk * Ld<T>::BE / 4;
    f32x4 x[NV];  // requested first: in flight while the choice is made
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int i = threadIdx.x + 256 * j;
      x[j] = i < n4 ? ((const f32x4*)(a.xn2 + (size_t)q * a.ldw))[i] : f4_zero();
    }
    // Every wave makes the choice for itself: its weight loads leave without a barrier.  SHARE: the waves make one sequence's
    // each, and an expert that several chose is read once, by the first of them.  Bound by the bytes of the experts (2048 x
    // 1024 in bf16, four sequences, 6 of 32 and 4 identities each: 21 choices of 17 experts): 39.4 -> 35.5 us in front of latent
    // attention, 31.6 -> 28.3 of mamba; with tiles of two blocks, three workgroups per CU instead of two and no second round of
    // them, 30.5 and 26.4.  k_ld_out does not do so: there a sequence's sum would be taken in an order that depends on what the
    // others chose.
    float idw = 0.f, w = 0.f;
    int id = -1;
    unsigned mates = 0;  // byte q: 1 + the place where later sequence q chose the same expert
    if constexpr (SHARE) {
      const int qw = wave % B;
      int my_id = 0;
      float my_w = 0.f;
      const float wf = moe_route<RP>(a.z + (size_t)qw * a.ldz, a.corr, a.n_out, a.top, a.over_chosen, lane,
                                     [&](int kk, int i, float wt) __attribute__((always_inline)) {
        if (i >= a.n_expert) idw += wt;
        my_id = lane == kk ? (i >= a.n_expert ? -1 : i) : my_id;
        my_w = lane == kk ? wt : my_w;
      });
      if (lane < a.top) {
        rid[qw][lane] = my_id;
        rwt[qw][lane] = my_w * wf;
      }
      if (part == 0 && k == 0 && wave == q && lane == 0) {
        a.id_w[q] = idw * wf;
        if (a.shared) a.sh_g[q] = sigmoid1(a.z[(size_t)q * a.ldz + a.n_out]);
      }
      __syncthreads();
      id = rid[q][k];
      bool first = id >= 0;
#pragma unroll
      for (int o = 0; o < B; ++o) {
        const unsigned long long hit = __builtin_amdgcn_ballot_w64(lane < a.top && rid[o][lane < a.top ? lane : 0] == id);
        if (o == q || !hit) continue;
        if (o < q) first = false;
        else mates |= (unsigned)(__builtin_ctzll(hit) + 1) << (8 * o);
      }
      if (part == 0 && threadIdx.x == 0) a.ids[q * a.top + k] = id;
      if (!first) return;  // the whole workgroup agrees
      id = __builtin_amdgcn_readfirstlane(id);
      mates = (unsigned)__builtin_amdgcn_readfirstlane((int)mates);
      w = rwt[q][k];
    } else {
      const float wf = moe_route<RP>(a.z + (size_t)q * a.ldz, a.corr, a.n_out, a.top, a.over_chosen, lane,
                                     [&](int kk, int i, float wt) __attribute__((always_inline)) {
        const bool ident = i >= a.n_expert;
        if (ident) idw += wt;
        if (kk == k) {
          id = ident ? -1 : i;
          w = wt;
        }
      });
      w *= wf;
      idw *= wf;
      if (part == 0 && threadIdx.x == 0) {
        a.ids[q * a.top + k] = id;
        if (k == 0) {
          a.id_w[q] = idw;
          if (a.shared) a.sh_g[q] = sigmoid1(a.z[(size_t)q * a.ldz + a.n_out]);
        }
      }
      if (id < 0) return;  // identity expert: no tensors (the whole workgroup agrees)
    }
    const T* base = (const T*)a.gu + (size_t)id * 2 * a.ffp * a.ldw;
    const int items = a.ffp / 2;
    int it = part * 4 + wave;
    auto set_rows = [&](int i) __attribute__((always_inline)) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int j = i * 2 + (r & 1);
        row[r] = base + (size_t)((j >> 4) * 32 + (j & 15) + (r >> 1) * 16) * a.ldw;
      }
    };
    if (it < items) {
      set_rows(it);
      ld_load<T, R, U>(t, row, 0, nblk, nch, lane);
    }
#pragma unroll
    for (int j = 0; j < NV; ++j)
      if ((int)threadIdx.x + 256 * j < total4) ((f32x4*)xs)[ld_slot<T>(threadIdx.x + 256 * j)] = x[j];
    // vector j > 0: the j-th of the mates, in rising order of their sequences
    int n = 1, dst[SB];
    float wj[SB];
    dst[0] = pair;
    wj[0] = w;
    if constexpr (SHARE) {
#pragma unroll
      for (int j = 1; j < B; ++j) {
        dst[j] = pair;
        wj[j] = 0.f;
      }
#pragma unroll
      for (int o = 1; o < B; ++o) {
        const int ko = (int)(mates >> (8 * o) & 255) - 1;
        if (ko < 0) continue;  // uniform
        f32x4* xo = (f32x4*)xs + (size_t)n * total4;
#pragma unroll
        for (int j = 0; j < NV; ++j) {
          const int i = threadIdx.x + 256 * j;
          if (i < total4) xo[ld_slot<T>(i)] = i < n4 ? ((const f32x4*)(a.xn2 + (size_t)o * a.ldw))[i] : f4_zero();
        }
#pragma unroll
        for (int j = 1; j < B; ++j)
          if (j == n) {
            dst[j] = o * a.top + ko;
            wj[j] = rwt[o][ko];
          }
        ++n;
      }
    }
    __syncthreads();
    auto rows_of = [&](auto cnt) __attribute__((always_inline)) {
      constexpr int N = decltype(cnt)::value;
      while (it < items) {
        float acc[R][N] = {};
        ld_rows<T, R, U, N>(t, row, nblk, nch, xs, total4 * 4, lane, acc);
        const int cur = it;
        it += a.nwg_e * 4;
        if (it < items) {
          set_rows(it);
          ld_load<T, R, U>(t, row, 0, nblk, nch, lane);
        }
        float g, u;
        ld_gate_up(ld_sums(acc, lane), g, u);
        const LdOwn own = ld_own<R, N>(lane);
        if (own.on && own.r < 2 && own.q < n) {
          int d = dst[0];
          float wt = wj[0];
#pragma unroll
          for (int j = 1; j < N; ++j) {
            d = own.q == j ? dst[j] : d;
            wt = own.q == j ? wj[j] : wt;
          }
          a.he[(size_t)d * a.ffp + cur * 2 + own.r] = wt * gated1(a.act, g, u);
        }
      }
    };
    if (n == 1) rows_of(std::integral_constant<int, 1>());
    else if (SB == 2 || n == 2) rows_of(std::integral_constant<int, SB < 2 ? 1 : 2>());
    else rows_of(std::integral_constant<int, SB>());  // three of four: what the fourth place holds is finite or not, and not stored
    return;
  }
  wg -= ne;
  if constexpr (HEADS) {  // ---- cache rows
    const int i = wg * 4 + wave, q = i / a.hr.G, g = i - q * a.hr.G;
    if (q < B)
      heads_cache_row(a.hr, a.raw + (size_t)q * a.ldv, (T*)a.cache + (size_t)a.t.slot[q] * a.slot_elems, a.t.pos[q], g, lane);
    return;
  }
  if (wg < a.nwg_m) {  // ---- the mixer's second projection
    const int nblk = Ld<T>::blocks(a.ldm), nch = a.ldm / Ld<T>::E, xstride = nblk * Ld<T>::BE;
    const int items = (a.rows + R - 1) / R;
    int item = wg * 4 + wave;
    auto set_rows = [&](int it) __attribute__((always_inline)) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        int i = it * R + r;
        i = i < a.rows ? i : a.rows - 1;
        row[r] = (const T*)a.wm + (size_t)i * a.ldm;
      }
    };
    if (item < items) {
      set_rows(item);
      ld_load<T, R, U>(t, row, 0, nblk, nch, lane);
    }
    for (int q = 0; q < B; ++q) {
      const float* v = a.v + (size_t)q * a.ldv;
      f32x4* x4 = (f32x4*)(xs + (size_t)q * xstride);
      if (!a.vnorm) {
        ld_stage<T, 256>(x4, v, a.n4, xstride >> 2, 1.f, threadIdx.x);
      } else {
        float s = 0.f;
        for (int i = threadIdx.x; i < a.n; i += 256) s = __builtin_fmaf(v[i], v[i], s);
        const float rs = 1.0f / sqrtf(block_sum(s, red) / (float)a.n + a.eps);
        for (int i = threadIdx.x; i < xstride; i += 256)
          xs[(size_t)q * xstride + Ld<T>::place(i)] = i < a.n ? v[i] * rs * a.vnorm[i] : 0.f;
      }
    }
    __syncthreads();
    while (item < items) {
      float acc[R][B] = {};
      ld_rows<T, R, U, B>(t, row, nblk, nch, xs, xstride, lane, acc);
      const int cur = item;
      item += a.nwg_m * 4;
      if (item < items) {
        set_rows(item);
        ld_load<T, R, U>(t, row, 0, nblk, nch, lane);
      }
      const float v = ld_sums(acc, lane);
      const LdOwn own = ld_own<R, B>(lane);
      const int i = cur * R + own.r;
      if (own.on && i < a.rows) a.om[(size_t)own.q * a.ldo + i] = v;
    }
    return;
  }
  wg -= a.nwg_m;
  if (!a.latent || wg >= B) return;  // ---- cache row of sequence wg
  const float* rr = a.raw + (size_t)wg * a.ldv + a.qr;
  const int pos = a.t.pos[wg];
  float s = 0.f;
  for (int i = threadIdx.x; i < a.R; i += 256) s = __builtin_fmaf(rr[i], rr[i], s);
  const float rk = 1.0f / sqrtf(block_sum(s, red) / (float)a.R + a.eps);
  T* crow = (T*)a.cache + (size_t)a.t.slot[wg] * a.slot_elems + (size_t)pos * a.row;
  for (int i = threadIdx.x; i < a.row; i += 256) {
    float v = 0.f;
    if (i < a.R) {
      v = rr[i] * rk * a.kvn[i];
    } else if (i >= a.Rp && i - a.Rp < a.dr) {
      const int j = i - a.Rp;
      v = rr[a.R + j];
      if (j < a.dims) {
        const float2 cs = a.rope[(size_t)pos * (a.dims >> 1) + (j >> 1)];
        const float o = rr[a.R + (j ^ 1)];
        v = (j & 1) ? v * cs.x + o * cs.y : v * cs.x - o * cs.y;
      }
    }
    crow[i] = (T)v;
  }
}

// ---- k_ld_scan: 16 lanes per channel, 16 channels per workgroup.  grid (channels / 16, B) ----------------------------
struct LdScanArgs {
  const float *xc, *xz, *dbc;  // [B][xc_ld], [B][2 C] (z half), [B][rankp + 2 N]
  const void* wdt;             // [C][rankp]
  const float *dt_b, *A2, *D;
  float* state;
  float* y;                    // [B][y_ld]
  size_t slot_stride;
  int C, N, rankp, xc_ld, y_ld;
  LdTabs t;
};
template <class T, int NSL /* states per lane */>
__global__ __launch_bounds__(256) void k_ld_scan(const LdScanArgs a) {
  constexpr int E = Tile<T>::N;
  const int q = blockIdx.y, g = threadIdx.x & 15;
  const int c = blockIdx.x * 16 + ((int)threadIdx.x >> 4);
  const bool live = c < a.C;
  const int cc = live ? c : a.C - 1;
  const float* dbc = a.dbc + (size_t)q * (a.rankp + 2 * a.N);
  float* st = a.state + (size_t)a.t.slot[q] * a.slot_stride + (size_t)cc * a.N;
  const bool fresh = a.t.pos[q] == 0;
  float A2[NSL], S[NSL], Bn[NSL], Cn[NSL];
#pragma unroll
  for (int j = 0; j < NSL; ++j) {  // neighbouring lanes own neighbouring states
    const int n = j * 16 + g;
    const bool in = n < a.N;
    A2[j] = in ? a.A2[(size_t)cc * a.N + n] : 0.f;
    S[j] = in && !fresh ? st[n] : 0.f;
    Bn[j] = in ? dbc[a.rankp + n] : 0.f;
    Cn[j] = in ? dbc[a.rankp + a.N + n] : 0.f;
  }
  const float x = a.xc[(size_t)q * a.xc_ld + cc], z = a.xz[(size_t)q * 2 * a.C + a.C + cc];
  float s = 0.f;
  for (int k = g * E; k < a.rankp; k += 16 * E) {
    const typename Tile<T>::frag w = *(const typename Tile<T>::frag*)((const T*)a.wdt + (size_t)cc * a.rankp + k);
#pragma unroll
    for (int e = 0; e < E; ++e) s = __builtin_fmaf((float)w[e], dbc[k + e], s);
  }
  const float dt = softplus1(group_sum<16>(s) + a.dt_b[cc]), dx = dt * x;
  float y = 0.f;
#pragma unroll
  for (int j = 0; j < NSL; ++j) {
    const int n = j * 16 + g;
    S[j] = __builtin_fmaf(__builtin_amdgcn_exp2f(dt * A2[j]), S[j], dx * Bn[j]);
    y = __builtin_fmaf(S[j], Cn[j], y);
    if (live && n < a.N) st[n] = S[j];
  }
  y = group_sum<16>(y);
  if (g == 0 && live) a.y[(size_t)q * a.y_ld + c] = __builtin_fmaf(a.D[c], x, y) * silu1(z);
}

// ---- k_ld_absorb: Q row of every head: W_uk^T q_n and the rotated part.  grid (H nwg, B) ------------------------------
struct LdAbsorbArgs {
  const float* q;     // [B][H (dnp + drp)]
  const void* ukT;    // [H][Rp][dnp]
  const float2* rope;
  void* Q;            // T [B][H][row]
  int H, nwg, dnp, dr, drp, Rp, row, dims;
  LdTabs t;
};
template <class T>
__global__ __launch_bounds__(256) void k_ld_absorb(const LdAbsorbArgs a) {
  constexpr int E = Tile<T>::N;
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  float* v = (float*)smem_raw;  // [dnp]
  const int b = blockIdx.y, h = (int)blockIdx.x / a.nwg, part = (int)blockIdx.x - h * a.nwg;
  const float* q = a.q + ((size_t)b * a.H + h) * (a.dnp + a.drp);
  for (int i = threadIdx.x; i < a.dnp; i += 256) v[i] = q[i];
  T* Q = (T*)a.Q + ((size_t)b * a.H + h) * a.row;
  if (part == 0) {
    const int pos = a.t.pos[b];
    for (int j = threadIdx.x; j < a.drp; j += 256) {
      float r = j < a.dr ? q[a.dnp + j] : 0.f;
      if (j < a.dims) {
        const float2 cs = a.rope[(size_t)pos * (a.dims >> 1) + (j >> 1)];
        const float o = q[a.dnp + (j ^ 1)];
        r = (j & 1) ? r * cs.x + o * cs.y : r * cs.x - o * cs.y;
      }
      Q[a.Rp + j] = (T)r;
    }
  }
  __syncthreads();
  // eight lanes per row
  for (int i = part * 32 + ((int)threadIdx.x >> 3); i < a.Rp; i += a.nwg * 32) {
    const T* w = (const T*)a.ukT + ((size_t)h * a.Rp + i) * a.dnp;
    float s = 0.f;
    for (int k = (threadIdx.x & 7) * E; k < a.dnp; k += 8 * E) {
      const typename Tile<T>::frag f = *(const typename Tile<T>::frag*)(w + k);
#pragma unroll
      for (int e = 0; e < E; ++e) s = __builtin_fmaf((float)f[e], v[k + e], s);
    }
    s = group_sum<8>(s);
    if ((threadIdx.x & 7) == 0) Q[i] = (T)s;
  }
}

// Merge of the time splits of one head: p [splits][C + 4] (C columns, running maximum, sum); its ns filled splits meet in
// sum [256 / (C / 4) groups][C / 4], summed over the groups by the caller.  Returns 1 / sum of the weights and, in grp, the
// number of groups.  fac: one factor per split, ns <= 256
__device__ __forceinline__ float ld_merge_splits(const float* p, int ns, int C, float* fac, float* red, f32x4* sum, int& grp) {
  // column groups of four; 256 / (C / 4) thread groups share the splits and meet in LDS
  const int c4 = C >> 2, g = (int)threadIdx.x / c4, lane = threadIdx.x & 63;
  grp = c4 < 256 ? 256 / c4 : 1;
  const int ahead = g < grp ? grp : 0;
  constexpr int U = 8;
  f32x4 x[U];
  const int i0 = (int)threadIdx.x - g * c4;
  auto request = [&](int i, int s) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < U; ++j) {
      const int k = s + j * grp;
      x[j] = *(const f32x4*)(p + (size_t)(k < ns ? k : ns - 1) * (C + 4) + 4 * i);
    }
  };
  float l;
  const float* f;
  if (ns <= 64) {  // uniform: every wave has all maxima and sums in its lanes, and no barrier before the columns
    if (ahead) request(i0, g);
    float mk = -INFINITY, lk = 0.f;
    if (lane < ns) {
      const float2 ml = *(const float2*)(p + (size_t)lane * (C + 4) + C);
      mk = ml.x;
      lk = ml.y;
    }
    const float m = wave_max(mk);
    const float fk = lane < ns ? __builtin_amdgcn_exp2f(mk - m) : 0.f;  // an empty split: exp2(-inf) = 0
    l = wave_sum(fk * lk);
    float* own = fac + (threadIdx.x & ~63u);
    own[lane] = fk;
    f = own;
  } else {
    float m = -INFINITY;
    for (int s = threadIdx.x; s < ns; s += 256) m = fmaxf(m, p[(size_t)s * (C + 4) + C]);
    m = block_max(m, red);
    l = 0.f;
    for (int s = threadIdx.x; s < ns; s += 256) {
      const float* ps = p + (size_t)s * (C + 4) + C;
      const float fs = __builtin_amdgcn_exp2f(ps[0] - m);
      fac[s] = fs;
      l = __builtin_fmaf(fs, ps[1], l);
    }
    l = block_sum(l, red);
    f = fac;
    if (ahead) request(i0, g);
  }
  if (ahead) {
    for (int i = i0; i < c4; i += 256) {
      if (i != i0) request(i, g);
      f32x4 v = f4_zero();
      for (int s = g; s < ns; s += U * grp) {
        if (s != g) request(i, s);
#pragma unroll
        for (int j = 0; j < U; ++j)
          if (s + j * grp < ns) v = fma_s(f[s + j * grp], x[j], v);
      }
      sum[g * c4 + i] = v;
    }
  }
  __syncthreads();
  return 1.0f / l;
}

// ---- k_ld_values: merge of the time splits, then W_uv of the head.  grid (H nwg, B) ----------------------------------
// A chain of trips (position; maxima, sums and columns of the splits; W_uv beside them), so a head is cut until the launch has 256
// workgroups or a wave one group of rows: 4 x 16 heads of 128 over 512 latents and 10 splits 7.2 us with the maxima and sums behind
// barriers of their own in front of the columns, 6.9 with both at once, 5.5 with 256 workgroups instead of 128.
struct LdValuesArgs {
  const float* part;  // [B H][nsplit][Rp + 4]
  const void* uv;     // [H][dvp][Rp]
  float* o;           // [B][H dvp]
  int H, nwg, nsplit, Rp, dvp;
  const int32_t* pos;
};
template <class T>
__global__ __launch_bounds__(256) void k_ld_values(const LdValuesArgs a) {
  constexpr int R = 4, U = 1;
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  float* xs = (float*)smem_raw;
  __shared__ float fac[256];
  __shared__ float red[KH_WAVES_MAX];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int b = blockIdx.y, h = (int)blockIdx.x / a.nwg, part = (int)blockIdx.x - h * a.nwg;
  const float* p = a.part + ((size_t)b * a.H + h) * a.nsplit * (size_t)(a.Rp + 4);
  const int nblk = Ld<T>::blocks(a.Rp), nch = a.Rp / Ld<T>::E;
  const int items = a.dvp / R;
  int item = part * 4 + wave;
  const T* row[R];
  LdTile<T, R, U> t;
  auto set_rows = [&](int it) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < R; ++r) row[r] = (const T*)a.uv + ((size_t)h * a.dvp + it * R + r) * a.Rp;
  };
  if (item < items) {
    set_rows(item);
    ld_load<T, R, U>(t, row, 0, nblk, nch, lane);
  }
  const int c4 = a.Rp >> 2;
  f32x4* sum = (f32x4*)(xs + (size_t)nblk * Ld<T>::BE);  // [grp][c4]
  int grp;
  const float inv = ld_merge_splits(p, lat_active_splits(a.pos[b] + 1, a.nsplit, LatCfg<T>::KT), a.Rp, fac, red, sum, grp);
  for (int i = threadIdx.x; i < nblk * Ld<T>::BE / 4; i += 256) {
    f32x4 v = f4_zero();
    if (i < c4)
      for (int k = 0; k < grp; ++k) v += sum[k * c4 + i];
    ((f32x4*)xs)[ld_slot<T>(i)] = v * inv;
  }
  __syncthreads();
  while (item < items) {
    float acc[R][1] = {};
    ld_rows<T, R, U, 1>(t, row, nblk, nch, xs, 0, lane, acc);
    const int cur = item;
    item += a.nwg * 4;
    if (item < items) {
      set_rows(item);
      ld_load<T, R, U>(t, row, 0, nblk, nch, lane);
    }
    const float v = ld_sums(acc, lane);
    const LdOwn own = ld_own<R, 1>(lane);
    if (own.on) a.o[((size_t)b * a.H + h) * a.dvp + cur * R + own.r] = v;
  }
}

// ---- k_ld_merge: attention over heads: merge of the time splits, output gate.  grid (H, B) --------------------------
struct LdMergeArgs {
  const float* part;  // [B H][nsplit][C + 4]
  const float* gate;  // [B][ldg]: logits head by head, gs apart (nullptr: none)
  float* o;           // [B][ldo], heads gs apart
  int H, nsplit, C, gs, ldg, ldo;
  KeySpan span;
  const int32_t* pos;
};
static __global__ __launch_bounds__(256) void k_ld_merge(const LdMergeArgs a) {
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  f32x4* sum = (f32x4*)smem_raw;
  __shared__ float fac[256];
  __shared__ float red[KH_WAVES_MAX];
  const int b = blockIdx.y, h = blockIdx.x, pos = a.pos[b], i = (int)threadIdx.x, c4 = a.C >> 2;
  f32x4 g = f4_zero();
  const bool live = 4 * i < a.gs;
  if (a.gate && live) g = *(const f32x4*)(a.gate + (size_t)b * a.ldg + (size_t)h * a.gs + 4 * i);
  int grp;
  const float inv = ld_merge_splits(a.part + ((size_t)b * a.H + h) * a.nsplit * (size_t)(a.C + 4),
                                    lat_active_splits(pos + 1 - a.span.first(pos), a.nsplit), a.C, fac, red, sum, grp);
  if (!live) return;
  f32x4 v = f4_zero();
  for (int k = 0; k < grp; ++k) v += sum[k * c4 + i];
#pragma unroll
  for (int j = 0; j < 4; ++j) v[j] *= a.gate ? inv * sigmoid1(g[j]) : inv;
  *(f32x4*)(a.o + (size_t)b * a.ldo + (size_t)h * a.gs + 4 * i) = v;
}

// ---- k_ld_enter: x_out = W [x ; embedding output], a pass of a loop that enters through a matrix --------------------
struct LdEnterArgs {
  const void* w;      // [W][2 ld]
  const float* x;     // [B][ld] (nullptr: the embedding output itself)
  float* x_out;       // [B][ld]
  LdEmbed emb;
  int W, ld, ks;
  LdTabs t;
};
// Workgroup = 8 waves = 8 / ks groups of ks waves; a group owns R rows, its waves share the blocks.
template <class T, int B>
__global__ __launch_bounds__(512) void k_ld_enter(const LdEnterArgs a) {
  constexpr int R = 2, U = 4, BE = Ld<T>::BE;
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  float* xs = (float*)smem_raw;
  __shared__ float comb[8][R * B];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int K = 2 * a.ld, nblk = Ld<T>::blocks(K), nch = K / Ld<T>::E, n4 = a.ld >> 2;
  const int kp = wave % a.ks, item = ((int)blockIdx.x * (8 / a.ks) + wave / a.ks) * R;
  const int per = (nblk + a.ks - 1) / a.ks, b0 = kp * per, b1 = b0 + per < nblk ? b0 + per : nblk;
  const T* row[R];
#pragma unroll
  for (int r = 0; r < R; ++r) row[r] = (const T*)a.w + (size_t)(item + r < a.W ? item + r : a.W - 1) * K;
  LdTile<T, R, U> t;
  ld_load<T, R, U>(t, row, b0, b1, nch, lane);
  for (int q = 0; q < B; ++q) {
    f32x4* xq = (f32x4*)(xs + (size_t)q * nblk * BE);
    for (int i = threadIdx.x; i < nblk * BE / 4; i += 512) {
      f32x4 v = f4_zero();
      if (i < n4 && a.x) v = ((const f32x4*)(a.x + (size_t)q * a.ld))[i];
      else if (i < 2 * n4) v = ld_embed<T>(a.emb, a.t.tok[q], a.t.pos[q], a.ld, i < n4 ? i : i - n4);
      xq[ld_slot<T>(i)] = v;
    }
  }
  __syncthreads();
  float acc[R][B] = {};
  for (int b = b0; b < b1; b += U) {
    if (b != b0) ld_load<T, R, U>(t, row, b, b1, nch, lane);
    ld_fma<T, R, U, B>(t, xs, nblk * BE, b, b1, lane, acc);
  }
  {
    const float v = ld_sums(acc, lane);
    const LdOwn own = ld_own<R, B>(lane);
    if (own.on) comb[wave][own.n] = v;
  }
  __syncthreads();
  if (kp == 0 && lane < R * B) {
    float v = 0.f;
    for (int k = 0; k < a.ks; ++k) v += comb[wave + k][lane];
    const int q = lane / R, i = item + (lane & (R - 1));
    if (i < a.W) a.x_out[(size_t)q * a.ld + i] = v;
  }
}

// ---- k_ld_out ----------------------------------------------------------------------------------------------------
struct LdOutArgs {
  const void* wo;         // [W][ldv]
  const float* v;         // [B][ld_v] mixer vector
  const void *down, *sdown;  // experts [W][ffp] each; shared [W][sffp]
  const float *he, *hs;   // [B][top][ffp] (weighted), [B][sffp]
  const int32_t* ids;     // [B][top]
  const float *id_w, *sh_g, *xn2, *x_cur;  // id_w, sh_g: nullptr = none, 1
  const float* bias;      // of W_o, or nullptr
  float* x_out;           // [B][ld]
  int W, ld, ld_v, ldv, top, ffp, sffp, moe, ks;
  float mult;             // of everything that is added to the residual
};
// Workgroup = 8 waves = 8 / ks groups of ks waves; a group owns R rows, its waves share the blocks: first those that all
// sequences share (mixer, shared expert: a weight block meets B vectors), then every sequence's experts.  The vectors come
// from the caches as they are needed, lanes behind a row's end repeat its last chunk against zeros: no LDS but the final sum,
// no barrier before it, and 16 waves a CU run freely.  Bound by latency: with the vectors staged in LDS, four sequences of
// 2048 columns took 96 KB (8 waves a CU, two rounds of workgroups) and a load, a staging and two barriers per sequence:
// 44.9 -> 26.3 us a layer at four (bf16, 105 ... 139 MB of weights), 8.0 -> 6.1 at one of 1024 (fp32).  Four rows a wave: with
// two, the vectors were half of what a CU draws through its L1 (31 ... 40 bytes a ns): 26.2 -> 20.9 us at four sequences, 15.7 ->
// 13.9 at two, 9.7 -> 8.8 at four of 1024, 5.96 -> 5.62 at one of 1024 in fp32; with eight, the waves are too few: 22.6, 13.3, 12.0.
constexpr int kLdOutRows = 4;
template <class T, int B>
__global__ __launch_bounds__(512, 4) void k_ld_out(const LdOutArgs a) {
  constexpr int R = kLdOutRows, U = 2;
  typedef typename Tile<T>::frag frag;
  constexpr int E = Ld<T>::E, P = Ld<T>::P;
  __shared__ float comb[8][R * B];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nbv = Ld<T>::blocks(a.ldv), nbs = a.moe && a.sffp ? Ld<T>::blocks(a.sffp) : 0, nbc = nbv + nbs;
  const int nbe = Ld<T>::blocks(a.ffp), per_q = a.moe ? a.top * nbe : 0;
  const int kp = wave % a.ks, grp = (int)blockIdx.x * (8 / a.ks) + wave / a.ks;
  const int item = grp * R;
  int ri[R];
#pragma unroll
  for (int r = 0; r < R; ++r) ri[r] = item + r < a.W ? item + r : a.W - 1;
  float acc[R][B] = {};
  float rx = 0.f, rn = 0.f, rw = 0.f, rb = 0.f;
  if (kp == 0 && lane < R * B) {
    const int q = lane / R, i = item + (lane & (R - 1));
    if (i < a.W) {
      rx = a.x_cur[(size_t)q * a.ld + i];
      if (a.bias) rb = a.bias[i];
      if (a.id_w) {
        rn = a.xn2[(size_t)q * a.ld + i];
        rw = a.id_w[q];
      }
    }
  }
  // chunk of the lane in block bb of a row of `n` elements
  auto chunk = [&](int n, int bb, bool& in) __attribute__((always_inline)) {
    const int left = n / E - bb * 64;
    in = lane < left;
    return bb * 64 + (in ? lane : left - 1);
  };
  auto dot = [&](const frag& w, const f32x4 (&x)[P], float s) __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < P; ++p)
#pragma unroll
      for (int i = 0; i < 4; ++i) s = __builtin_fmaf((float)w[4 * p + i], x[p][i], s);
    return s;
  };
  // ---- blocks that all sequences share
  {
    const int per = (nbc + a.ks - 1) / a.ks, u0 = kp * per, u1 = u0 + per < nbc ? u0 + per : nbc;
    for (int u = u0; u < u1; ++u) {
      const bool sh = u >= nbv;
      const int n = sh ? a.sffp : a.ldv, ldx = sh ? a.sffp : a.ld_v;
      const T* base = (const T*)(sh ? a.sdown : a.wo);
      const float* v = sh ? a.hs : a.v;
      bool in;
      const int c = chunk(n, sh ? u - nbv : u, in);
      frag w[R];
#pragma unroll
      for (int r = 0; r < R; ++r) w[r] = ld_nt((const frag*)(base + (size_t)ri[r] * n) + c);
      f32x4 x[B][P];
#pragma unroll
      for (int q = 0; q < B; ++q)
#pragma unroll
        for (int p = 0; p < P; ++p) x[q][p] = *(const f32x4*)(v + (size_t)q * ldx + (size_t)c * E + 4 * p);
#pragma unroll
      for (int q = 0; q < B; ++q) {
        const float g = sh && a.sh_g ? a.sh_g[q] : 1.f;
#pragma unroll
        for (int p = 0; p < P; ++p) x[q][p] = in ? x[q][p] * g : f4_zero();
#pragma unroll
        for (int r = 0; r < R; ++r) acc[r][q] = dot(w[r], x[q], acc[r][q]);
      }
    }
  }
  // ---- expert blocks, sequence by sequence
  if (per_q) {
    const int per = (per_q + a.ks - 1) / a.ks, e0 = kp * per, e1 = e0 + per < per_q ? e0 + per : per_q;
#pragma unroll
    for (int q = 0; q < B; ++q)
      for (int e = e0; e < e1; e += U) {
        frag w[R][U];
        f32x4 x[U][P];
        bool in[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          in[u] = false;
          if (e + u >= e1) continue;  // uniform
          const int k = (e + u) / nbe, id = a.ids[q * a.top + k];
          if (id < 0) continue;  // identity expert
          const int c = chunk(a.ffp, e + u - k * nbe, in[u]);
          const T* base = (const T*)a.down + (size_t)id * a.W * a.ffp;
#pragma unroll
          for (int r = 0; r < R; ++r) w[r][u] = ld_nt((const frag*)(base + (size_t)ri[r] * a.ffp) + c);
          const float* v = a.he + (size_t)(q * a.top + k) * a.ffp + (size_t)c * E;
#pragma unroll
          for (int p = 0; p < P; ++p) x[u][p] = *(const f32x4*)(v + 4 * p);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          if (e + u >= e1) continue;
          const int k = (e + u) / nbe;
          if (a.ids[q * a.top + k] < 0) continue;
#pragma unroll
          for (int p = 0; p < P; ++p) x[u][p] = in[u] ? x[u][p] : f4_zero();
#pragma unroll
          for (int r = 0; r < R; ++r) acc[r][q] = dot(w[r][u], x[u], acc[r][q]);
        }
      }
  }
  {
    const float v = ld_sums(acc, lane);
    const LdOwn own = ld_own<R, B>(lane);
    if (own.on) comb[wave][own.n] = v;
  }
  __syncthreads();
  if (kp == 0 && lane < R * B) {
    float v = 0.f;
    for (int k = 0; k < a.ks; ++k) v += comb[wave + k][lane];
    const int q = lane / R, i = item + (lane & (R - 1));
    if (i < a.W) a.x_out[(size_t)q * a.ld + i] = __builtin_fmaf(a.mult, __builtin_fmaf(rw, rn, v) + rb, rx);
  }
}

// ---- k_ld_head ---------------------------------------------------------------------------------------------------
struct LdHeadArgs {
  const float* x;        // [B][ld]
  const float *w, *b;    // final norm (rms: b may be nullptr)
  const void* head;      // [V][ld]
  float* logits;         // [B][V]
  float* part_val;       // argmax partials of sequence 0 (nullptr: none)
  int32_t* part_idx;
  int W, ld, V, rms;
  float eps, cap;
};
template <class T, int B, int NV>
__global__ __launch_bounds__(ld_in_wg(B, NV)) void k_ld_head(const LdHeadArgs a) {
  constexpr int R = 4, U = ld_in_tile(B, NV), NT = kLdNorm, NW = ld_in_wg(B, NV) / 64;
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  float* xs = (float*)smem_raw;
  __shared__ float red[64];
  __shared__ float sv[NW];
  __shared__ int si[NW];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nblk = Ld<T>::blocks(a.ld), nch = a.ld / Ld<T>::E, xstride = nblk * Ld<T>::BE;
  const int items = (a.V + R - 1) / R;
  const int item = ((wave + NW / 2) % NW) * (int)gridDim.x + (int)blockIdx.x, step = NW * (int)gridDim.x;  // as in k_ld_in
  auto set_rows = [&](int it, const T* (&row)[R]) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      int i = it * R + r;
      i = i < a.V ? i : a.V - 1;
      row[r] = (const T*)a.head + (size_t)i * a.ld;
    }
  };
  constexpr int Q = ld_rows_at_once(B, NV);
  const int n4 = a.ld >> 2;
  f32x4 nw[NV], nb[NV], v[Q][NV];
  float shift[Q];
  auto get = [&](int q, f32x4 (&x)[NV], float& sh) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int i = threadIdx.x + NT * j;
      x[j] = i < n4 ? ((const f32x4*)(a.x + (size_t)q * a.ld))[i] : f4_zero();
    }
    sh = a.rms ? 0.f : a.x[(size_t)q * a.ld];
  };
  const bool norms = wave < NT / 64;
  if (norms) {
    if (Q == B) {
#pragma unroll
      for (int q = 0; q < Q; ++q) get(q, v[q], shift[q]);
    }
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int i = threadIdx.x + NT * j;
      nw[j] = i < n4 ? ((const f32x4*)a.w)[i] : f4_zero();
      nb[j] = a.b && i < n4 ? ((const f32x4*)a.b)[i] : f4_zero();
    }
  }
  LdTile<T, R, U> t;
  if (!norms) ld_items_begin(t, item, items, nblk, nch, lane, set_rows);
#pragma unroll 1
  for (int q0 = 0; q0 < B; q0 += Q) {
    if (Q < B) {
      if (norms) get(q0, v[0], shift[0]);  // Q = 1
      if (q0) __syncthreads();             // red is free again
    }
    ld_norm<T, NT, NV, Q>(v, nw, nb, shift, a.rms, a.W, n4, xstride >> 2, a.eps, red, (f32x4*)(xs + (size_t)q0 * xstride), xstride >> 2,
                          nullptr, 0);
  }
  if (norms) ld_items_begin(t, item, items, nblk, nch, lane, set_rows);
  __syncthreads();
  float bv = -INFINITY;
  int bi = 0x7fffffff;
  const LdOwn own = ld_own<R, B>(lane);
  ld_items<B>(t, item, step, items, nblk, nch, xs, xstride, lane, set_rows, [](int) {}, [&](int it, float v) __attribute__((always_inline)) {
    if (!own.on) return;
    const int i = it * R + own.r;
    if (a.cap > 0.f) v = a.cap * tanhf(v / a.cap);
    if (i < a.V) {
      a.logits[(size_t)own.q * a.V + i] = v;
      if (own.q == 0) amax_merge(bv, bi, v, i);
    }
  });
  if (a.part_val) {
    wave_amax(bv, bi);
    if (lane == 0) {
      sv[wave] = bv;
      si[wave] = bi;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
      for (int w = 1; w < NW; ++w) amax_merge(bv, bi, sv[w], si[w]);
      a.part_val[blockIdx.x] = bv;
      a.part_idx[blockIdx.x] = bi;
    }
  }
}
}  // namespace khm
