// kh_lgemm.h — GEMM of the layer-list models on the matrix cores: out[token][feature] = X[token][K] . W[feature][K],
// storage type T = bf16 or fp32 on both sides (kh_tile.h), fp32 accumulation.
//
//   * One workgroup = 4 waves (2 x 2) = a BM-token x BN-feature tile; K advances 128 bytes per stage through two rings of
//     LDS stages, XS of tokens and WS of weights, filled by the LDS-DMA path (global_load_lds_dwordx4): no staging
//     registers, and XS - 1 and WS - 1 stages are in flight while one is multiplied.  The big tiles use two stages, which
//     leaves room for two workgroups per CU: one multiplies while the other waits (128 x 128: 0.43 - 0.50 of the bf16 peak,
//     against 0.28 - 0.33 with three stages and one workgroup).  Experts' weights come from HBM, each tile for two or three
//     workgroups only, and wait for it longer than a stage's products take: the 80 KB that two workgroups leave each other
//     hold a third stage of weights (2048 tokens, 6 of 32 experts, 2048 x 2048: 141 -> 130 us; 1100 tokens, 7 of 32,
//     1024 x 1024: 41 -> 36).  Weights that all tokens share come from the L2, and two stages do as well there.  Measured
//     and not kept: stages of 64 bytes, five of them (30 % slower: requests of half lines), fragments read one half stage
//     ahead of their products (up to 20 % slower), the tiles of an expert on one XCD (+3 % at 2048 columns, -2 % at 1024).
//   * Token tiles of 16 go to the two waves of a column in turn; a wave multiplies those that hold rows, so a tile that is
//     not full costs what it holds.
//   * LDS rows are 128 bytes.  Chunk c (16 bytes) of row r sits in slot c ^ (r & 7): the lanes of a fragment read
//     (16 rows, same chunk) touch all 64 banks.  The DMA writes slots in lane order, so the permutation is applied
//     to the GLOBAL address each lane requests.
//   * Weights are the first MFMA operand: a lane ends with four consecutive features of one token, which is what
//     every epilogue stores.
//   * Every row length is padded to KH_LPAD elements at load (zero weights), so K needs no tail; token and feature
//     tails are clamped on load and masked on store.
//   * Grouped form (experts): a device-side tile list maps blockIdx.y to (expert, first row, rows); the rows of X are
//     gathered through an index list.  Batched form (heads): blockIdx.z strides.
#pragma once
#include <math.h>
#include <type_traits>
#include <vector>

#include "kh_q8ring.h"
#include "kh_tile.h"

#define KH_LPAD 64  // K granule of every weight row, in elements (128 bytes of bf16, 256 of fp32)

namespace khm {

enum LgEpi {
  LG_T = 0,        // out T (+ bias)
  LG_F32 = 1,      // out fp32 (+ bias)
  LG_SOFTPLUS = 2, // out fp32 = softplus(acc + bias[feature])
  LG_GATED = 3,    // weight rows come as 16 gate rows, 16 up rows, ...: out T = the gated unit, half the features
  LG_SPLIT = 4,    // features [0, n_split) -> out T, the rest -> out2 fp32
  LG_SOFTCAP = 5,  // out fp32 = cap * tanh(acc / cap); cap 0: plain
};

struct LgTile {  // one token tile of a grouped launch
  int group, row0, rows, pad;
};

struct LgArgs {
  const void* W;        // [N][ldw]
  const void* X;        // [M][ldx]
  void* out;            // [M][ldo]
  float* out2;          // LG_SPLIT: [M][ldo2]
  const float* bias;    // LG_SOFTPLUS; LG_T / LG_F32: optional
  const int32_t* gather;   // row of X for row m (grouped, optional)
  const LgTile* tiles;     // grouped launch
  const int32_t* n_tiles;  // number of valid entries of tiles
  size_t w_group;       // grouped: elements between the weights of two groups
  size_t w_z, x_z, o_z; // batched: elements per blockIdx.z
  int M, N, K, ldw, ldx, ldo, ldo2, n_split;
  float cap;
  GateAct act;          // LG_GATED
};

// WM x WN: waves along the tokens and the features
template <class T, int BM, int BN, bool GROUPED, int WM = 2, int WN = 2>
struct LgCfg {
  static constexpr bool WIDE = WM * WN == 8;  // one workgroup of eight waves per CU: the whole LDS is its
  static constexpr int XS = WIDE ? 160 * 8 / (BM + BN) : BM + BN >= 192 ? 2 : (BM + BN >= 128 ? 3 : 4);  // stages of the tokens' ring
  static constexpr int WS = !WIDE && BM + BN == 256 && GROUPED ? 3 : XS;                                 // ... of the weights'
  static constexpr int LDS = (XS * BM + WS * BN) * 128;
};

// Biases ahead of the stores, because a load behind them waits for them (LG_SOFTPLUS, 2048 x 4096 of K 128 in bf16 28.7 -> 23.7 us)?
// Not in fp32 outside LG_SOFTPLUS: there the loop's registers come out differently, and 64 x 64 tiles are slower as a whole (606
// tokens x 2048 of K 7168 241 -> 257 us, x 3072 of K 2048 75.4 -> 79.4; 2048 x 1024 of K 3584 130 -> 138), 64 x 128 2 % faster.
template <class T, int EPI>
constexpr bool lg_bias_first() { return EPI == LG_SOFTPLUS || (sizeof(T) == 2 && (EPI == LG_T || EPI == LG_F32)); }
// biases of features f .. f + 3, f a multiple of four (no bias: zeros)
template <int EPI>
__device__ __forceinline__ f32x4 lg_bias(const LgArgs& a, int f) {
  f32x4 b = f4_zero();
  if (EPI == LG_SOFTPLUS || a.bias) {
#pragma unroll
    for (int i = 0; i < 4; ++i) b[i] = a.bias[f + i < a.N ? f + i : 0];
  }
  return b;
}
// features f .. f + 3 of one token; b: their biases, where they come first
template <class T, int EPI>
__device__ __forceinline__ void lg_store(const LgArgs& a, int tok, int f, f32x4 v, const f32x4& b) {
  typedef Tile<T> TL;
  if (lg_bias_first<T, EPI>() && EPI != LG_SOFTPLUS) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] += b[i];
  } else if ((EPI == LG_T || EPI == LG_F32) && a.bias) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] += a.bias[f + i < a.N ? f + i : 0];
  }
  if (EPI == LG_T) {
    T* o = (T*)a.out + (size_t)blockIdx.z * a.o_z + (size_t)tok * a.ldo + f;
    if (f + 3 < a.N && (a.ldo & 3) == 0) {
      *(typename TL::quad*)o = to_quad<T>(v);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (f + i < a.N) o[i] = (T)v[i];
    }
  } else {
    f32x4 y = v;
    if (EPI == LG_SOFTPLUS) {
#pragma unroll
      for (int i = 0; i < 4; ++i) y[i] = softplus1(v[i] + b[i]);
    } else if (EPI == LG_SOFTCAP) {
#pragma unroll
      for (int i = 0; i < 4; ++i) y[i] = a.cap > 0.f ? a.cap * tanhf(v[i] / a.cap) : v[i];
    }
    // destination of the four features: one array, unless they straddle LG_SPLIT's border
    const bool to_t = EPI == LG_SPLIT && f + 3 < a.n_split, cut = EPI == LG_SPLIT && !to_t && f < a.n_split;
    float* o = EPI == LG_SPLIT ? a.out2 + (size_t)tok * a.ldo2 + (f - a.n_split) : (float*)a.out + (size_t)tok * a.ldo + f;
    const int ld = EPI == LG_SPLIT ? a.ldo2 : a.ldo;
    if (to_t) {
      T* ot = (T*)a.out + (size_t)tok * a.ldo + f;
#pragma unroll
      for (int i = 0; i < 4; ++i) ot[i] = (T)y[i];
    } else if (!cut && f + 3 < a.N && (ld & 3) == 0) {
      *(f32x4*)o = y;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (f + i >= a.N) continue;
        if (EPI == LG_SPLIT && f + i < a.n_split) ((T*)a.out)[(size_t)tok * a.ldo + f + i] = (T)y[i];
        else o[i] = y[i];
      }
    }
  }
}

template <class T, int BM, int BN, int EPI, bool GROUPED, int WM = 2, int WN = 2>
__global__ __launch_bounds__(64 * WM * WN, BM == 192 ? 2 : 1) void k_lgemm(const LgArgs a) {
  typedef Tile<T> TL;
  typedef typename TL::frag frag;
  constexpr int NWV = WM * WN;
  constexpr int XS = LgCfg<T, BM, BN, GROUPED, WM, WN>::XS, WS = LgCfg<T, BM, BN, GROUPED, WM, WN>::WS;
  static_assert(XS >= 2 && WS >= XS, "order of the requests");
  static_assert(LgCfg<T, BM, BN, GROUPED, WM, WN>::LDS <= 160 * 1024, "fits a CU");
  constexpr int TM = BM / (16 * WM), TN = BN / (16 * WN);    // 16-wide tiles per wave: tokens, features
  constexpr int NX = BM / (8 * NWV), NW = BN / (8 * NWV);    // LDS-DMA requests per wave and stage
  static_assert(EPI != LG_GATED || TN % 2 == 0, "a gate tile and its up tile are one wave's");
  extern __shared__ __attribute__((aligned(1024))) char smem_raw[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const char* W = (const char*)a.W;
  const char* X = (const char*)a.X;
  int m_lo = 0, m_n = a.M;  // rows [m_lo, m_lo + m_n) of the row index space belong to this launch / group
  int mt0;                  // first row of the tile
  if (GROUPED) {
    if ((int)blockIdx.y >= *a.n_tiles) return;  // uniform: the grid is an upper bound
    const LgTile t = a.tiles[blockIdx.y];
    W += (size_t)t.group * a.w_group * sizeof(T);
    m_lo = t.row0;
    m_n = t.rows;
    mt0 = t.row0;
  } else {
    mt0 = (int)blockIdx.y * BM;
  }
  W += (size_t)blockIdx.z * a.w_z * sizeof(T);
  X += (size_t)blockIdx.z * a.x_z * sizeof(T);
  const int f0 = (int)blockIdx.x * BN;
  const int m_last = m_lo + m_n - 1;
  // ---- staging addresses: request j of wave w covers rows 8 (NWV j + w) .. +8 of the token tile, or of the feature tile
  unsigned xoff[NX], woff[NW];
  const int sub = lane >> 3, ch = (lane & 7) ^ sub;
#pragma unroll
  for (int j = 0; j < NX; ++j) {
    int m = mt0 + 8 * (NWV * j + wave) + sub;
    m = m < m_last ? m : m_last;
    const int row = GROUPED && a.gather ? a.gather[m] : m;
    xoff[j] = (unsigned)row * (unsigned)(a.ldx * (int)sizeof(T)) + 16u * ch;
  }
#pragma unroll
  for (int j = 0; j < NW; ++j) {
    int f = f0 + 8 * (NWV * j + wave) + sub;
    f = f < a.N ? f : a.N - 1;
    woff[j] = (unsigned)f * (unsigned)(a.ldw * (int)sizeof(T)) + 16u * ch;
  }
  const unsigned lds0 = (unsigned)__builtin_amdgcn_readfirstlane((int)kh_lds_addr(smem_raw)) + 1024u * wave;
  auto issue_x = [&](int slot) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < NX; ++j) {
      dma_x4_keep(X, xoff[j], lds0 + (unsigned)(slot * BM * 128 + j * 1024 * NWV));
      xoff[j] += 128;
    }
  };
  auto issue_w = [&](int slot) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < NW; ++j) {
      dma_x4_keep(W, woff[j], lds0 + (unsigned)(XS * BM * 128 + slot * BN * 128 + j * 1024 * NWV));
      woff[j] += 128;
    }
  };
  const int nk = a.K * (int)sizeof(T) / 128;  // stages
  f32x4 acc[TN][TM];
#pragma unroll
  for (int n = 0; n < TN; ++n)
#pragma unroll
    for (int m = 0; m < TM; ++m) acc[n][m] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < WS - 1; ++j) {  // as WS - 1 steps before the first would request them
    if (j >= WS - XS && j - (WS - XS) < nk) issue_x(j - (WS - XS));
    if (j < nk) issue_w(j);
  }
  const int wm = wave % WM, wn = wave / WM;
  const int fr = lane & 15, fh = lane >> 4;
  const int fo0 = fr * 128 + ((fh ^ (fr & 7)) << 4);  // this lane's fragment within 16 rows, first half of the stage
  constexpr int LATER = WS > XS ? NW : 0;             // requests of a step behind the ones that are waited for
  // LIVE: token tiles of this wave that hold rows
  auto loop = [&](auto live) __attribute__((always_inline)) {
    constexpr int LIVE = decltype(live)::value;
    int xslot = 0, wslot = 0, xfill = XS - 1, wfill = WS - 1;
    auto next = [](int s, int n) __attribute__((always_inline)) { return s + 1 == n ? 0 : s + 1; };
    for (int k = 0; k < nk; ++k) {
      // stage k has landed when at most the requests behind it are outstanding
      if (k + WS - 2 < nk) wait_vm<LATER + (XS - 2) * (NX + NW)>();
      else wait_vm<0>();
      __syncthreads();
      if (k + XS - 1 < nk) issue_x(xfill);
      if (k + WS - 1 < nk) issue_w(wfill);
      // both halves of the stage are requested from LDS before the first product: the second half arrives under the
      // products of the first (left to itself the compiler reads one half at a time; 0.40 -> 0.43 ... 0.50 of the peak)
      frag fx[2][LIVE], fw[2][TN];
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const char* sx = smem_raw + xslot * BM * 128 + (fo0 ^ (b << 6));
        const char* sw = smem_raw + XS * BM * 128 + wslot * BN * 128 + (fo0 ^ (b << 6));
#pragma unroll
        for (int m = 0; m < LIVE; ++m) fx[b][m] = *(const frag*)(sx + (WM * m + wm) * 2048);
#pragma unroll
        for (int n = 0; n < TN; ++n) fw[b][n] = *(const frag*)(sw + (wn * TN + n) * 2048);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int n = 0; n < TN; ++n)
#pragma unroll
          for (int m = 0; m < LIVE; ++m) acc[n][m] = TL::mma(fw[b][n], fx[b][m], acc[n][m]);
      xslot = next(xslot, XS);
      wslot = next(wslot, WS);
      xfill = next(xfill, XS);
      wfill = next(wfill, WS);
    }
  };
  const int tiles_m = (m_last - mt0) / 16 + 1;  // of the workgroup, with rows in them; they go to the waves in turn
  const int live = (tiles_m - wm + WM - 1) / WM;
  if (TM == 1 || (TM <= 4 && live <= 1)) loop(std::integral_constant<int, 1>{});
  else if (TM == 2 || (TM <= 4 && live == 2)) loop(std::integral_constant<int, TM < 2 ? 1 : 2>{});
  else if (TM <= 4 && live == 3) loop(std::integral_constant<int, TM < 3 ? 1 : 3>{});
  else if (TM == 6 && live <= 2) loop(std::integral_constant<int, TM < 2 ? 1 : 2>{});
  else if (TM == 6 && live <= 4) loop(std::integral_constant<int, TM < 4 ? 1 : 4>{});
  else if (TM == 6 && live == 5) loop(std::integral_constant<int, TM < 5 ? 1 : 5>{});
  else loop(std::integral_constant<int, TM>{});
  // ---- epilogue: lane (fr, fh) of tile (n, m): token mt0 + .. + fr, features f .. f + 3
  auto feature = [&](int n) __attribute__((always_inline)) { return f0 + wn * (BN / WN) + n * 16 + 4 * fh; };
  constexpr bool BIAS = lg_bias_first<T, EPI>();
  f32x4 bias[BIAS ? TN : 1];
  if constexpr (BIAS) {
#pragma unroll
    for (int n = 0; n < TN; ++n) bias[n] = lg_bias<EPI>(a, feature(n));
  }
#pragma unroll
  for (int m = 0; m < TM; ++m) {
    const int tok = mt0 + (WM * m + wm) * 16 + fr;
    if (tok > m_last) continue;
    if (EPI == LG_GATED) {
#pragma unroll
      for (int n = 0; n + 1 < TN; n += 2) {
        const int f = f0 + wn * (BN / WN) + n * 16;  // a multiple of 32: gate tile; the up tile follows
        const int c = (f >> 1) + 4 * fh;
        f32x4 v;
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = gated1(a.act, acc[n][m][i], acc[n + 1][m][i]);
        if (f < a.N) *(typename TL::quad*)((T*)a.out + (size_t)tok * a.ldo + c) = to_quad<T>(v);
      }
    } else {
#pragma unroll
      for (int n = 0; n < TN; ++n) lg_store<T, EPI>(a, tok, feature(n), acc[n][m], bias[BIAS ? n : 0]);
    }
  }
}

// Tile choice.  Plain / batched launches: the largest tile that still gives the chip enough workgroups (one of four waves per CU is
// not: nobody covers its barriers).  In bf16 there are two forms of eight waves, one workgroup per CU with the whole LDS, where
// the tiles fill the CUs once: 256 x 256 in two stages, which a CU reads half as much for (2048 tokens x 8192 x 2048: 69.8 -> 64.9 us;
// with rounds that are less than 200 of 256 full it loses that), and 128 x 128 in five, from 129 tiles on (2048 x 2048, K 4096 /
// 2048: 57 / 31 us as 512 workgroups of 64 x 128, 44 / 25 so; 144 tiles of 1100 tokens, K 4096 / 2048 43 / 24 -> 38 / 22; 128
// tiles: 12.7 us instead of 9.9).  Experts gain nothing from either (130 us of gate and up with 256 x 256, 137 with 256 x 128): their
// tiles are a third empty or wait for HBM.  Where 64 x 64 leaves half of the CUs idle, 32 x 64: what one CU pulls is the time (160
// features of K 4096, 2048 / 732 tokens: 25.2 / 24.0 -> 18.6 / 17.1 us).  Grouped launches: BM = the row granule the tile list was built with (lg_group_bm).
// (rows: token and choice pairs, over `groups` outputs; w_bytes: weights of all experts of the gate and up product, N columns)
// 192 rows for 128 where an expert's share lies so close below 128 or 256 that some of them pass it, and what those bring is a second
// round of workgroups (two fit a CU): more than 512 tiles of 128 rows are expected, the experts' rows spread as independent choices
// would, and those of 192 are one round.  us a prompt with 128 / 192 rows, 32 experts of 1024 x 1024: Gusorax, 7 choices, 1036 / 1100 / 1165
// tokens in fp32 2042 / 2110 / 2200 -> 1971 / 2000 / 2144, in bf16 700 / 707 / 733 -> 700 / 717 / 733; Gufanex, 6 choices, 1360 / 1450 / 1530
// tokens in fp32 3395 / 3555 / 3685 -> 3364 / 3566 / 3761, in bf16 1268 / 1296 / 1292 -> 1219 / 1260 / 1325; 28 experts of 1152 x 640, fp32, 930 /
// 960 / 1010 tokens 1369 / 1427 / 1457 -> 1340 / 1357 / 1390.  Where 128 rows are one round as well, 192 only make the longest workgroup longer and
// the ring of weights shorter: experts of 512 x 512, 540 / 1700 tokens in fp32 894 / 1820 -> 988 / 1992, of 1024 x 1024, Gufanex, 700 tokens
// 2911 -> 3167, 540 tokens in bf16 715 -> 748 (in fp32 the other way, 1858 -> 1780).  Several rounds hide the second (2048
// tokens: 128.7 / 131.5), and more weights wait for HBM longer than two stages of them cover (740 tokens, 6 of 36, 2048 x 2048, 268
// MB: the prompt 1299 / 1354).
static inline int lg_group_bm(long rows, int groups, int experts, int N, size_t w_bytes) {
  const long per = rows / (groups > 0 ? groups : 1);
  if (per <= 64) return per > 24 ? 64 : 32;
  const double sd = sqrt((double)per), most = per + 2.0 * sd;
  const long n = (per + 127) / 128, tiles = experts * n * ((N + 127) / 128);
  const double pass = 0.5 * erfc((128.0 * n + 0.5 - per) / (sd * sqrt(2.0)));  // share of the experts with a tile more
  const bool second = most > 128.0 * n && tiles * (n + pass) > 512.0 * n;
  return second && most <= 192.0 * n && tiles <= 512 && w_bytes <= (128u << 20) ? 192 : 128;
}
template <class T, int EPI>
int lg_launch(hipStream_t s, const LgArgs& a, int zdim = 1, int group_bm = 0, int max_tiles = 0) {
  auto go = [&](auto kern, int BM, int BN, int lds, int wg) -> int {
    if (lds > 64 * 1024) {  // the dynamic-LDS opt-in is per (device, kernel): once
      struct Done { int dev; const void* fn; };
      static thread_local std::vector<Done> done;
      int dev = 0;
      (void)hipGetDevice(&dev);
      bool hit = false;
      for (const auto& d : done) hit = hit || (d.dev == dev && d.fn == (const void*)kern);
      if (!hit) {
        const hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (e != hipSuccess) return (int)e;
        done.push_back({dev, (const void*)kern});
      }
    }
    const int gy = a.tiles ? max_tiles : (a.M + BM - 1) / BM;
    hipLaunchKernelGGL(kern, dim3((a.N + BN - 1) / BN, gy, zdim), dim3(wg), lds, s, a);
    return KH_OK;
  };
  auto tiles = [&](int BM, int BN) { return (long)((a.N + BN - 1) / BN) * ((a.M + BM - 1) / BM) * zdim; };
#define KH_LG_GO(BM, BN, G) return go(k_lgemm<T, BM, BN, EPI, G>, BM, BN, LgCfg<T, BM, BN, G>::LDS, 256)
#define KH_LG_WIDE(BM, BN) return go(k_lgemm<T, BM, BN, EPI, false, 2, 4>, BM, BN, LgCfg<T, BM, BN, false, 2, 4>::LDS, 512)
  if constexpr (EPI == LG_T || EPI == LG_GATED) {
    if (a.tiles) {
      if (group_bm == 192) KH_LG_GO(192, 128, true);
      if (group_bm == 128) KH_LG_GO(128, 128, true);
      if (group_bm == 64) KH_LG_GO(64, 128, true);
      KH_LG_GO(32, 64, true);
    }
  } else if (a.tiles) {
    return KH_ERR_INTERNAL;
  }
  if constexpr (sizeof(T) == 2 && (EPI == LG_T || EPI == LG_F32)) {
    const long t = tiles(128, 128), w = tiles(256, 256);
    auto full = [&](int bm) { return 4L * ((a.M + bm - 1) / bm * bm) <= 5L * a.M; };  // a fifth of the rows empty at most
    if ((w % 256 == 0 || w % 256 >= 200) && full(256)) KH_LG_WIDE(256, 256);
    if (t > 128 && t <= 256 && full(128)) KH_LG_WIDE(128, 128);
  }
  if (a.M > 64 && tiles(128, 128) >= 400) KH_LG_GO(128, 128, false);
  if (a.M <= 32 || tiles(64, 64) <= 128) KH_LG_GO(32, 64, false);
  if (tiles(64, 128) >= 400) KH_LG_GO(64, 128, false);
  KH_LG_GO(64, 64, false);
#undef KH_LG_GO
#undef KH_LG_WIDE
}
}  // namespace khm
