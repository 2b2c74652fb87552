// kh_model_pair.hip — prompt passes of .bin models on the pair GEMMs (kh_pair.h): launch shapes, one pass of up to
// KH_PAIR_TMAX prompt tokens.  The reference feeds the prompt one token per forward pass (demo/main.cpp:20-22).  gfx950 only.
#include <stdio.h>
#include <stdlib.h>

#include <algorithm>
#include <vector>

#include "kh_model_internal.h"
#include "kh_pattn.h"
#include "kh_pattn_pair.h"

using namespace khm;

namespace {
// Tile and K split of one GEMM from a model of its time (us): a workgroup's stage takes at least `lat` (one or more stages in
// flight against memory latency), `n` workgroups side by side on a CU take n `sat` per stage together, every workgroup of a CU has
// a start and an end, and partial rows are written and read back.  Where some CUs have a workgroup more than others, n lies
// between the most and the mean: they compete for what lies behind the CUs as well.  The numbers were fitted to all twelve tile
// and split combinations of the four GEMMs of five models (Llama-3.2-1B, TinyLlama, Qwen2.5-0.5B, stories15M; Llama-2-7B int8) at 40 ...
// 2000 tokens, 44 lengths: the choice is on average 0.4 % (fp32, 14 % at worst) and 0.01 % (int8, 0.2 %) behind the fastest
// combination measured, their sum 0.2 and 0.00 %; with the busiest CU alone and numbers from 18 combinations of two models 2.4
// (29) and 0.7 (16), the sum 2.1 and 0.5 %.  They belong to the tile and the 256 CUs, not to a model; other widths take them as they are.
// The largest tile of a type is the largest whose registers do not spill: 8 x 2 fragments a wave for fp32, 7 x 2 (112
// tokens) for int8, where 8 x 2 spills 18 to 24 registers, the sums of a 64-column group standing beside the accumulators.
// Against the tiled fp32-MFMA kernel (k_pg_gemm), us at 40 / 128 / 512 / 2000 tokens, w1 + w3 of either model:
// 38 / 48 / 108 / 388 against 46 / 76 / 287 / 1089 (fp32); 56 / 88 / 232 / 816 against 126 / 210 / 792 / 3032 (int8).
// Only wq + wk + wv of 64 fp32 tokens or less were faster there (18 us against 24); whole prompts of 32 tokens and less take
// 0.67 to 0.94 of its time, on Llama-3.2-1B 1.03.
struct PairShape {
  int tile;  // index into kPairTiles
  int kz;    // K slices across workgroups (residual GEMMs)
};
struct PairTile {
  int bm, bn, occ;  // occ: workgroups that share a CU
  double lat, sat;
};
const PairTile kPairTiles[2][4] = {
    {{128, 128, 2, 1.028, 0.752}, {64, 128, 2, 0.592, 0.471}, {32, 128, 2, 0.484, 0.348}, {32, 64, 2, 0.389, 0.228}},  // fp32
    {{112, 128, 2, 1.346, 0.885}, {64, 128, 2, 0.850, 0.592}, {32, 128, 2, 0.615, 0.414}, {128, 256, 1, 2.116, 2.116}}};  // int8
// of a workgroup: its start and end; of partial rows: of their time at 4 TB/s; weight of the busiest CU against the mean
const struct {
  double ends, part, most;
} kPairCost[2] = {{1.833, 0.650, 0.444}, {2.167, 0.929, 1.0}};

// resid: a product that is added to the residual (wo, w2).  gated: w1 + w3, whose scales the product behind it has to fold in twice
// as often where a tile leaves them per 32 columns.  With and without 1.15 for it: passes of 33 to 64 tokens take 32 x 128 instead of 32
// x 64, us, TinyLlama 33 2172 / 2158, 50 2229 / 2184, 64 2279 / 2208, Qwen2.5-0.5B 41 1597 / 1580, 64 1651 / 1612; elsewhere the choice
// is the same (Llama-3.2-1B and the shortest passes of all three, where 32 x 64 are more workgroups on idle CUs).
PairShape pair_shape(bool q, int T, int N, int K, bool resid, bool gated, double* time_us = nullptr) {
  PairShape best{0, 1};
  double best_us = -1.0;
  for (int i = 0; i < 4; ++i)
    for (int kz = 1; kz <= (resid ? KH_PG_KZ_MAX : 1); kz *= 2) {
      const PairTile& t = kPairTiles[q][i];
      const int stages = K / (q ? 64 : 32);
      if (kz > 1 && stages / kz < 4) break;
      const long wgs = (long)((N + t.bn - 1) / t.bn) * ((T + t.bm - 1) / t.bm) * kz;
      const long most = (wgs + 255) / 256, rounds = (most - 1) / t.occ;
      const double last = kPairCost[q].most * most + (1.0 - kPairCost[q].most) * std::max(wgs / 256.0, 1.0) - (double)(rounds * t.occ);
      double us = rounds * std::max(t.lat, t.occ * t.sat) + std::max(t.lat, last * t.sat);
      us = us * stages / kz + kPairCost[q].ends * most;
      if (kz > 1) us += kPairCost[q].part * kz * T * N * 8 / 4.0e6;
      if (gated && t.bn < 128) us *= 1.15;
      if (best_us < 0 || us < best_us) {
        best_us = us;
        best = PairShape{i, kz};
      }
    }
  if (time_us) *time_us = best_us;
  return best;
}
// the four GEMMs of a layer
struct PairDims {
  int N[4], K[4];
};
PairDims pair_dims(const kh_config& c) {
  return {{c.dim + 2 * c.kv_dim, c.dim, 2 * c.hidden_dim, c.dim}, {c.dim, c.dim, c.dim, c.hidden_dim}};
}

template <bool Q, int EPI, int TM, int TN, int WM, int WN, int NST>
int pair_go(hipStream_t s, KhPairArgs a, int kz) {
  typedef PairCfg<Q, EPI == KH_PG_RESID, TM, TN, WM, WN, NST> C;
  auto kern = k_pair_gemm<Q, EPI, TM, TN, WM, WN, NST>;
  if (C::LDS > 64 * 1024) {  // the dynamic-LDS opt-in is per (device, kernel): once
    static thread_local std::vector<int> done;
    int dev = 0;
    (void)hipGetDevice(&dev);
    bool hit = false;
    for (int d : done) hit = hit || d == dev;
    if (!hit) {
      KH_CHECK_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS));
      done.push_back(dev);
    }
  }
  a.tiles_t = (a.T + C::BM - 1) / C::BM;
  a.tiles_f = (a.N + C::BN - 1) / C::BN;
  hipLaunchKernelGGL(kern, dim3((a.tiles_f * a.tiles_t + 7) / 8 * 8, kz), dim3(64 * C::NW), C::LDS, s, a);
  return KH_OK;
}
// *kz_out: K slices whose partial rows the next RMSNorm has to add (0: the epilogue added itself)
// *fine_out: SWIGLU left a scale per 32 columns instead of 64
template <int EPI>
int pair_launch(kh_model* m, const KhPairArgs& a, int* kz_out, int* fine_out = nullptr) {
  PairShape sh = pair_shape(m->cfg.is_quant, a.T, a.N, a.K, EPI == KH_PG_RESID, EPI == KH_PG_SWIGLU);
  if (const char* e = dbg("KH_PAIR_SHAPE")) {  // test hook "tile,kz"
    int t = 0, kz = 1;
    if (sscanf(e, "%d,%d", &t, &kz) == 2 && t >= 0 && t < 4 && (kz == 1 || kz == 2 || kz == 4))
      sh = PairShape{t, EPI == KH_PG_RESID ? kz : 1};
  }
  while (sh.kz > 1 && sh.kz * a.T > m->pg_part_rows) sh.kz /= 2;  // (a hook set behind the allocation)
  if (fine_out) *fine_out = kPairTiles[m->cfg.is_quant][sh.tile].bn < 128;
  if (kz_out) *kz_out = sh.kz > 1 ? sh.kz : 0;
  if (m->cfg.is_quant) {
    switch (sh.tile) {
      case 0: return pair_go<true, EPI, 7, 2, 1, 4, 2>(m->stream, a, sh.kz);
      case 1: return pair_go<true, EPI, 4, 2, 1, 4, 3>(m->stream, a, sh.kz);
      case 2: return pair_go<true, EPI, 2, 2, 1, 4, 4>(m->stream, a, sh.kz);
      default: return pair_go<true, EPI, 4, 4, 2, 4, 3>(m->stream, a, sh.kz);
    }
  }
  switch (sh.tile) {
    case 0: return pair_go<false, EPI, 8, 2, 1, 4, 2>(m->stream, a, sh.kz);
    case 1: return pair_go<false, EPI, 4, 2, 1, 4, 3>(m->stream, a, sh.kz);
    case 2: return pair_go<false, EPI, 2, 2, 1, 4, EPI == KH_PG_RESID ? 3 : 4>(m->stream, a, sh.kz);
    default: return pair_go<false, EPI, 1, 2, 2, 2, 6>(m->stream, a, sh.kz);
  }
}
}  // namespace

// Host-only view of pair_shape for the four GEMMs of a layer; KH_PAIR_SHAPE is not applied.
extern "C" int kh_plan_pair_shapes(int32_t dim, int32_t hidden_dim, int32_t kv_dim, int32_t is_quant, int32_t T, int32_t* out16) {
  if (!out16 || dim <= 0 || hidden_dim <= 0 || kv_dim <= 0 || T <= 0 || T > KH_PAIR_TMAX) return KH_ERR_INVALID_ARG;
  kh_config c{};
  c.dim = dim;
  c.hidden_dim = hidden_dim;
  c.kv_dim = kv_dim;
  c.is_quant = is_quant != 0;
  if (!pair_geometry(c)) return KH_ERR_UNSUPPORTED;
  const PairDims d = pair_dims(c);
  for (int i = 0; i < 4; ++i) {
    const PairShape s = pair_shape(c.is_quant, T, d.N[i], d.K[i], i & 1, i == 2);
    const PairTile& t = kPairTiles[c.is_quant][s.tile];
    int32_t* o = out16 + 4 * i;
    o[0] = t.bm;
    o[1] = t.bn;
    o[2] = s.kz;
    o[3] = (d.N[i] + t.bn - 1) / t.bn * ((T + t.bm - 1) / t.bm) * s.kz;
  }
  return KH_OK;
}

namespace khm {
// Pair slabs advance in 32-column blocks, int8 groups in 64, and k_pair_gemm addresses a matrix and a slab with 32 bits:
// other widths stay with k_pg_gemm.
bool pair_geometry(const kh_config& c) {
  const int g = c.is_quant ? 64 : 32;
  const int64_t wide = std::max(c.dim, c.hidden_dim), lim = (int64_t)1 << 32;
  return c.dim % g == 0 && c.hidden_dim % g == 0 && wide * c.dim * (c.is_quant ? 1 : 4) <= lim && wide * KH_PAIR_TMAX * 4 <= lim;
}

// Is the last of T tokens of a pass cheaper in the pass than as a step of its own?  The step reads a layer's weights once more
// (5 TB/s behind 10 us of launches a layer); in the pass the token may open another row of tiles.  Time to the first token, ms,
// step of its own / in the pass, T tokens.  Taken: Llama-3.2-1B 193 3.65 / 3.12, 257 3.96 / 3.86, 641 6.50 / 6.12; TinyLlama 641
// 6.95 / 6.58, 705 7.50 / 7.31, 1473 13.3 / 11.9; Qwen2.5-0.5B 513 3.88 / 3.32, 833 4.74 / 4.48, 1153 5.62 / 5.19; Llama-2-7B
// int8 113 8.93 / 7.51, 225 12.0 / 11.0, 673 26.4 / 25.9.  Not taken: Llama-3.2-1B 513 5.33 / 5.63, 1025 8.17 / 8.59; TinyLlama 1409
// 11.65 / 11.95; Llama-2-7B int8 65 6.88 / 7.22, 321 14.5 / 15.3, 641 23.4 / 24.8.  Of 34 lengths, most of them where the last token
// opens a row of tiles, the rule errs at one, Qwen2.5-0.5B 1665 6.96 / 6.77.
bool pair_takes_last(const kh_config& c, int T) {
  if (T < 2) return false;
  const PairDims d = pair_dims(c);
  double more = 0.0, bytes = 0.0;
  for (int i = 0; i < 4; ++i) {
    double with = 0.0, without = 0.0;
    (void)pair_shape(c.is_quant, T, d.N[i], d.K[i], i & 1, i == 2, &with);
    (void)pair_shape(c.is_quant, T - 1, d.N[i], d.K[i], i & 1, i == 2, &without);
    more += with - without;
    bytes += (double)d.N[i] * d.K[i] * (c.is_quant ? 1 : 4);
  }
  return more < 10.0 + bytes / 5.0e6;
}

int pair_part_rows(const kh_config& c, int rows) {
  int most = 0;
  for (int T = 1; T <= rows; ++T)
    for (int K : {c.dim, c.hidden_dim}) {
      const int kz = pair_shape(c.is_quant, T, c.dim, K, true, false).kz;
      if (kz > 1) most = std::max(most, kz * T);
    }
  return most;
}

namespace {
template <int HS, int QT>
void pa_go(const KhPaArgs& a, hipStream_t s) {
  hipLaunchKernelGGL(k_pa_pack<HS>, dim3((a.pos0 + a.T + 31) / 32, a.kv_heads), dim3(256), 0, s, a);
  hipLaunchKernelGGL((k_pa_attn<HS, 4, QT>), dim3(a.kv_heads * a.kv_mul * ((a.T + 16 * QT - 1) / (16 * QT))), dim3(256), 0, s, a);
}
// bytes of one layer's K / V rows as pairs; 0: no kernel for this head size
size_t pa_bytes(const kh_config& c, int positions) {
  auto block = [](auto g) { return (size_t)decltype(g)::FR * 1024 + 2 * sizeof(float); };
  const size_t n = (size_t)c.kv_head_num * ((positions + 31) / 32);
  switch (c.head_size) {
    case 48: return n * block(PaGeom<48>{});
    case 64: return n * block(PaGeom<64>{});
    case 128: return n * block(PaGeom<128>{});
    default: return 0;
  }
}

// Attention of a slice with its operands as pairs; false: the caller takes pg_slice_attention (fp32 matrix cores).
// Packing reads all of the layer's rows whatever T is, so it needs enough query tokens and enough work.  Whole prompt
// passes, ms, fp32 matrix cores against pairs, T @ first position: Llama-3.2-1B 256 @ 0 2.78 / 2.79, 512 @ 0 4.14 / 4.03,
// 256 @ 2048 3.45 / 3.11, 2048 @ 2048 18.8 / 14.2; Llama-2-7B int8 256 @ 0 10.7 / 10.6, 128 @ 1024 8.35 / 8.19,
// 1024 @ 1024 41.8 / 35.2.  128 @ 0 and 64 @ 2048 gain nothing.
bool pa_pays(int T, int pos0) {
  if (dbg_off("KH_PG_ATTN") || dbg("KH_PG_ATTN_QT") || dbg_off("KH_PAIR_ATTN")) return false;
  return T >= 128 && (size_t)T * (2 * (size_t)pos0 + T) >= 65536;
}
}  // namespace
// The slab of a layer is given up (not the call) above KH_PA_WS_MAX and where memory for it is refused.  It at least doubles.
void pair_prepare(kh_model* m, int n, int pos0) {
  const kh_config& c = m->cfg;
  size_t need = 0;
  for (int t0 = 0; t0 < n; t0 += m->pg_rows) {
    const int T = std::min(n - t0, m->pg_rows);
    const size_t b = pa_pays(T, pos0 + t0) ? pa_bytes(c, pos0 + t0 + T) : 0;
    if (b <= KH_PA_WS_MAX) need = std::max(need, b);
  }
  if (need <= m->pa_ws_bytes) return;
  const size_t most = std::min(KH_PA_WS_MAX, pa_bytes(c, c.cache_len)), twice = std::min(std::max(need, 2 * m->pa_ws_bytes), most);
  if (m->pa_ws) (void)hipFree(m->pa_ws);
  m->pa_ws = nullptr;
  m->pa_ws_bytes = 0;
  for (size_t b : {twice, need}) {
    if (dalloc(&m->pa_ws, b) == KH_OK) {
      m->pa_ws_bytes = b;
      return;
    }
    (void)hipGetLastError();
    m->pa_ws = nullptr;
  }
}
namespace {
bool pair_attention(kh_model* m, int l, int T, int pos0) {
  const kh_config& c = m->cfg;
  const size_t need = pa_bytes(c, pos0 + T);
  if (!pa_pays(T, pos0) || need == 0 || need > m->pa_ws_bytes) return false;
  KhPaArgs a{};
  a.blocks = (pos0 + T + 31) / 32;
  a.q = m->pg_q;
  a.kc = m->kcache + (size_t)l * c.cache_len * c.kv_dim;
  a.vc = m->vcache + (size_t)l * c.cache_len * c.kv_dim;
  a.slab = m->pa_ws;
  a.inv = (float*)(m->pa_ws + need - 2 * (size_t)c.kv_head_num * a.blocks * sizeof(float));
  a.out = m->pg_att;
  a.out_e = m->pg_ae;
  a.stage = KH_PAIR_STAGE(c.is_quant);
  a.tcap = m->pg_rows;
  a.dim = c.dim; a.kv_dim = c.kv_dim; a.kv_heads = c.kv_head_num; a.kv_mul = c.kv_mul; a.T = T; a.pos0 = pos0;
  switch (c.head_size) {
    case 48: pa_go<48, 2>(a, m->stream); break;
    case 64: pa_go<64, 2>(a, m->stream); break;
    default: pa_go<128, 1>(a, m->stream); break;
  }
  return true;
}
}  // namespace

// forward of T (<= pg_rows) prompt tokens at positions pos0..: fills their K/V cache rows.  last: logits are taken from the last
// token's row in front of the last layer
int launch_prefill_pair_chunk(kh_model* m, const int32_t* toks, int T, int pos0, bool last) {
  const kh_config& c = m->cfg;
  int rc;
  if ((rc = kh_embedding_f32_host(toks, T, m->tok_emb, m->pg_x, c.dim, c.vocab_size, (void*)m->stream)) != KH_OK) return rc;
  char *xn = (char*)m->pg_xn, *h = (char*)m->pg_h;  // pair slabs: four bytes a number, like the fp32 slabs
  int fine = 0;
  int kz = 0;  // K slices of the last residual GEMM still to be added to pg_x
  const bool rope_fuse = !dbg_off("KH_PG_ROPE_FUSE");
  for (int l = 0; l < c.layer_num; ++l) {
    const LayerW& W = m->layers[l];
    auto rmsnorm = [&](const float* w) {
      hipLaunchKernelGGL(k_pair_rmsnorm, dim3(T), dim3(KH_WG), 0, m->stream, m->pg_x, w, xn, m->pg_xs, c.dim, c.rms_eps, T,
                         (const float*)m->pg_part, kz);
      kz = 0;
    };
    KhPairArgs base{};
    base.T = T;
    base.pos0 = pos0;
    base.tcap = T;
    base.keep = last && l < c.layer_num - 1;
    base.xe_ld = m->pg_rows;
    base.xs = m->pg_xs;
    base.part = m->pg_part;
    base.head_size = c.head_size;
    base.sin_cache = m->sin_cache;
    base.cos_cache = m->cos_cache;
    rmsnorm(W.att_norm);
    {
      KhPairArgs a = base;
      a.w[0] = W.wq; a.w[1] = W.wk; a.w[2] = W.wv;
      a.X = xn; a.out = m->pg_q;
      a.kc = m->kcache + (size_t)l * c.cache_len * c.kv_dim;
      a.vc = m->vcache + (size_t)l * c.cache_len * c.kv_dim;
      a.rows0 = l == c.layer_num - 1 ? 0 : c.dim;  // nobody asks for the last layer's queries
      a.rows1 = c.kv_dim; a.N = a.rows0 + 2 * c.kv_dim; a.ldo = c.dim; a.K = c.dim;
      a.rope = !rope_fuse ? KH_PG_ROPE_OFF
               : (c.rope_mode == KH_ROPE_HALF ? (c.head_size % 32 == 0 ? KH_PG_ROPE_TILES : KH_PG_ROPE_OFF) : KH_PG_ROPE_PAIRS);
      if ((rc = pair_launch<KH_PG_QKV>(m, a, nullptr)) != KH_OK) return rc;
      if (a.rope == KH_PG_ROPE_OFF)
        hipLaunchKernelGGL(k_pg_rope, dim3(T), dim3(KH_WG), 0, m->stream, m->pg_q, a.kc, m->sin_cache, m->cos_cache, a.rows0, c.kv_dim,
                           c.head_size, pos0, c.rope_mode);
    }
    // the prompt phase leaves K/V rows and nothing else: the last layer's attention, wo and feed-forward feed nothing
    if (l == c.layer_num - 1) break;
    // the attention kernels leave pairs where 64 columns are of one head
    bool pairs = c.head_size % 64 == 0;
    if (!pair_attention(m, l, T, pos0)) pairs = pg_slice_attention(m, l, T, pos0, pairs ? KH_PA_PAIRS : KH_PA_ROWS, m->pg_rows);
    if (!pairs) hipLaunchKernelGGL(k_pair_convert, dim3(T), dim3(KH_WG), 0, m->stream, (const float*)m->pg_att, xn, m->pg_ae, c.dim, m->pg_rows,
                                   KH_PAIR_STAGE(c.is_quant) / 4);
    {
      KhPairArgs a = base;
      a.w[0] = W.wo;
      a.X = pairs ? (const char*)m->pg_att : xn; a.xe = m->pg_ae; a.out = m->pg_x;
      a.rows0 = a.N = a.ldo = a.K = c.dim;
      if ((rc = pair_launch<KH_PG_RESID>(m, a, &kz)) != KH_OK) return rc;
    }
    rmsnorm(W.ffn_norm);
    {
      KhPairArgs a = base;
      a.w[0] = W.w1; a.w[1] = W.w3;
      a.X = xn; a.pairs = h; a.out_e = m->pg_he;
      a.rows0 = c.hidden_dim; a.N = 2 * c.hidden_dim; a.ldo = c.hidden_dim; a.K = c.dim;
      if ((rc = pair_launch<KH_PG_SWIGLU>(m, a, nullptr, &fine)) != KH_OK) return rc;
    }
    {
      KhPairArgs a = base;
      a.w[0] = W.w2;
      a.X = h; a.xe = m->pg_he; a.fine = fine; a.out = m->pg_x;
      a.rows0 = a.N = a.ldo = c.dim; a.K = c.hidden_dim;
      if ((rc = pair_launch<KH_PG_RESID>(m, a, &kz)) != KH_OK) return rc;
    }
  }
  return kh_launch_status();
}
}  // namespace khm
