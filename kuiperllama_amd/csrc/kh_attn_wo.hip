// kh_attn_wo.hip - launches of kh_attn_wo.h: attention and the output projection of a decoded token in one launch.
#include "kh_attn_wo.h"

#include <stdlib.h>

#include <algorithm>

#include "kh_model_internal.h"

namespace khm {

// Which models take it, and in what shape.  fp32 weights; at most eight key / value groups of at most 512 columns (two float4 a
// lane, ten heads), head sizes that the attention is instantiated for, vectors that two float4 a thread cover: every group is
// one vector more that k_ffn13_parts stages (eight of 2048 floats cost it 0.9 us), and its keys and values are read by every
// slice.  At most 2048 columns, whatever the threads of ffn13: k_pf_wo_parts keeps eight tokens' vectors in 64 KB.  us a launch at
// position 48, attention + wo -> one launch | ffn13: Llama-3.2-1B 3.4 + 4.5 -> 5.0 | 21.3 -> 22.2;
// TinyLlama 3.3 + 4.5 -> 4.9 | 15.5 -> 15.9; Qwen2.5-0.5B 3.4 + 2.6 -> 4.2 | 6.95 -> 7.15; stories15M 3.6 + 2.3 -> 3.9 | 2.4 -> 2.75.
// A token: -3.9 / -6.1 / -8.4 / -12 %; with 200 - 240 positions -2 / -2.4 / -1.9 / -3 %.  From KH_ATTN_MIN_TS on attention is split over time.
namespace {
// Positions below which the joint launch is the faster form.  Its time grows by some 1 us a layer from position 48 to 127 and by 0.4
// more with the second tile a wave, for every slice reads its group's keys and values; what it saves is 1.3 - 2 us, less 0.1 a
// part in ffn13, and up to 1 us more where wo has 1536 rows.  Slices of a part run on 8 / gcd(parts, 8) of the XCDs: 3, 5 and 7 parts
// bring their keys into all of them.  `staged`: floats of parts that the workgroups of ffn13 read; from 1536 columns on they decide.
// Fitted to 85 geometries at eight positions, each as a model of 8 layers and as one of 18 - 24, which gain more behind position 100.
// Per cent of a step saved at position 16 / 80 / 144 / 208 (head size x heads - groups; 1 % from one instance of a model to the next):
//                             8 layers                   18 - 24 layers
//   48 x 6-6 (stories15M)     11.9   7.0   4.1   2.5     12.7   4.6   0.9   1.8
//   48 x 15-5                  8.3   4.8   1.6  -0.8      9.2   5.0   4.5   4.5
//   48 x 24-6                  1.8  -0.3  -1.0  -1.3      2.2   0.8  -0.9  -1.6
//   48 x 28-7                  0.8  -1.6  -2.9  -2.1      0.6   0.1  -1.3  -1.6
//   48 x 24-8                 -1.9  -4.3  -6.0  -6.5     -1.2  -3.0  -4.0  -4.6
//   64 x 12-3                 10.2   5.1   2.5  -0.2     10.9   4.3   3.4   3.2
//   64 x 16-4                  7.0   2.2  -0.6  -2.0      8.0   4.0   2.0   0.8
//   64 x 15-5                  6.5   2.4  -3.2  -3.3      6.3   3.3   1.2   0.3
//   64 x 12-6                  8.3   3.7   0.6  -1.3      8.6   3.0   1.7   1.2
//   64 x 18-6                  1.7  -1.0  -3.5  -4.4      2.6   0.8  -1.6  -2.6
//   64 x 14-7                  5.4  -0.9  -4.1  -4.1      5.0   1.8   0.4  -0.3
//   64 x 8-8                  10.5   4.9   1.2   0.1     10.6   4.9   2.7   1.5
//   64 x 16-8                  4.9   0.5  -2.7  -3.6      5.6   2.1   0.1  -1.0
//   64 x 24-8, 3072 hidden     3.8   0.6  -1.5  -2.3      4.0   1.3  -0.4  -0.4    9.4 million staged
//   64 x 32-8, 4096            1.8  -0.4  -1.1  -2.3      2.0   0.0  -0.4  -0.9   16.8 million
//   64 x 32-8, 8192            3.6   1.9   1.1   0.3      5.0   3.2   2.5   2.0    8.4 million (Llama-3.2-1B)
// Mean of positions 0 - 255 over all 85: 3.3 and 4.2 %; with 256 for all of them 3.0 and 4.1, 19 of them slower at some position.
int joint_end(int dim, int head_size, int parts, long staged) {
  if (dim >= 1536) return staged <= 8750000 ? 256 : (staged <= 11000000 ? 128 : 64);
  const bool wide = dim >= 1024;
  if (head_size == 48) return !wide || parts <= 5 ? 256 : (parts == 6 ? 128 : (parts == 7 ? 64 : 0));
  switch (parts) {
    case 4: return wide ? 192 : 256;
    case 5: return 128;
    case 6: return wide ? 64 : 192;
    case 7: return wide ? 64 : 128;
    case 8: return wide ? 128 : 256;
    default: return 256;
  }
}
}  // namespace
kh_model::AttnWoPlan plan_attn_wo(const kh_config& c, const kh_model::Shape& ffn, int t_long) {
  kh_model::AttnWoPlan p;
  const int hs = c.head_size, cols = c.kv_mul * hs, mv = kh_stage_maxv(c.dim, ffn.wg);
  if (c.is_quant || (hs != 48 && hs != 64)) return p;
  if (c.kv_head_num > KH_AWO_PARTS_MAX || cols > 512 || c.dim != c.head_num * hs || mv < 1 || mv > 2) return p;
  if ((size_t)KH_PF_BMAX * c.dim * sizeof(float) > (64u << 10)) return p;
  p.parts = c.kv_head_num;
  p.cols4 = cols / 4;
  p.lpr = p.cols4 <= 16 ? 16 : (p.cols4 <= 32 ? 32 : 64);
  p.nu = (p.cols4 + p.lpr - 1) / p.lpr;
  const int rows = KH_AWO_WAVES * (64 / p.lpr);
  auto slices = [&](int rw) { return (c.dim + rows * rw - 1) / (rows * rw); };
  // the most rows a workgroup (its attention is the same for few) that leave three quarters of the CUs with one, or fewer CUs
  // where half as many rows would be more than one workgroup a CU: sixteen waves of up to 115 registers are alone there, and two
  // rounds take 7.8 instead of 5.6 us (Llama-3.2-1B).  256 steps of 8 layers, 288 / 144 workgroups: 768 columns, 12-6 heads 45.8 / 39.8
  // ms, 1536, 24-3 heads 72.4 / 65.0; apart 40.6 and 67.0
  for (p.rw = p.lpr == 64 ? 8 / p.nu : 2; p.rw > 1 && p.parts * slices(p.rw) < 192 && p.parts * slices(p.rw / 2) <= 256;) p.rw /= 2;
  p.slices = slices(p.rw);
  if (p.parts * p.slices > 256) return kh_model::AttnWoPlan{};
  p.lds = attn_wo_lds_bytes(hs, c.kv_mul);
  const char* hook = dbg("KH_ATTN_WO");
  const int pays = hook ? atoi(hook) : joint_end(c.dim, hs, p.parts, (long)ffn.grid * p.parts * c.dim);
  p.end = std::min(pays, std::min(KH_ATTN_MIN_TS, t_long - 1));  // one split, and no group path
  return p.end > 0 ? p : kh_model::AttnWoPlan{};
}

namespace {
KhAttnWoArgs attn_args(kh_model* m, int l) {
  const kh_config& c = m->cfg;
  KhAttnWoArgs a{};
  a.kcache_layer = m->kcache + (size_t)l * c.cache_len * c.kv_dim;
  a.vcache_layer = m->vcache + (size_t)l * c.cache_len * c.kv_dim;
  a.wo = (const float*)m->layers[l].wo.w;
  a.dim = c.dim;
  a.kv_dim = c.kv_dim;
  a.kv_mul = c.kv_mul;
  return a;
}
template <int DN>
void go(const kh_model::AttnWoPlan& p, hipStream_t s, const KhAttnWoArgs& a) {
  auto l = [&](auto k) { hipLaunchKernelGGL(k, dim3(p.parts, p.slices), dim3(128 * KH_AWO_WAVES), p.lds, s, a); };
  if (p.lpr == 16) p.rw == 2 ? l(k_attn_wo<DN, 16, 1, 2>) : l(k_attn_wo<DN, 16, 1, 1>);
  else if (p.lpr == 32) p.rw == 2 ? l(k_attn_wo<DN, 32, 1, 2>) : l(k_attn_wo<DN, 32, 1, 1>);
  else if (p.nu == 2) p.rw == 4 ? l(k_attn_wo<DN, 64, 2, 4>) : p.rw == 2 ? l(k_attn_wo<DN, 64, 2, 2>) : l(k_attn_wo<DN, 64, 2, 1>);
  else if (p.rw >= 4) p.rw == 8 ? l(k_attn_wo<DN, 64, 1, 8>) : l(k_attn_wo<DN, 64, 1, 4>);
  else p.rw == 2 ? l(k_attn_wo<DN, 64, 1, 2>) : l(k_attn_wo<DN, 64, 1, 1>);
}
}  // namespace

void launch_attn_wo(kh_model* m, int l) {
  KhAttnWoArgs a = attn_args(m, l);
  a.q = m->q;
  a.d_pos = m->d_pos;
  a.out = m->wo_part;
  if (m->cfg.head_size == 48) go<3>(m->awo, m->stream, a);
  else go<4>(m->awo, m->stream, a);
}

void launch_ffn13_parts(kh_model* m, const KhFfn13Args& f) {
  KhFfn13PartsArgs a{f, m->wo_part, m->x1, m->awo.parts};
  const int wg = m->sh_ffn.wg, mv = kh_stage_maxv(f.dim, wg), pn = (m->awo.parts + 1) / 2;
  auto l = [&](auto k) { hipLaunchKernelGGL(k, dim3(m->sh_ffn.grid), dim3(wg), fused_lds_bytes(false, f.dim), m->stream, a); };
  auto by_parts = [&](auto u, auto v) {
    constexpr int U = decltype(u)::value, MV = decltype(v)::value;
    if (pn == 1) l(k_ffn13_parts<U, MV, 2>);
    else if (pn == 2) l(k_ffn13_parts<U, MV, 4>);
    else if (pn == 3) l(k_ffn13_parts<U, MV, 6>);
    else l(k_ffn13_parts<U, MV, 8>);
  };
  auto by_depth = [&](auto u) {
    if (mv == 1) by_parts(u, std::integral_constant<int, 1>{});
    else by_parts(u, std::integral_constant<int, 2>{});
  };
  if (m->sh_ffn.u >= 8) by_depth(std::integral_constant<int, 8>{});
  else if (m->sh_ffn.u >= 4) by_depth(std::integral_constant<int, 4>{});
  else by_depth(std::integral_constant<int, 2>{});
}

void launch_pf_attn_parts(kh_model* m, int l, int nvalid, int pos0) {
  KhAttnWoArgs a = attn_args(m, l);
  a.q = m->pf_q;
  a.out = m->pf_att;
  a.pos0 = pos0;
  auto go = [&](auto k) { hipLaunchKernelGGL(k, dim3(m->awo.parts, nvalid), dim3(64 * KH_AWO_WAVES), m->awo.lds, m->stream, a); };
  if (m->cfg.head_size == 48) go(k_pf_attn_parts<3>);
  else go(k_pf_attn_parts<4>);
}
void launch_pf_wo_parts(kh_model* m, int l, int nvalid) {
  const kh_model::AttnWoPlan& p = m->awo;
  KhPfWoPartsArgs a{m->pf_att, (const float*)m->layers[l].wo.w, m->pf_x, m->cfg.dim, p.parts, p.cols4, nvalid};
  const int rows = KH_AWO_WAVES * (64 / p.lpr), lds = nvalid * m->cfg.dim * 4;  // at most 64 KB: plan_attn_wo
  auto go = [&](auto k) {
    hipLaunchKernelGGL(k, dim3((m->cfg.dim + rows - 1) / rows), dim3(64 * KH_AWO_WAVES), lds, m->stream, a);
  };
  if (p.lpr == 16) go(k_pf_wo_parts<16, 1>);
  else if (p.lpr == 32) go(k_pf_wo_parts<32, 1>);
  else if (p.nu == 1) go(k_pf_wo_parts<64, 1>);
  else go(k_pf_wo_parts<64, 2>);
}
}  // namespace khm

extern "C" int kh_plan_attn_wo(int32_t dim, int32_t hidden_dim, int32_t head_num, int32_t kv_head_num, int32_t seq_len, int32_t is_quant,
                               int32_t* out4) {
  if (!out4 || dim <= 0 || hidden_dim <= 0 || head_num <= 0 || kv_head_num <= 0 || head_num % kv_head_num || dim % head_num || seq_len <= 0)
    return KH_ERR_INVALID_ARG;
  kh_config c{};
  c.dim = dim;
  c.hidden_dim = hidden_dim;
  c.head_num = head_num;
  c.kv_head_num = kv_head_num;
  c.kv_mul = head_num / kv_head_num;
  c.head_size = dim / head_num;
  c.kv_dim = c.head_size * kv_head_num;
  c.is_quant = is_quant;
  kh_model::Shape sh[5];
  khm::plan_decode_shapes(is_quant != 0, dim, hidden_dim, c.kv_dim, dim, sh);
  int32_t at[8];
  const int rc = kh_plan_attention(head_num, c.kv_mul, c.head_size, seq_len, 0, at);
  if (rc != KH_OK) return rc;
  const kh_model::AttnWoPlan p = khm::plan_attn_wo(c, sh[2], at[3]);
  out4[0] = p.end > 0 ? p.end : 0;
  out4[1] = p.end > 0 ? p.parts : 0;
  out4[2] = p.end > 0 ? KH_AWO_WAVES * (64 / p.lpr) * p.rw : 0;
  out4[3] = p.end > 0 ? p.parts * p.slices : 0;
  return KH_OK;
}
