// kh_pattn_pair.h — causal attention of a prompt slice on the fp16 matrix cores, operands kept to 32-bit accuracy as pairs
// of halves (kh_pair.h; reference: cpu/mha_kernel.cpp:5-61, cuda/mha_kernel.cu:47-110, one query token at a time).
//
// k_pa_pack first lays this layer's K and V rows 0 .. pos0 + T - 1 out as pairs in the order of the MFMA fragments: blocks
// of 32 positions, every fragment 64 lanes x 16 bytes, so that the attention reads nothing but whole kilobytes.  The K and
// the V part of a block carry a scale each, from the largest finite number in it (a row that is not finite must not take the
// bits of the positions in front of it).  Nothing is kept from one pass to the next and nothing is assumed of the cache.
//
// k_pa_attn: one workgroup owns (head, QT x 16 query tokens), its NW waves split the 32-position blocks:
//   S^T[pos, tok] = K . Q^T         rows of the two 16-row tiles u are positions 8 (i >> 2) + 4 u + (i & 3), so that a lane
//                                   ends with eight consecutive positions 8 (l >> 4) .. + 7 of its token l & 15:
//   O^T[d, tok]  += V^T . P^T       the B operand of v_mfma_f32_16x16x32_f16 as it stands
// Products lo hi, hi lo, hi hi in this order, so the sum is rounded at its full size only in the last ones.  Online softmax
// in the log2 domain as in kh_pattn.h.  The matrix core rounds sums down, which would not average out over thousands of
// positions and shifts scores by their size: half of a score's columns are summed with the sign turned (kh_pattn.h), a block's P V starts from zero, is added to O in fp32 (times 1 / the block's scale), and every second block of a
// wave carries -P.
//
// Q is split once per workgroup and kept in LDS; K and V of the next block are requested when the last product of the
// present one has read them: held twice they would not leave room for two waves per SIMD, which cover one another's softmax.
// Bound by the softmax and the matrix cores about evenly.  Two query tiles for heads of 48 and 64 (one was 2 % slower over a
// whole prompt of 1899 tokens of TinyLlama, four 0.3 %, with fewer workgroups for short prompts; eight waves instead of four
// 2 %), one for 128 (two spill).  Attention of one layer, us, fp32 matrix cores -> pack + attention: TinyLlama, 1899 tokens
// 187 -> 5.1 + 70; Llama-2-7B, 776 tokens 106 -> 10.8 + 40; Llama-3.2-1B, 512 tokens 23.5 -> 5.0 + 11.5.
#pragma once
#include "kh_pair.h"

struct KhPaArgs {
  const float* q;      // [T][dim], RoPE applied
  const float* kc;     // this layer's cache rows [cache_len][kv_dim]
  const float* vc;
  char* slab;          // [kv_heads][blocks][KF + VF] fragments of 1 KB
  float* inv;          // [kv_heads][blocks] 1 / scale of K, of V
  float* out;          // heads of 64 and 128: rows of pairs [T][dim], else of fp32
  unsigned char* out_e;  // 1 / the scales of the pairs, for tcap tokens
  int stage;           // columns of a stage of the GEMM that reads them
  int dim, kv_dim, kv_heads, kv_mul, T, pos0, blocks, tcap;
};
template <int HS>
struct PaGeom {
  static constexpr int NC = (HS + 31) / 32, ND = HS / 16;    // 32-column chunks of a K row, 16-column tiles of a V row
  static constexpr int KF = 4 * NC, VF = 2 * ND, FR = KF + VF;  // fragments: K [NC][hi, lo][u], V [ND][hi, lo]
};
__device__ __forceinline__ void pa_split(const float (&v)[8], float s, f16x8& hi, f16x8& lo) {
#pragma unroll
  for (int i = 0; i < 8; i += 2) {
    const float a = v[i] * s, b = v[i + 1] * s;
    const f16x2 h = pair_cvt(a, b), l = pair_cvt(a - (float)h[0], b - (float)h[1]);
    hi[i] = h[0]; hi[i + 1] = h[1];
    lo[i] = l[0]; lo[i + 1] = l[1];
  }
}

// |v|, zero for infinities and NaN
__device__ __forceinline__ float pa_finite(float v) { return fabsf(v) < INFINITY ? fabsf(v) : 0.f; }
// one workgroup of four waves per (block of 32 positions, kv head); positions past the slice become zeros
template <int HS>
__global__ __launch_bounds__(256) void k_pa_pack(const KhPaArgs a) {
  using G = PaGeom<HS>;
  constexpr int KT = (2 * G::NC + 3) / 4, VT = (G::ND + 3) / 4;
  __shared__ float top_lds[2][4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 15, lj = lane >> 4;
  const int blk = blockIdx.x, g = blockIdx.y, p0 = blk * 32, n = a.pos0 + a.T;
  char* dst = a.slab + ((size_t)g * a.blocks + blk) * G::FR * 1024 + lane * 16;
  float kv[KT][8], vv[VT][8], top = 0.f, vtop = 0.f;
#pragma unroll
  for (int k = 0; k < KT; ++k) {
    const int task = wave + 4 * k, u = task & 1, d = (task >> 1) * 32 + 8 * lj;
    const int p = p0 + 8 * (li >> 2) + 4 * u + (li & 3);
    const bool in = p < n && d < HS;
    const float* r = a.kc + (size_t)(in ? p : 0) * a.kv_dim + g * HS + (in ? d : 0);
    const f32x4 x = *(const f32x4*)r, y = *(const f32x4*)(r + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      kv[k][e] = in ? x[e] : 0.f;
      kv[k][e + 4] = in ? y[e] : 0.f;
      top = fmaxf(top, fmaxf(pa_finite(kv[k][e]), pa_finite(kv[k][e + 4])));
    }
  }
#pragma unroll
  for (int k = 0; k < VT; ++k) {
    const int d = (wave + 4 * k) * 16 + li;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int p = p0 + 8 * lj + e;
      const bool in = p < n && d < HS;
      const float x = a.vc[(size_t)(in ? p : 0) * a.kv_dim + g * HS + (in ? d : 0)];
      vv[k][e] = in ? x : 0.f;
      vtop = fmaxf(vtop, pa_finite(vv[k][e]));
    }
  }
  for (int o = 32; o; o >>= 1) {
    top = fmaxf(top, __shfl_xor(top, o));
    vtop = fmaxf(vtop, __shfl_xor(vtop, o));
  }
  if (lane == 0) {
    top_lds[0][wave] = top;
    top_lds[1][wave] = vtop;
  }
  __syncthreads();
  auto scale = [&](const float(&t)[4]) { return pair_scale(fmaxf(fmaxf(t[0], t[1]), fmaxf(t[2], t[3]))); };
  const float s = scale(top_lds[0]), vs = scale(top_lds[1]);
  if (threadIdx.x == 0) *(float2*)(a.inv + 2 * ((size_t)g * a.blocks + blk)) = make_float2(pair_inv(s), pair_inv(vs));
  f16x8 hi, lo;
#pragma unroll
  for (int k = 0; k < KT; ++k) {
    const int task = wave + 4 * k, c = task >> 1, u = task & 1;
    if (c < G::NC) {
      pa_split(kv[k], s, hi, lo);
      *(f16x8*)(dst + ((c * 2 + 0) * 2 + u) * 1024) = hi;
      *(f16x8*)(dst + ((c * 2 + 1) * 2 + u) * 1024) = lo;
    }
  }
#pragma unroll
  for (int k = 0; k < VT; ++k) {
    const int dt = wave + 4 * k;
    if (dt < G::ND) {
      pa_split(vv[k], vs, hi, lo);
      *(f16x8*)(dst + (G::KF + dt * 2 + 0) * 1024) = hi;
      *(f16x8*)(dst + (G::KF + dt * 2 + 1) * 1024) = lo;
    }
  }
}

template <int HS, int NW, int QT>
__global__ __launch_bounds__(64 * NW, 2) void k_pa_attn(const KhPaArgs a) {
  using G = PaGeom<HS>;
  constexpr int LDO = HS + 4;
  __shared__ __attribute__((aligned(16))) float o_lds[NW][16][LDO];
  __shared__ __attribute__((aligned(16))) char q_lds[QT][G::NC * 2][1024];
  __shared__ float qs_lds[QT][16], m_lds[NW][16], l_lds[NW][16];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, lj = lane >> 4;
  // workgroup -> (kv group, head in it, token tile): heads and tiles that share K / V share an XCD's L2; long tiles first
  const int b = (int)blockIdx.x, g = b % a.kv_heads, rest = b / a.kv_heads;
  const int h = g * a.kv_mul + rest % a.kv_mul;
  const int n_tt = (a.T + 16 * QT - 1) / (16 * QT);
  const int t0 = (n_tt - 1 - rest / a.kv_mul) * 16 * QT;
  const int t_last = t0 + 16 * QT - 1 < a.T - 1 ? t0 + 16 * QT - 1 : a.T - 1;
  const int n_pb = ((a.pos0 + t_last) >> 5) + 1;
  const char* base = a.slab + (size_t)g * a.blocks * G::FR * 1024;  // uniform: fragments are read at scalar base + lane
  const unsigned lane16 = lane * 16;
  const float* inv = a.inv + 2 * (size_t)g * a.blocks;

  f16x8 kf[G::KF], vf[G::VF];
  float ki = 1.f, vi = 1.f;
  auto load_k = [&](int pb) __attribute__((always_inline)) {
    const char* s = base + (size_t)pb * G::FR * 1024;
#pragma unroll
    for (int i = 0; i < G::KF; ++i) kf[i] = *(const f16x8*)(s + i * 1024 + lane16);
    ki = inv[2 * pb];
  };
  auto load_v = [&](int pb) __attribute__((always_inline)) {
    const char* s = base + ((size_t)pb * G::FR + G::KF) * 1024;
#pragma unroll
    for (int i = 0; i < G::VF; ++i) vf[i] = *(const f16x8*)(s + i * 1024 + lane16);
    vi = inv[2 * pb + 1] * 0x1p-14f;  // P is scaled by 2^14
  };
  if (wave < n_pb) {
    load_k(wave);
    load_v(wave);
  }
  // query tile qi: column l & 15 of both products (columns past the slice repeat its last token); a scale per token
  for (int qi = wave; qi < QT; qi += NW) {
    const int t = t0 + 16 * qi + li, tq = t < a.T ? t : a.T - 1;
    const float* row = a.q + (size_t)tq * a.dim + (size_t)h * HS;
    float v[G::NC][8], top = 0.f;
#pragma unroll
    for (int c = 0; c < G::NC; ++c) {
      const int d = 32 * c + 8 * lj;
      const bool in = d < HS;
      const f32x4 x = *(const f32x4*)(row + (in ? d : 0)), y = *(const f32x4*)(row + (in ? d : 0) + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[c][e] = in ? x[e] : 0.f;
        v[c][e + 4] = in ? y[e] : 0.f;
        top = fmaxf(top, fmaxf(fabsf(v[c][e]), fabsf(v[c][e + 4])));
      }
    }
    top = fmaxf(top, __shfl_xor(top, 16));
    top = fmaxf(top, __shfl_xor(top, 32));
    const float s = pair_scale(top);
#pragma unroll
    for (int c = 0; c < G::NC; ++c) {
      f16x8 hi, lo;
      pa_split(v[c], 2 * c < G::NC ? s : -s, hi, lo);
      *(f16x8*)&q_lds[qi][2 * c][lane * 16] = hi;
      *(f16x8*)&q_lds[qi][2 * c + 1][lane * 16] = lo;
    }
    if (lj == 0) qs_lds[qi][li] = pair_inv(s) * ((1.0f / sqrtf((float)HS)) * 1.4426950408889634f);
  }
  __syncthreads();

  const f32x4 zero4 = {0.f, 0.f, 0.f, 0.f};
  float m[QT], l[QT], qs[QT];
  f32x4 o[QT][G::ND];
#pragma unroll
  for (int qi = 0; qi < QT; ++qi) {
    m[qi] = -INFINITY;
    l[qi] = 0.f;
    qs[qi] = qs_lds[qi][li];
#pragma unroll
    for (int d = 0; d < G::ND; ++d) o[qi][d] = zero4;
  }
  auto block = [&](int pb, auto odd) __attribute__((always_inline)) {
    constexpr float PS = decltype(odd)::value ? -16384.f : 16384.f;  // p <= 1
    const int next = pb + NW;
    const float ki0 = ki, vi0 = decltype(odd)::value ? -vi : vi;
#pragma unroll
    for (int qi = 0; qi < QT; ++qi) {
      const int first = a.pos0 + t0 + 16 * qi;        // position of the tile's first token
      if (qi < QT - 1 && pb * 32 > first + 15) continue;  // wholly above the diagonal (never the last tile)
      int at = lane * 16;
      if constexpr (HS > 64) asm volatile("" : "+v"(at));  // or all of Q is kept in registers across the blocks, and they spill
      f32x4 sa[2] = {zero4, zero4}, sb[2] = {zero4, zero4};
#pragma unroll
      for (int c = 0; c < G::NC; ++c) {
        const f16x8 qh = *(const f16x8*)&q_lds[qi][2 * c][at], ql = *(const f16x8*)&q_lds[qi][2 * c + 1][at];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          f32x4& t = 2 * c < G::NC ? sa[u] : sb[u];
          t = mfma_pair(kf[(c * 2 + 1) * 2 + u], qh, t);
          t = mfma_pair(kf[c * 4 + u], ql, t);
        }
      }
#pragma unroll
      for (int c = 0; c < G::NC; ++c) {
        const f16x8 qh = *(const f16x8*)&q_lds[qi][2 * c][at];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          f32x4& t = 2 * c < G::NC ? sa[u] : sb[u];
          t = mfma_pair(kf[c * 4 + u], qh, t);
        }
      }
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int r = 0; r < 4; ++r) sa[u][r] -= sb[u][r];
      if (qi == QT - 1 && next < n_pb) load_k(next);
      if (pb * 32 + 31 > first) {
        const int my = first + li, p = pb * 32 + 8 * lj;
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int r = 0; r < 4; ++r) sa[u][r] = p + 4 * u + r <= my ? sa[u][r] : -INFINITY;
      }
      const float kq = __builtin_amdgcn_fmed3f(ki0 * qs[qi], 0x1p-126f, 0x1p127f);  // 0 would make NaNs of the masked scores
      float tm = fmaxf(fmaxf(fmaxf(sa[0][0], sa[0][1]), fmaxf(sa[0][2], sa[0][3])),
                       fmaxf(fmaxf(sa[1][0], sa[1][1]), fmaxf(sa[1][2], sa[1][3])));
      tm = fmaxf(tm, __shfl_xor(tm, 16));
      tm = fmaxf(tm, __shfl_xor(tm, 32));
      const float m_new = fmaxf(m[qi], tm * kq);
      const float m_ref = m_new == -INFINITY ? 0.f : m_new;  // a token that has seen no position yet
      const float alpha = __builtin_amdgcn_exp2f(m[qi] - m_ref);
      m[qi] = m_new;
      float p[8], sum = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        p[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(sa[e >> 2][e & 3], kq, -m_ref));
        sum += p[e];
      }
      l[qi] = __builtin_fmaf(l[qi], alpha, sum);
      f16x8 ph, pl;
      pa_split(p, PS, ph, pl);
#pragma unroll
      for (int d = 0; d < G::ND; ++d) {
        f32x4 t = mfma_pair(vf[2 * d + 1], ph, zero4);
        t = mfma_pair(vf[2 * d], pl, t);
        t = mfma_pair(vf[2 * d], ph, t);
#pragma unroll
        for (int r = 0; r < 4; ++r) o[qi][d][r] = __builtin_fmaf(t[r], vi0, o[qi][d][r] * alpha);
      }
    }
    if (next < n_pb) load_v(next);
  };
  for (int pb = wave; pb < n_pb; pb += 2 * NW) {
    block(pb, std::false_type{});
    if (pb + NW < n_pb) block(pb + NW, std::true_type{});
  }

  // merge the waves' partials in fixed order, one query tile at a time
#pragma unroll
  for (int qi = 0; qi < QT; ++qi) {
    if (qi > 0) __syncthreads();
    float lq = l[qi];
    lq += __shfl_xor(lq, 16);
    lq += __shfl_xor(lq, 32);
    if (lj == 0) {
      m_lds[wave][li] = m[qi];
      l_lds[wave][li] = lq;
    }
#pragma unroll
    for (int d = 0; d < G::ND; ++d) *(f32x4*)&o_lds[wave][li][16 * d + 4 * lj] = o[qi][d];
    __syncthreads();
    constexpr bool pairs = HS % 64 == 0;  // the 16 chunks of 64 columns in neighbouring lanes
    const int tok = pairs ? (tid >> 4) & 15 : tid & 15, t = t0 + 16 * qi + tok;
    if (t < a.T) {
      float M = m_lds[0][tok];
#pragma unroll
      for (int w = 1; w < NW; ++w) M = fmaxf(M, m_lds[w][tok]);  // finite: a token sees its own position
      float f[NW], L = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        f[w] = __builtin_amdgcn_exp2f(m_lds[w][tok] - M);
        L += f[w] * l_lds[w][tok];
      }
      for (int grp = pairs ? (tid >> 8) * 16 + (tid & 15) : tid >> 4; grp < HS / 4; grp += 4 * NW) {
        f32x4 r = zero4;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
          const f32x4 x = *(const f32x4*)&o_lds[w][tok][4 * grp];
#pragma unroll
          for (int e = 0; e < 4; ++e) r[e] += f[w] * x[e];
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) r[e] /= L;
        const int k = h * HS + 4 * grp;
        if constexpr (pairs) pair_emit((char*)a.out + (size_t)t * a.dim * 4, a.out_e, a.tcap, t, k >> 2, a.dim >> 2, a.stage >> 2, r);
        else *(f32x4*)(a.out + (size_t)t * a.dim + k) = r;
      }
    }
  }
}
