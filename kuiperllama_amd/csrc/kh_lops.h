// kh_lops.h — per-token kernels of the layer-list models: embedding, the residual update fused with the one or two norms
// of a parallel block (layer norm or RMS norm), the causal convolution.  Everything that touches the residual stream is fp32.
#pragma once
#include "kh_tile.h"

namespace khm {

// Tables of one pass: T tokens of up to S sequences, concatenated.  All arrays live on the device.
struct PassTabs {
  const int32_t *tok, *pos, *seg;              // [T]: token id, position in its sequence, segment
  const int32_t *seg_slot, *seg_row0, *seg_n, *seg_pos0;  // [S]: state slot, first row, rows, position of the first row
};

// what one layer leaves to be added to the residual stream
template <class T>
struct AddArgs {
  const float* mix;       // [T][ld] mixer output (nullptr: nothing pending)
  // experts: sum_k w[t][k] y[slot[t][k]] (slot < 0: not a stored row), identity weight, gated shared expert
  const T* y;             // expert output rows [rows][ld]
  const int32_t* y_slot;  // [T][top]
  const float* y_w;       // [T][top]
  const float* id_w;      // [T]
  const T* sh;            // [T][ld] shared expert's output
  const float* sh_g;      // [T] its gate (nullptr: 1)
  int top;
};

// One workgroup per token.  The time is that of the rows behind the experts: a token's slots and weights lie in the lanes of a
// wave, and four rows are requested together (2048 tokens of 2048 columns and six experts 30.8 -> 25.5 us, 1100 of 1024 and seven
// 9.3 -> 7.9; the norms' parameters requested ahead of the sums: no change).
// x += mult * pending; (loop entry) x += x0, x += step; then xn1 / xn2 = norms of x, or cat = [x | x0] for a loop that enters
// through a matrix.  The embedding output is scale * embed[token] + pos[position].
// Rows of every array are ld (a multiple of KH_LPAD) elements with zeros behind the W valid ones.
template <class T>
struct CombineArgs {
  float *x, *x0;
  AddArgs<T> add;
  const T *embed, *pos_emb;                // pos_emb nullptr: none
  const int32_t *tok, *pos;
  const float* step;                       // one row or nullptr
  const float *w1, *b1, *w2, *b2;          // norm parameters (w1 nullptr: no norm output)
  T *xn1, *xn2;
  T* cat;                                  // [T][2 ld] or nullptr
  const T* xn2_prev;                       // identity experts' input: the xn2 the pending layer read
  int W, ld, from_embed, add_x0, rms;      // rms: no mean, biases may be nullptr
  float eps, mult, emb_scale;
};
template <class T>
__device__ __forceinline__ f32x4 quad_f(const T* p) {
  const typename Tile<T>::quad q = *(const typename Tile<T>::quad*)p;
  return f32x4{(float)q.x, (float)q.y, (float)q.z, (float)q.w};
}
__device__ __forceinline__ f32x4 fma_s(float s, f32x4 a, f32x4 b) {
  f32x4 r;
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = __builtin_fmaf(s, a[i], b[i]);
  return r;
}
template <class T>
__global__ __launch_bounds__(256) void k_combine(const CombineArgs<T> a) {
  typedef typename Tile<T>::quad quad;
  constexpr int U = 4;  // expert rows requested together
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  f32x4* row = (f32x4*)smem_raw;  // [ld / 4]
  __shared__ float red[KH_WAVES_MAX];
  const int t = blockIdx.x, n4 = a.ld >> 2, lane = threadIdx.x & 63;
  const size_t o = (size_t)t * a.ld;
  float s = 0.f;
  const int top = a.add.y ? a.add.top : 0;
  // lane k: choice k
  const int my_slot = lane < top ? a.add.y_slot[(size_t)t * top + lane] : -1;
  const float my_w = lane < top ? a.add.y_w[(size_t)t * top + lane] : 0.f;
  const T* e = a.from_embed ? a.embed + (size_t)a.tok[t] * a.ld : nullptr;
  const T* ep = a.from_embed && a.pos_emb ? a.pos_emb + (size_t)a.pos[t] * a.ld : nullptr;
  const float idw = a.add.y && a.add.id_w ? a.add.id_w[t] : 0.f, shg = a.add.sh && a.add.sh_g ? a.add.sh_g[t] : 1.f;
  for (int i = threadIdx.x; i < n4; i += 256) {
    const int c = 4 * i;
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    f32x4 v, d = zero, x0 = zero, st = zero;
    quad idq{}, shq{};
    if (a.add.mix) d = *(const f32x4*)(a.add.mix + o + c);
    if (!a.from_embed) v = *(const f32x4*)(a.x + o + c);
    if (a.add_x0 || (a.cat && !a.from_embed)) x0 = *(const f32x4*)(a.x0 + o + c);
    if (a.step) st = *(const f32x4*)(a.step + c);
    if (a.add.sh) shq = *(const quad*)(a.add.sh + o + c);
    if (idw != 0.f) idq = *(const quad*)(a.xn2_prev + o + c);
    if (a.from_embed) {
      v = quad_f(e + c) * a.emb_scale;
      if (ep) v += quad_f(ep + c);
      *(f32x4*)(a.x0 + o + c) = v;
      x0 = v;
    }
    if (a.add.mix) {
      f32x4 f = zero;
      for (int k0 = 0; k0 < top; k0 += U) {
        quad r[U];
        int sl[U];
        float w[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int k = k0 + u < top ? k0 + u : 63;  // lanes behind `top` hold -1
          sl[u] = __builtin_amdgcn_readlane(my_slot, k);
          w[u] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(my_w), k));
          r[u] = *(const quad*)(a.add.y + (size_t)max(sl[u], 0) * a.ld + c);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const f32x4 q = {(float)r[u].x, (float)r[u].y, (float)r[u].z, (float)r[u].w};
          if (sl[u] >= 0) f = fma_s(w[u], q, f);
        }
      }
      if (idw != 0.f) f = fma_s(idw, f32x4{(float)idq.x, (float)idq.y, (float)idq.z, (float)idq.w}, f);
      if (a.add.sh) f = fma_s(shg, f32x4{(float)shq.x, (float)shq.y, (float)shq.z, (float)shq.w}, f);
      d += f;
      v = fma_s(a.mult, d, v);
    }
    if (a.add_x0) v += x0;
    if (a.step) v += st;
    *(f32x4*)(a.x + o + c) = v;
    if (a.cat) {
      *(quad*)(a.cat + 2 * o + c) = to_quad<T>(v);
      *(quad*)(a.cat + 2 * o + a.ld + c) = to_quad<T>(a.from_embed ? v : x0);
    }
    row[i] = v;
    s += (v.x + v.y) + (v.z + v.w);
  }
  if (!a.w1) return;
  const float mean = a.rms ? 0.f : block_sum(s, red) / (float)a.W;
  float q = 0.f;
  for (int i = threadIdx.x; i < n4; i += 256) {
    const f32x4 v = row[i];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float d = 4 * i + k < a.W ? v[k] - mean : 0.f;
      q = __builtin_fmaf(d, d, q);
    }
  }
  const float rstd = 1.0f / sqrtf(block_sum(q, red) / (float)a.W + a.eps);
  for (int i = threadIdx.x; i < n4; i += 256) {
    const int c = 4 * i;
    const f32x4 v = row[i];
    f32x4 y;
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    const f32x4 w1 = *(const f32x4*)(a.w1 + c), b1 = a.b1 ? *(const f32x4*)(a.b1 + c) : zero;
#pragma unroll
    for (int k = 0; k < 4; ++k) y[k] = (v[k] - mean) * rstd * w1[k] + b1[k];  // pads: weights and biases are zero
    *(quad*)(a.xn1 + o + c) = to_quad<T>(y);
    if (a.w2) {
      const f32x4 w2 = *(const f32x4*)(a.w2 + c), b2 = a.b2 ? *(const f32x4*)(a.b2 + c) : zero;
#pragma unroll
      for (int k = 0; k < 4; ++k) y[k] = (v[k] - mean) * rstd * w2[k] + b2[k];
      *(quad*)(a.xn2 + o + c) = to_quad<T>(y);
    }
  }
}

// norm of gathered rows: out[r] = norm(x[rows[r]]); rows of ld elements on both sides.  rms: no mean, b may be nullptr
template <class T>
__global__ __launch_bounds__(256) void k_gather_norm(const float* x, const int32_t* rows, const float* w, const float* b,
                                                     T* out, int W, int ld, float eps, int rms) {
  __shared__ float red[KH_WAVES_MAX];
  const float* r = x + (size_t)rows[blockIdx.x] * ld;
  float s = 0.f;
  for (int i = threadIdx.x; i < W; i += 256) s += r[i];
  const float mean = rms ? 0.f : block_sum(s, red) / (float)W;
  float q = 0.f;
  for (int i = threadIdx.x; i < W; i += 256) {
    const float d = r[i] - mean;
    q = __builtin_fmaf(d, d, q);
  }
  const float rstd = 1.0f / sqrtf(block_sum(q, red) / (float)W + eps);
  for (int i = threadIdx.x; i < W; i += 256)
    out[(size_t)blockIdx.x * ld + i] = (T)((r[i] - mean) * rstd * w[i] + (b ? b[i] : 0.f));
}

// ---- causal depthwise convolution + silu -----------------------------------------------------------------------
// Inputs are the first C columns of xz rows.  Inputs before a segment's first row come from the sequence's conv state
// [taps - 1][C] (position 0: zeros).
template <class T>
struct ConvArgs {
  const T* xz;          // [T][ldx]
  T* out;               // [T][ldo]
  const float *w, *b;   // [C][taps], [C]
  float* state;         // + slot * slot_stride
  size_t slot_stride;
  int C, ldx, ldo, taps;
  PassTabs p;
};
// E channels (16 bytes) of KH_CONV_TT consecutive tokens of one chunk (kh_scan.h: tokens of one segment) per thread; the taps
// of the channels stay in registers.  With four taps all rows are requested at once (2048 tokens of 4096 channels: 20
// us; token by token, every token's rows behind the one before it, 32), and the channels' taps and biases as quads (19.2 -> 13.3:
// one at a time, every load of a wave touches 64 lines).
// TAPS: number of taps, 0 = any (weights re-read per token).  grid (C / (256 E), chunks x KH_CONV_PER)
#define KH_CONV_TT 8
#define KH_CONV_CH 64  // tokens of a chunk
#define KH_CONV_PER (KH_CONV_CH / KH_CONV_TT)
struct ScanChunk {
  int seg, row0, n, flags;  // flags: 1 = first of its segment, 2 = last of its segment
};
template <class T, int TAPS>
__global__ __launch_bounds__(256) void k_conv_silu(const ConvArgs<T> a, const ScanChunk* chunks) {
  constexpr int E = Tile<T>::N, TT = KH_CONV_TT;
  typedef typename Tile<T>::frag frag;
  const ScanChunk ck = chunks[blockIdx.y / KH_CONV_PER];
  const int u0 = (int)(blockIdx.y % KH_CONV_PER) * TT, n = ck.n - u0;
  const int c = (blockIdx.x * 256 + threadIdx.x) * E;
  if (n <= 0 || c >= a.C) return;
  // whole fragments, but for the last lane of a row that ends inside its channels (with scalar loads for all lanes there, 2048
  // tokens of 4100 channels take 26.2 us instead of 21.5, of 1100 13.0 instead of 12.0)
  const bool vec = c + E <= a.C && (a.ldx & (E - 1)) == 0;
  const int t0 = ck.row0 + u0, i0 = t0 - a.p.seg_row0[ck.seg];  // rows of the segment in front of the first token
  const int taps = TAPS ? TAPS : a.taps;
  const bool fresh = a.p.seg_pos0[ck.seg] == 0;
  const float* st = a.state + (size_t)a.p.seg_slot[ck.seg] * a.slot_stride;
  auto row = [&](int t, float (&in)[E]) __attribute__((always_inline)) {
    const T* x = a.xz + (size_t)t * a.ldx;
    if (vec) {
      const frag f = *(const frag*)(x + c);
#pragma unroll
      for (int e = 0; e < E; ++e) in[e] = (float)f[e];
    } else {
#pragma unroll
      for (int e = 0; e < E; ++e) in[e] = c + e < a.C ? (float)x[c + e] : 0.f;
    }
  };
  auto before = [&](int j, float (&in)[E]) __attribute__((always_inline)) {  // input j < 0 of the segment
#pragma unroll
    for (int e = 0; e < E; ++e) in[e] = !fresh && c + e < a.C ? st[(size_t)(taps - 1 + j) * a.C + c + e] : 0.f;
  };
  auto emit = [&](int t, const float (&v)[E]) __attribute__((always_inline)) {  // output rows are padded to whole fragments
    frag f;
#pragma unroll
    for (int e = 0; e < E; ++e) f[e] = (T)(c + e < a.C ? silu_t<T>(v[e]) : 0.f);
    *(frag*)(a.out + (size_t)t * a.ldo + c) = f;
  };
  float bias[E];
  auto quads = [&](const float* p, float* v, int n) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < n; i += 4) {
      const f32x4 q = *(const f32x4*)(p + i);
#pragma unroll
      for (int j = 0; j < 4; ++j) v[i + j] = q[j];
    }
  };
  if (vec) {
    quads(a.b + c, bias, E);
  } else {
#pragma unroll
    for (int e = 0; e < E; ++e) bias[e] = c + e < a.C ? a.b[c + e] : 0.f;
  }
  if constexpr (TAPS != 0) {
    float w[E][TAPS], pre[TAPS - 1][E];
    frag x[TT];
#pragma unroll
    for (int k = 0; k < TAPS - 1; ++k) {
      const int j = i0 - (TAPS - 1) + k;
      if (j >= 0) row(t0 - (TAPS - 1) + k, pre[k]);
      else before(j, pre[k]);
    }
#pragma unroll
    for (int u = 0; u < TT; ++u) {
      const int t = t0 + (u < n ? u : n - 1);
      if (vec) {
        x[u] = *(const frag*)(a.xz + (size_t)t * a.ldx + c);
      } else {
#pragma unroll
        for (int e = 0; e < E; ++e) x[u][e] = c + e < a.C ? a.xz[(size_t)t * a.ldx + c + e] : (T)0.f;
      }
    }
    if (vec && (E * TAPS) % 4 == 0) {  // a lane's taps lie side by side: one at a time a wave's loads touch 64 lines each
      quads(a.w + (size_t)c * TAPS, &w[0][0], E * TAPS);
    } else {
#pragma unroll
      for (int e = 0; e < E; ++e)
#pragma unroll
        for (int k = 0; k < TAPS; ++k) w[e][k] = c + e < a.C ? a.w[(size_t)(c + e) * TAPS + k] : 0.f;
    }
#pragma unroll
    for (int u = 0; u < TT; ++u) {
      if (u >= n) break;
      float v[E];
#pragma unroll
      for (int e = 0; e < E; ++e) {
        v[e] = bias[e];
#pragma unroll
        for (int k = 0; k < TAPS; ++k) {
          const int r = u - (TAPS - 1) + k;
          v[e] = __builtin_fmaf(w[e][k], r < 0 ? pre[r < 0 ? TAPS - 1 + r : 0][e] : (float)x[r < 0 ? 0 : r][e], v[e]);
        }
      }
      emit(t0 + u, v);
    }
  } else {
    for (int u = 0; u < TT && u < n; ++u) {
      float v[E], in[E];
#pragma unroll
      for (int e = 0; e < E; ++e) v[e] = bias[e];
      for (int k = 0; k < taps; ++k) {
        const int j = i0 + u - (taps - 1) + k;
        if (j >= 0) row(t0 + u - (taps - 1) + k, in);
        else before(j, in);
#pragma unroll
        for (int e = 0; e < E; ++e) v[e] = __builtin_fmaf(c + e < a.C ? a.w[(size_t)(c + e) * taps + k] : 0.f, in[e], v[e]);
      }
      emit(t0 + u, v);
    }
  }
}
template <class T>
void conv_launch(hipStream_t s, const ConvArgs<T>& a, const ScanChunk* chunks, int n_chunks) {
  constexpr int CW = 256 * Tile<T>::N;
  const dim3 g((a.C + CW - 1) / CW, n_chunks * KH_CONV_PER);
  if (a.taps == 4) hipLaunchKernelGGL((k_conv_silu<T, 4>), g, dim3(256), 0, s, a, chunks);
  else hipLaunchKernelGGL((k_conv_silu<T, 0>), g, dim3(256), 0, s, a, chunks);
}
}  // namespace khm
