// kh_scan.h — selective scan:  S[c, n] <- exp(dt_c A[c, n]) S[c, n] + dt_c x_c B_n ;  y_c = sum_n S[c, n] C_n + D_c x_c ;
// out = y silu(z).  fp32 throughout; the state of a sequence stays in its slot between calls.
//
// A lane owns 8 or 16 states of one channel, G = 2^g lanes share a channel (their partial y meet in a DPP
// reduction), 256 / G channels per workgroup.  Prompts are cut into CHUNKS of up to KH_SCAN_CH tokens that run side by
// side:  k_scan_ends  computes every chunk's end state from a zero start and its sum of dt (the chunk's decay is
// exp(A sum dt));  k_scan_carry  walks the chunks of a segment and turns the end states into start states;
// k_scan_out  runs each chunk from its start state, writes the outputs and, in a segment's last chunk, the slot's
// state.  Segments of one chunk (and decoding) need k_scan_out only.
#pragma once
#include <type_traits>

#include "kh_lops.h"

#define KH_SCAN_CH KH_CONV_CH  // tokens of a chunk
#define KH_SCAN_MAX_STATE 256  // 32 lanes x 8

namespace khm {

template <class T>
struct ScanArgs {
  const T* x;            // [T][ldx] convolved inputs
  const T* z;            // [T][ldz] gate (nullptr in k_scan_ends)
  const float* dt;       // [T][C]
  const float* bc;       // [T][2 N]: B then C
  const float *A2, *D;   // A2 = -exp(A_log) log2(e)  [C][N], D [C]
  T* out;                // [T][ldo]
  float* state;          // + slot * slot_stride: [C][N]
  size_t slot_stride;
  float *ends, *dtsum;   // [chunks][C][N], [chunks][C]
  const ScanChunk* chunks;
  PassTabs p;
  int C, N, ldx, ldz, ldo, gshift;
  // with outputs: the last taps - 1 inputs of the convolution become its sequence's state, where a segment ends
  const T* cx;           // [T][ldz]
  float* conv;           // + slot * slot_stride: [taps - 1][C]
  int taps;
};

template <int G>
__device__ __forceinline__ float scan_group_sum(float v) { return group_sum<G>(v); }

// B and C rows of the chunk go to LDS: [n_tok][2 N].  A state costs 28 cycles of a wave a token (36 with its output), half of
// them the exponential, a token about 200 more (loads, conversions, silu): NS states a lane share those.  Inputs are requested
// U tokens ahead.  2048 tokens of 4096 x 16: 45 + 61 us with 8 states a lane, requests in front of their own tokens and the
// library's exponential in the gate; 44 + 52 us with 16.  The convolution's state is written here, 1.8 us, not by a launch of
// its own, 4.7 and its start.
template <class T, bool OUT, int NS, int G>
__global__ __launch_bounds__(256) void k_scan(const ScanArgs<T> a) {
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  float* bc = (float*)smem_raw;
  const ScanChunk ck = a.chunks[blockIdx.y];
  if (!OUT && (ck.flags & 2)) return;  // nobody continues from a last chunk's zero-start end
  const int N = a.N;
  constexpr int NP = G * NS;  // LDS rows padded to whole lanes
  for (int i = threadIdx.x; i < ck.n * NP * 2; i += 256) {
    const int t = i / (2 * NP), r = i - t * (2 * NP), which = r >= NP, n = r - which * NP;
    bc[i] = n < N ? a.bc[(size_t)(ck.row0 + t) * (2 * N) + which * N + n] : 0.f;
  }
  const int g = threadIdx.x & (G - 1);
  const int c = blockIdx.x * (256 / G) + (int)threadIdx.x / G;
  const bool live = c < a.C;
  const int cc = live ? c : a.C - 1;
  const int n0 = g * NS;
  constexpr int U = 4;  // tokens requested together
  float xv[U], dv[U], zv[U];
  auto request = [&](int t0) __attribute__((always_inline)) {  // uniform rows, one offset a lane
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const size_t t = (size_t)(ck.row0 + (t0 + u < ck.n ? t0 + u : ck.n - 1));
      xv[u] = (float)(a.x + t * a.ldx)[cc];
      dv[u] = (a.dt + t * a.C)[cc];
      if (OUT) zv[u] = (float)(a.z + t * a.ldz)[cc];
    }
  };
  request(0);
  float A2[NS], S[NS];
  const size_t sbase = (size_t)cc * N;
  const bool alone = (ck.flags & 3) == 3;
  const int slot = a.p.seg_slot[ck.seg];
  float* st = a.state + (size_t)slot * a.slot_stride + sbase;
  const bool fresh = a.p.seg_pos0[ck.seg] == 0;
#pragma unroll
  for (int j = 0; j < NS; ++j) {
    const int n = n0 + j;
    A2[j] = n < N ? a.A2[sbase + n] : 0.f;
    S[j] = 0.f;
    if (OUT && n < N) {
      // start state: a segment of several chunks has all of them from k_scan_carry, its first too - the last one's workgroup
      // writes the slot's state in this launch
      if (!alone) S[j] = a.ends[(size_t)blockIdx.y * a.C * N + sbase + n];
      else if (!fresh) S[j] = st[n];
    }
  }
  const float D = OUT ? a.D[cc] : 0.f;
  float dts = 0.f;
  __syncthreads();
  for (int t0 = 0; t0 < ck.n; t0 += U) {
    float x[U], d[U], z[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      x[u] = xv[u];
      d[u] = dv[u];
      if (OUT) z[u] = zv[u];
    }
    if (t0 + U < ck.n) request(t0 + U);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (t0 + u >= ck.n) break;
      const float* b = bc + (size_t)(t0 + u) * 2 * NP + n0;
      const float dx = d[u] * x[u];
      float y = 0.f;
#pragma unroll
      for (int j = 0; j < NS; ++j) {
        S[j] = __builtin_fmaf(__builtin_amdgcn_exp2f(d[u] * A2[j]), S[j], dx * b[j]);
        if (OUT) y = __builtin_fmaf(S[j], b[NP + j], y);
      }
      dts += d[u];
      if (OUT) {
        y = scan_group_sum<G>(y);
        y = __builtin_fmaf(D, x[u], y);
        if (g == 0 && live) (a.out + (size_t)(ck.row0 + t0 + u) * a.ldo)[c] = (T)(y * silu_t<T>(z[u]));
      }
    }
  }
  if (!live) return;
#pragma unroll
  for (int j = 0; j < NS; ++j) {
    const int n = n0 + j;
    if (n >= N) continue;
    if (OUT) {
      if (ck.flags & 2) st[n] = S[j];
    } else {
      a.ends[(size_t)blockIdx.y * a.C * N + sbase + n] = S[j];
    }
  }
  if (!OUT && g == 0) a.dtsum[(size_t)blockIdx.y * a.C + c] = dts;
  if (OUT && (ck.flags & 2) && g == 0) {
    const int n = a.p.seg_n[ck.seg], last = ck.row0 + ck.n, m = a.taps - 1;
    float* cs = a.conv + (size_t)slot * a.slot_stride + c;
    for (int j = 0; j < m; ++j) {  // ascending: entry j reads entry j + n > j of the old state
      float v = 0.f;
      if (n - m + j >= 0) v = (float)a.cx[(size_t)(last - m + j) * a.ldz + c];
      else if (!fresh) v = cs[(size_t)(j + n) * a.C];
      cs[(size_t)j * a.C] = v;
    }
  }
}

// ends[k] (end of chunk k from zero) -> start state of chunk k, for every segment's chunks in order.
// grid (C N / 256, segments with more than one chunk); chunk0 / nchunk per such segment
template <class T>
__global__ __launch_bounds__(256) void k_scan_carry(const ScanArgs<T> a, const int32_t* chunk0, const int32_t* nchunk) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x, CN = (size_t)a.C * a.N;
  if (i >= CN) return;
  const int k0 = chunk0[blockIdx.y], nk = nchunk[blockIdx.y];
  const int seg = a.chunks[k0].seg;
  const float A2 = a.A2[i];
  const int c = (int)(i / a.N);
  float S = a.p.seg_pos0[seg] == 0 ? 0.f : a.state[(size_t)a.p.seg_slot[seg] * a.slot_stride + i];
  constexpr int U = 8;  // chunks requested together: one at a time 15 us for 32 chunks of 4096 x 16, 8 with eight
  for (int kb = k0; kb < k0 + nk; kb += U) {
    float e[U], d[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const bool in = kb + u + 1 < k0 + nk;
      e[u] = in ? a.ends[(size_t)(kb + u) * CN + i] : 0.f;
      d[u] = in ? a.dtsum[(size_t)(kb + u) * a.C + c] : 0.f;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (kb + u >= k0 + nk) break;
      a.ends[(size_t)(kb + u) * CN + i] = S;
      S = __builtin_fmaf(__builtin_amdgcn_exp2f(A2 * d[u]), S, e[u]);
    }
  }
}

// 16 states a lane where that leaves every SIMD two waves, else 8
template <class T, bool OUT>
int scan_launch(hipStream_t s, const ScanArgs<T>& a, int nchunks) {
  const bool wide = a.N > 8 && (long)((a.C + 255) / 256) * 4 * ((a.N + 15) / 16) * nchunks >= 2048;
  const int NS = wide ? 16 : 8;
  int G = 1;
  while (G * NS < a.N) G <<= 1;
  const dim3 grid((a.C + 256 / G - 1) / (256 / G), nchunks);
  const size_t lds = (size_t)KH_SCAN_CH * 2 * G * NS * 4;
  auto go = [&](auto kern) -> int {
    if (lds > 64 * 1024 &&
        hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
      return KH_ERR_UNSUPPORTED;
    hipLaunchKernelGGL(kern, grid, dim3(256), lds, s, a);
    return KH_OK;
  };
  auto by_group = [&](auto ns) -> int {
    constexpr int K = decltype(ns)::value;
    switch (G) {
      case 1: return go(k_scan<T, OUT, K, 1>);
      case 2: return go(k_scan<T, OUT, K, 2>);
      case 4: return go(k_scan<T, OUT, K, 4>);
      case 8: return go(k_scan<T, OUT, K, 8>);
      case 16: return go(k_scan<T, OUT, K, 16>);
      case 32:
        if constexpr (K == 8) return go(k_scan<T, OUT, 8, 32>);
      default: return KH_ERR_UNSUPPORTED;
    }
  };
  return wide ? by_group(std::integral_constant<int, 16>()) : by_group(std::integral_constant<int, 8>());
}
}  // namespace khm
