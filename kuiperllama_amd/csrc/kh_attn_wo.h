// kh_attn_wo.h - decode attention and the output projection in ONE launch, for models whose heads form few key / value
// groups (fp32 weights, positions below KH_ATTN_MIN_TS).
//
// A decode step is a chain of dependent launches, and the attention launch is its idlest: a handful of workgroups, 3.4 us, a
// few KB, followed by a launch boundary and wo's own start.  Here wo is cut along its columns into the PARTS that the key /
// value groups feed, and a workgroup owns (part, slice of rows): it requests its block of wo, computes the attention of the
// part's heads while the block travels - every slice of a part does so again, from K / V rows that the XCD's L2 holds -, and
// multiplies.  What it leaves is a partial sum per part and row; the launch that reads the residual next (k_ffn13_parts) adds
// them while it stages its vector, and leaves the sum for w2's epilogue.  A launch boundary, a launch's start and the trip of the
// attention output through memory go; `parts` vectors are staged instead of one (both ways measured: plan_attn_wo).
//
// The heads of a part are the columns of a 16-wide matrix product (kv_mul <= 16): a wave owns 16 timesteps, scores come from
// v_mfma_f32_16x16x4_f32 in the transposed form (S^T = K Q^T, then O^T += V^T P^T: the D layout of the first product is the B
// layout of the second).  The matrix core rounds its sums to one side, so a score is four sums of alternating sign and an
// output two.  Eight waves take 128 timesteps side by side and two tiles each beyond that; their (max, sum, output) meet in LDS.
//
// The B-token prompt path (kh_model_prefill) must leave the bits that steps leave: its tokens at these positions take the
// same attention (k_pf_attn_parts) and sum wo per part in the same order (k_pf_wo_parts).
#pragma once
#include "kh_attn.h"
#include "kh_common.h"
#include "kh_gemm.h"
#include "kh_gemv.h"
#include "kh_prefill.h"

#define KH_AWO_WAVES 8
#define KH_AWO_PARTS_MAX 8

struct KhAttnWoArgs {
  const float* q;             // [dim]; the prompt form: [tokens][dim]
  const float* kcache_layer;
  const float* vcache_layer;
  const int32_t* d_pos;       // nullptr: pos0
  const float* wo;            // [dim][dim]
  float* out;                 // partial sums [parts][dim]; the prompt form: attention outputs [tokens][dim]
  int pos0;                   // prompt form: position of token 0
  int dim, kv_dim, kv_mul;
};
// opart[waves][kv_mul][hs + 4] | m[waves][16] | l[waves][16] | x[kv_mul * hs]
static inline size_t attn_wo_lds_bytes(int head_size, int kv_mul) {
  return ((size_t)KH_AWO_WAVES * kv_mul * (head_size + 4) + 2 * KH_AWO_WAVES * 16 + (size_t)kv_mul * head_size) * sizeof(float);
}

// Attention of the kv_mul <= 16 heads of one group at `pos` < 256 -> xs[kv_mul * HS] in LDS, by the workgroup's first eight
// waves; two barriers, which its other waves meet too.
template <int DN>
__device__ __forceinline__ float* attn_parts_xs(int kv_mul, float* smem) {
  return smem + KH_AWO_WAVES * kv_mul * (16 * DN + 4) + 2 * KH_AWO_WAVES * 16;
}
template <int DN>
__device__ __forceinline__ void attn_parts_core(const float* __restrict__ q_g, const float* __restrict__ k_g,
                                                const float* __restrict__ v_g, int kv_stride, int kv_mul, int pos, float* smem) {
  constexpr int HS = 16 * DN, OS = HS + 4;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, lj = lane >> 4;
  float* opart = smem;
  float* mS = opart + KH_AWO_WAVES * kv_mul * OS;
  float* lS = mS + KH_AWO_WAVES * 16;
  float* xs = attn_parts_xs<DN>(kv_mul, smem);
  const float scale = 1.0f / sqrtf((float)HS);
  const f32x4 zero4 = {0.f, 0.f, 0.f, 0.f};
  auto run = [&](auto tiles) __attribute__((always_inline)) {
    constexpr int NT = decltype(tiles)::value;  // tiles of 16 timesteps a wave
    f32x4 qf[DN], kf[NT][DN];
    float vf[NT][4][DN];
    const float* qr = q_g + (size_t)(li < kv_mul ? li : kv_mul - 1) * HS + 4 * lj;  // columns past the group repeat its last head
#pragma unroll
    for (int c = 0; c < DN; ++c) qf[c] = *(const f32x4*)(qr + 16 * c);
#pragma unroll
    for (int j = 0; j < NT; ++j) {  // rows past the position: clamped re-reads of its row, masked below
      const int t0 = 16 * (wave + KH_AWO_WAVES * j);
      const float* kr = k_g + (size_t)(t0 + li < pos ? t0 + li : pos) * kv_stride + 4 * lj;
#pragma unroll
      for (int c = 0; c < DN; ++c) kf[j][c] = *(const f32x4*)(kr + 16 * c);
    }
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const int t0 = 16 * (wave + KH_AWO_WAVES * j) + 4 * lj;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float* vr = v_g + (size_t)(t0 + r < pos ? t0 + r : pos) * kv_stride + DN * li;
        if constexpr (DN == 4) {
          const f32x4 v = *(const f32x4*)vr;
#pragma unroll
          for (int d = 0; d < 4; ++d) vf[j][r][d] = v[d];
        } else {
#pragma unroll
          for (int d = 0; d < DN; ++d) vf[j][r][d] = vr[d];
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    float sv[NT][4];
    float m = -INFINITY;
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      f32x4 s[4] = {zero4, zero4, zero4, zero4};
#pragma unroll
      for (int c = 0; c < DN; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) s[e] = mfma16(kf[j][c][e], e & 1 ? -qf[c][e] : qf[c][e], s[e]);
      const int t0 = 16 * (wave + KH_AWO_WAVES * j) + 4 * lj;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        sv[j][r] = t0 + r <= pos ? ((s[0][r] - s[1][r]) + (s[2][r] - s[3][r])) * scale : -INFINITY;
        m = fmaxf(m, sv[j][r]);
      }
    }
    m = xor32_max(xor16_max(m));
    const float mref = m == -INFINITY ? 0.f : m;  // every score of the wave overflowed: weights of zero
    f32x4 oa[DN], ob[DN];
#pragma unroll
    for (int d = 0; d < DN; ++d) oa[d] = ob[d] = zero4;
    float l = 0.f;
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float p = expf(sv[j][r] - mref);
        l += p;
#pragma unroll
        for (int d = 0; d < DN; ++d) {
          if (r & 1) ob[d] = mfma16(vf[j][r][d], -p, ob[d]);
          else oa[d] = mfma16(vf[j][r][d], p, oa[d]);
        }
      }
    l = xor32_sum(xor16_sum(l));
    if (li < kv_mul) {
      // row i = 4 lj + r of the product is element DN i + d of the head
      f32x4* o = (f32x4*)(opart + (wave * kv_mul + li) * OS + 4 * DN * lj);
#pragma unroll
      for (int k = 0; k < DN; ++k) {
        f32x4 t;
#pragma unroll
        for (int e = 0; e < 4; ++e) t[e] = oa[(4 * k + e) % DN][(4 * k + e) / DN] - ob[(4 * k + e) % DN][(4 * k + e) / DN];
        o[k] = t;
      }
      if (lj == 0) {
        mS[wave * 16 + li] = m;
        lS[wave * 16 + li] = l;
      }
    }
  };
  if (16 * wave <= pos) {  // uniform: the wave has a timestep
    if (pos < 16 * KH_AWO_WAVES) run(std::integral_constant<int, 1>{});
    else run(std::integral_constant<int, 2>{});
  }
  __syncthreads();
  const int nact = pos < 16 * KH_AWO_WAVES ? (pos >> 4) + 1 : KH_AWO_WAVES;
  // one element a thread (plan_attn_wo: at most 512), clamped: no branch around the reads.  The waves' factors of a head are
  // computed by eight lanes; where the head is the whole wave's they are broadcast through scalar registers.
  const int e = tid < kv_mul * HS ? tid : 0, h = e / HS, d = e - h * HS;
  float ov[KH_AWO_WAVES];
#pragma unroll
  for (int w = 0; w < KH_AWO_WAVES; ++w) ov[w] = opart[((w < nact ? w : 0) * kv_mul + h) * OS + d];
  float num = 0.f, den;
  if constexpr (HS == 64) {
    const int w8 = lane & 7;
    const float mr = mS[(w8 < nact ? w8 : 0) * 16 + h], lr = lS[(w8 < nact ? w8 : 0) * 16 + h];
    const float mw = w8 < nact ? mr : -INFINITY;
    const float f = expf(mw - group_max<8>(mw));  // an absent wave: 0
    den = group_sum<8>(f * lr);
#pragma unroll
    for (int w = 0; w < KH_AWO_WAVES; ++w)
      num = __builtin_fmaf(__int_as_float(__builtin_amdgcn_readlane(__float_as_int(f), w)), ov[w], num);
  } else {
    float mv[KH_AWO_WAVES], M = -INFINITY;
#pragma unroll
    for (int w = 0; w < KH_AWO_WAVES; ++w) {
      const float t = mS[(w < nact ? w : 0) * 16 + h];
      mv[w] = w < nact ? t : -INFINITY;
      M = fmaxf(M, mv[w]);
    }
    den = 0.f;
#pragma unroll
    for (int w = 0; w < KH_AWO_WAVES; ++w) {
      const float f = expf(mv[w] - M);
      num = __builtin_fmaf(f, ov[w], num);
      den = __builtin_fmaf(f, lS[(w < nact ? w : 0) * 16 + h], den);
    }
  }
  if (tid < kv_mul * HS) xs[tid] = num / den;
  __syncthreads();
}

// LPR lanes a row of a part (a power of two), NU float4 a lane; RW rows a lane group: 8 * (64 / LPR) * RW rows a workgroup.
// grid: (parts, slices).  Eight waves for the attention and eight for the rows: a wave's loads retire in order, so requests of
// wo would stand in front of K and V, or behind them and the position that those wait for.
template <int DN, int LPR, int NU, int RW>
__global__ __launch_bounds__(128 * KH_AWO_WAVES) void k_attn_wo(const KhAttnWoArgs a) {
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  constexpr int HS = 16 * DN, RPI = 64 / LPR;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = blockIdx.x, dim = a.dim, cols4 = a.kv_mul * HS >> 2;
  if (wave < KH_AWO_WAVES) {
    attn_parts_core<DN>(a.q + (size_t)g * 4 * cols4, a.kcache_layer + (size_t)g * HS, a.vcache_layer + (size_t)g * HS, a.kv_dim,
                        a.kv_mul, *a.d_pos, (float*)smem_raw);
    return;
  }
  const int cl = lane & (LPR - 1);
  const int row0 = ((int)blockIdx.y * KH_AWO_WAVES + wave - KH_AWO_WAVES) * RPI * RW + lane / LPR;
  f32x4 w[RW][NU];
#pragma unroll
  for (int i = 0; i < RW; ++i) {
    const int row = row0 + i * RPI;
    const f32x4* wr = (const f32x4*)(a.wo + (size_t)(row < dim ? row : dim - 1) * dim + (size_t)g * 4 * cols4);
#pragma unroll
    for (int u = 0; u < NU; ++u) w[i][u] = ld_nt(wr + (cl + u * LPR < cols4 ? cl + u * LPR : 0));
  }
  __builtin_amdgcn_sched_barrier(0);
  __syncthreads();
  __syncthreads();
  const float* xs = attn_parts_xs<DN>(a.kv_mul, (float*)smem_raw);
  f32x4 xv[NU];
#pragma unroll
  for (int u = 0; u < NU; ++u) {
    const bool in = cl + u * LPR < cols4;
    const f32x4 t = ((const f32x4*)xs)[in ? cl + u * LPR : 0];
    xv[u] = in ? t : f32x4{0.f, 0.f, 0.f, 0.f};
  }
  float mine = 0.f;  // lane i of a group keeps its row i: one store
#pragma unroll
  for (int i = 0; i < RW; ++i) {
    float s = 0.f;
#pragma unroll
    for (int u = 0; u < NU; ++u) s = fma4(w[i][u], xv[u], s);
    s = group_sum<LPR>(s);
    mine = cl == i ? s : mine;
  }
  const int row = row0 + cl * RPI;
  if (cl < RW && row < dim) a.out[(size_t)g * dim + row] = mine;
}

// The same attention for prompt tokens at positions pos0 + blockIdx.y.  grid: (parts, tokens).
template <int DN>
__global__ __launch_bounds__(64 * KH_AWO_WAVES, 2) void k_pf_attn_parts(const KhAttnWoArgs a) {
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  const int g = blockIdx.x, t = blockIdx.y, cols = a.kv_mul * 16 * DN;
  const size_t at = (size_t)t * a.dim + (size_t)g * cols;
  attn_parts_core<DN>(a.q + at, a.kcache_layer + (size_t)g * 16 * DN, a.vcache_layer + (size_t)g * 16 * DN, a.kv_dim, a.kv_mul,
                      a.pos0 + t, (float*)smem_raw);
  const float* xs = attn_parts_xs<DN>(a.kv_mul, (float*)smem_raw);
  for (int e = threadIdx.x; e < cols; e += 64 * KH_AWO_WAVES) a.out[at + e] = xs[e];
}

// X[b] += wo . V[b] for up to KH_PF_BMAX tokens, summed per part as k_attn_wo and k_ffn13_parts do.  One row a lane group.
struct KhPfWoPartsArgs {
  const float* V;   // [tokens][dim]
  const float* wo;
  float* X;         // [tokens][dim], updated in place
  int dim, parts, cols4, nvalid;
};
template <int LPR, int NU>
__global__ __launch_bounds__(64 * KH_AWO_WAVES, 2) void k_pf_wo_parts(const KhPfWoPartsArgs a) {
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  constexpr int RPI = 64 / LPR;
  f32x4* xs = (f32x4*)smem_raw;  // [nvalid][dim]
  const int lane = threadIdx.x & 63, cl = lane & (LPR - 1), dim = a.dim, nvalid = a.nvalid;
  const int row = ((int)blockIdx.x * KH_AWO_WAVES + (int)(threadIdx.x >> 6)) * RPI + lane / LPR;
  const int rc = row < dim ? row : dim - 1;
  f32x4 w[KH_AWO_PARTS_MAX][NU];
#pragma unroll
  for (int p = 0; p < KH_AWO_PARTS_MAX; ++p) {
    if (p >= a.parts) break;  // uniform
    const f32x4* wr = (const f32x4*)(a.wo + (size_t)rc * dim) + p * a.cols4;
#pragma unroll
    for (int u = 0; u < NU; ++u) w[p][u] = wr[cl + u * LPR < a.cols4 ? cl + u * LPR : 0];
  }
  float x[KH_PF_BMAX], sum[KH_PF_BMAX];
#pragma unroll
  for (int b = 0; b < KH_PF_BMAX; ++b) x[b] = a.X[(size_t)(b < nvalid ? b : 0) * dim + rc];
  for (int i = threadIdx.x; i < nvalid * (dim >> 2); i += 64 * KH_AWO_WAVES) xs[i] = ((const f32x4*)a.V)[i];
  __syncthreads();
#pragma unroll
  for (int p = 0; p < KH_AWO_PARTS_MAX; ++p) {
    if (p >= a.parts) break;
#pragma unroll
    for (int b = 0; b < KH_PF_BMAX; ++b) {
      if (b >= nvalid) break;
      float s = 0.f;
#pragma unroll
      for (int u = 0; u < NU; ++u) {
        const bool in = cl + u * LPR < a.cols4;
        f32x4 v = xs[b * (dim >> 2) + p * a.cols4 + (in ? cl + u * LPR : 0)];
        if (!in) v = f32x4{0.f, 0.f, 0.f, 0.f};
        s = fma4(w[p][u], v, s);
      }
      s = group_sum<LPR>(s);
      sum[b] = p == 0 ? s : sum[b] + s;
    }
  }
  if (cl == 0 && row < dim) {
#pragma unroll
    for (int b = 0; b < KH_PF_BMAX; ++b)
      if (b < nvalid) a.X[(size_t)b * dim + row] = x[b] + sum[b];
  }
}

// ---- the launch behind it: x1 = x + the parts, and the feed-forward's first half of it ---------------------------------------
struct KhFfn13PartsArgs {
  KhFfn13Args f;
  const float* part;  // [parts][dim]
  float* x1;          // [dim]: the sum, for w2's epilogue
  int parts;
};
// Stager<true, false, MAXV> of kh_gemv.h over x + (part[0] + part[1] + ...), PN >= parts (the rest re-read and dropped)
template <int MAXV, int PN>
struct PartsStager {
  f32x4 xv[MAXV], wv[MAXV], pv[MAXV][PN];
  const f32x4 *x4, *w4, *p4;
  f32x4* x1;
  int M, parts;
  __device__ __forceinline__ PartsStager(const KhFfn13PartsArgs& a)
      : x4((const f32x4*)a.f.x), w4((const f32x4*)a.f.ffn_norm), p4((const f32x4*)a.part), x1((f32x4*)a.x1), M(a.f.dim),
        parts(a.parts) {}
  __device__ __forceinline__ void issue() {
    const int M4 = M >> 2;
#pragma unroll
    for (int v = 0; v < MAXV; ++v) {
      const int i = threadIdx.x + v * kh_wg(), ci = i < M4 ? i : 0;
      xv[v] = x4[ci];
      wv[v] = w4[ci];
#pragma unroll
      for (int p = 0; p < PN; ++p) pv[v][p] = p4[(p < parts ? p : parts - 1) * M4 + ci];
    }
  }
  __device__ __forceinline__ float finish(f32x4* xs, float eps, float* red) {
    const int M4 = M >> 2;
    float ss = 0.f;
#pragma unroll
    for (int v = 0; v < MAXV; ++v) {
      const int i = threadIdx.x + v * kh_wg();
      f32x4 sum = pv[v][0];  // of the parts first: the residual is the larger number, and rounds once
#pragma unroll
      for (int p = 1; p < PN; ++p) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float s = sum[e] + pv[v][p][e];
          sum[e] = p < parts ? s : sum[e];
        }
      }
      xv[v] = xv[v] + sum;
      const float t = fma4(xv[v], xv[v], 0.f);
      ss += i < M4 ? t : 0.f;
    }
#pragma unroll
    for (int v = 0; v < MAXV; ++v) {
      const int i = threadIdx.x + v * kh_wg();
      if (i < M4) xs[i] = wv[v] * xv[v];
    }
    return stage_rs(ss, M, eps, red);
  }
  // behind the loop over the rows: its loads would wait for a store ahead of them
  __device__ __forceinline__ void keep() {
    if (blockIdx.x != 0) return;
#pragma unroll
    for (int v = 0; v < MAXV; ++v) {
      const int i = threadIdx.x + v * kh_wg();
      if (i < M >> 2) x1[i] = xv[v];
    }
  }
};
template <int U, int MAXV, int PN>
__global__ __launch_bounds__(KH_WG_MAX, 2) void k_ffn13_parts(const KhFfn13PartsArgs a) {
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  f32x4* xs = (f32x4*)smem_raw;
  float* red = lds_red_ptr<false>(xs, a.f.dim);
  const int lane = threadIdx.x & 63, dim = a.f.dim;
  const void *w1 = a.f.w1.w, *w3 = a.f.w3.w;
  float* const h = a.f.h;
  const Gemv<false, U> g(dim, 0);
  PartsStager<MAXV, PN> st(a);
  auto pair = [&](int r) __attribute__((always_inline)) { return g.rows(w1, r, w3, r, nullptr, nullptr, dim); };
  float rs = 1.f;
  auto epi = [&](int r, float s0, float s1, const NoAux&) __attribute__((always_inline)) {
    if (lane == 0) h[r] = swiglu1(rs * s0, rs * s1);
  };
  gemv_pairs<1, /*ROLL=*/false>(g, xs, a.f.hidden, lane, nullptr, pair, [](int) __attribute__((always_inline)) { return NoAux{}; },
                       [&]() __attribute__((always_inline)) { st.issue(); },
                       [&]() __attribute__((always_inline)) { rs = st.finish(xs, a.f.eps, red); }, epi);
  st.keep();
}
