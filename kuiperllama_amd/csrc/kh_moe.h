// kh_moe.h — expert router and dispatch lists.
// Two forms, both fp32, ties to the lower index:
//   over all     scores s = softmax(z) over all router outputs; the `top` largest s + correction are chosen; the weights
//                are the chosen s
//   over chosen  the `top` largest z are chosen; the weights are the softmax over them alone
// Outputs from n_expert on are identity experts (no tensors).
#pragma once
#include "kh_lgemm.h"

#define KH_MOE_MAX_OUT 1024  // router outputs (16 per lane)
#define KH_MOE_MAX_TOP 32
#define KH_MOE_RT 16          // tokens of a routing workgroup
#define KH_MOE_LT 1024        // threads of a list workgroup: one per expert

namespace khm {

// The choice for one token by one wave; z in LDS or global [n_out], n_out <= 64 PER.  Calls pick(k, id, weight) for
// k = 0 .. top - 1 on every lane with wave-uniform values, in order of decreasing choice score.  Weights are to be
// multiplied by the returned factor.  corr nullptr: none.
template <int PER, class F>
__device__ __forceinline__ float moe_route(const float* z, const float* corr, int n_out, int top, bool over_chosen, int lane,
                                           F&& pick) {
  float s[PER], key[PER];
  float m = -INFINITY;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int i = j * 64 + lane;
    s[j] = i < n_out ? z[i] : -INFINITY;
    key[j] = corr && i < n_out ? corr[i] : 0.f;
    m = fmaxf(m, s[j]);
  }
  m = wave_max(m);
  float sum = 0.f;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    if (over_chosen) key[j] = s[j];
    s[j] = expf(s[j] - m);  // exp(-inf) = 0 beyond n_out
    sum += s[j];
  }
  if (!over_chosen) {
    sum = wave_sum(sum);
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      s[j] /= sum;
      key[j] = j * 64 + lane < n_out ? s[j] + key[j] : -INFINITY;
    }
  }
  float chosen = 0.f;
  for (int k = 0; k < top; ++k) {
    float v = key[0];
#pragma unroll
    for (int j = 1; j < PER; ++j) v = fmaxf(v, key[j]);
    v = wave_max(v);
    // the lowest index that holds the maximum, and its weight, without a second and a third reduction
    int id = 1 << 30;  // nobody's (a NaN): an identity expert of no weight
    float w = 0.f;
#pragma unroll
    for (int j = PER - 1; j >= 0; --j) {
      const unsigned long long has = __builtin_amdgcn_ballot_w64(key[j] == v);
      if (has) {
        const int at = __builtin_ctzll(has);
        id = j * 64 + at;
        w = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, s[j]), at));
      }
    }
#pragma unroll
    for (int j = 0; j < PER; ++j) key[j] = j * 64 + lane == id ? -INFINITY : key[j];
    chosen += w;
    pick(k, id, w);
  }
  return over_chosen ? 1.0f / chosen : 1.0f;  // the largest z contributes exp(0)
}

struct RouteArgs {
  const float* z;        // [T][ldz]: router outputs, then (shared expert) its gate logit
  const float* corr;     // [n_out] or nullptr
  int32_t* id;           // [T][top]
  float* w;              // [T][top]
  float* id_w;           // [T] summed weight of the chosen identity experts
  float* sh_g;           // [T] sigmoid of the shared expert's gate
  int32_t* count;        // [ceil(T / KH_MOE_RT)][n_expert]: choices of each expert by a workgroup's tokens
  int32_t* rank;         // [T][top]: which of them this one is
  int T, ldz, n_out, n_expert, top, shared, over_chosen;
};
template <int PER>
__device__ __forceinline__ void moe_route_token(const RouteArgs& a, const float* z, int t, int lane, int32_t* cnt) {
  float idw = 0.f, my_w = 0.f;
  int my_id = 0;
  const float f = moe_route<PER>(z, a.corr, a.n_out, a.top, a.over_chosen, lane, [&](int k, int id, float w) __attribute__((always_inline)) {
    if (id >= a.n_expert) idw += w;
    my_id = lane == k ? id : my_id;  // top <= KH_MOE_MAX_TOP < 64: lane k keeps choice k
    my_w = lane == k ? w : my_w;
  });
  if (lane < a.top) {
    a.id[(size_t)t * a.top + lane] = my_id;
    if (my_id < a.n_expert) a.rank[(size_t)t * a.top + lane] = atomicAdd(&cnt[my_id], 1);
    a.w[(size_t)t * a.top + lane] = my_w * f;
  }
  if (lane == 0) {
    a.id_w[t] = idw * f;
    if (a.shared) a.sh_g[t] = sigmoid1(z[a.n_out]);
  }
}
template <int PER>
__global__ __launch_bounds__(64 * KH_MOE_RT) void k_moe_route(const RouteArgs a) {
  __shared__ int32_t cnt[KH_MOE_MAX_OUT];
  for (int e = threadIdx.x; e < a.n_expert; e += 64 * KH_MOE_RT) cnt[e] = 0;
  __syncthreads();
  const int t = blockIdx.x * KH_MOE_RT + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (t < a.T) moe_route_token<PER>(a, a.z + (size_t)t * a.ldz, t, lane, cnt);
  __syncthreads();
  for (int e = threadIdx.x; e < a.n_expert; e += 64 * KH_MOE_RT) a.count[(size_t)blockIdx.x * a.n_expert + e] = cnt[e];
}
static inline int moe_blocks(int T) { return (T + KH_MOE_RT - 1) / KH_MOE_RT; }
static inline int moe_per(int n_out) { return n_out <= 64 ? 1 : (n_out <= 256 ? 4 : 16); }
static inline void moe_route_launch(hipStream_t s, const RouteArgs& a) {
  const dim3 g(moe_blocks(a.T)), b(64 * KH_MOE_RT);
  if (moe_per(a.n_out) <= 4) hipLaunchKernelGGL(k_moe_route<4>, g, b, 0, s, a);
  else hipLaunchKernelGGL(k_moe_route<16>, g, b, 0, s, a);
}

// Router of at most 64 outputs, product and choice in one launch: a workgroup takes 16 tokens, its 16 waves 128 bytes of K each
// in turn, straight from memory to fragments (nobody reads a row twice), and then a token each.  Bound by what one CU can
// pull, and by the chain of the choices: as a GEMM tile of 64 tokens every workgroup drew 64 rows of activations and 64 of
// weights through its CU, 13.3 us for 2048 tokens x 37 outputs x 2048 on 32 CUs, and the choices took 6.3 more; this 14.3
// (1100 tokens x 32 x 1024: 13.6 -> 10.4).  More outputs than 64 go through the GEMM.  NT: 16-wide tiles of outputs.
struct MoeGateArgs {
  const void *X, *W;  // [T][ldx], [n_out + shared][ldw], the storage type
  int ldx, ldw, K;
  RouteArgs r;
};
template <class T, int NT>
__global__ __launch_bounds__(64 * KH_MOE_RT) void k_moe_gate(const MoeGateArgs a) {
  typedef Tile<T> TL;
  typedef typename TL::frag frag;
  constexpr int N = 16 * NT, LD = N + 4, HALF = KH_MOE_RT / 2;
  __shared__ __attribute__((aligned(16))) float part[HALF][16][LD];
  __shared__ float zs[16][N + 1];
  __shared__ int32_t cnt[64];
  const RouteArgs& r = a.r;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), fr = lane & 15, fh = lane >> 4;
  const int t0 = (int)blockIdx.x * KH_MOE_RT, rows = r.n_out + r.shared;
  if (threadIdx.x < 64) cnt[threadIdx.x] = 0;
  const char* x = (const char*)a.X + (size_t)(t0 + fr < r.T ? t0 + fr : r.T - 1) * a.ldx * sizeof(T) + 16 * fh;
  const char* w[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n)
    w[n] = (const char*)a.W + (size_t)(16 * n + fr < rows ? 16 * n + fr : rows - 1) * a.ldw * sizeof(T) + 16 * fh;
  f32x4 acc[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) acc[n] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int np = a.K * (int)sizeof(T) / 128;
  for (int p = wave; p < np; p += 2 * KH_MOE_RT) {
    const bool two = p + KH_MOE_RT < np;  // uniform
    frag fx[4], fw[4][NT];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const size_t at = (size_t)(b < 2 || !two ? p : p + KH_MOE_RT) * 128 + 64 * (b & 1);
      fx[b] = *(const frag*)(x + at);
#pragma unroll
      for (int n = 0; n < NT; ++n) fw[b][n] = *(const frag*)(w[n] + at);
    }
#pragma unroll
    for (int b = 0; b < 4; ++b)
      if (b < 2 || two)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[n] = TL::mma(fw[b][n], fx[b], acc[n]);
  }
  // lane: outputs 16 n + 4 fh + i of token fr
  if (wave >= HALF)
#pragma unroll
    for (int n = 0; n < NT; ++n) *(f32x4*)&part[wave - HALF][fr][16 * n + 4 * fh] = acc[n];
  __syncthreads();
  if (wave < HALF)
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      f32x4* q = (f32x4*)&part[wave][fr][16 * n + 4 * fh];
      *q = acc[n] + *q;
    }
  __syncthreads();
  if (threadIdx.x < 16 * N) {
    const int t = threadIdx.x / N, f = threadIdx.x - t * N;
    float z = part[0][t][f];
#pragma unroll
    for (int h = 1; h < HALF; ++h) z += part[h][t][f];
    zs[t][f] = z;
  }
  __syncthreads();
  if (t0 + wave < r.T) moe_route_token<1>(r, zs[wave], t0 + wave, lane, cnt);
  __syncthreads();
  if ((int)threadIdx.x < r.n_expert) r.count[(size_t)blockIdx.x * r.n_expert + threadIdx.x] = cnt[threadIdx.x];
}
template <class T>
void moe_gate_launch(hipStream_t s, const MoeGateArgs& a) {
  const dim3 g(moe_blocks(a.r.T)), b(64 * KH_MOE_RT);
  switch ((a.r.n_out + a.r.shared + 15) / 16) {
    case 1: hipLaunchKernelGGL((k_moe_gate<T, 1>), g, b, 0, s, a); break;
    case 2: hipLaunchKernelGGL((k_moe_gate<T, 2>), g, b, 0, s, a); break;
    case 3: hipLaunchKernelGGL((k_moe_gate<T, 3>), g, b, 0, s, a); break;
    default: hipLaunchKernelGGL((k_moe_gate<T, 4>), g, b, 0, s, a); break;
  }
}

// Dispatch lists: rows grouped by expert (row -> token), slot of every (token, choice) in that order (-1: identity expert),
// and the token tiles of the grouped GEMMs, the rows of an expert spread evenly over as few tiles as hold them (the GEMM skips
// what a tile lacks in units of 16 rows).  Latency alone: one workgroup per routing workgroup adds up the counts of all of
// them, four requests a thread at once, and places its own tokens.  One workgroup that counted every choice in LDS, where 64
// lanes meet on a few counters, took 11.5 us for 2048 x 6 choices of 32 experts and 8.4 for 1100 x 7; with the counts from the
// router this takes 4.9.
struct ListArgs {
  const int32_t *id, *count;  // [T][top], [blocks][n_expert]
  int32_t *rows, *slot;       // slot: ranks before, slots behind
  LgTile* tiles;
  int32_t* n_tiles;
  int T, top, n_expert, bm;
};
static_assert(KH_MOE_LT >= KH_MOE_MAX_OUT, "one thread per expert");
static __global__ __launch_bounds__(KH_MOE_LT) void k_moe_lists(const ListArgs a) {
  __shared__ int32_t tot[KH_MOE_MAX_OUT], pre[KH_MOE_MAX_OUT], part[2][2][KH_MOE_LT];
  const int E = a.n_expert, n_cnt = (int)gridDim.x * E, tid = threadIdx.x;
  for (int e = tid; e < E; e += KH_MOE_LT) tot[e] = pre[e] = 0;
  __syncthreads();
  for (int i0 = tid; i0 < n_cnt; i0 += 4 * KH_MOE_LT) {  // four requests at once
    int c[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) c[j] = i0 + j * KH_MOE_LT < n_cnt ? a.count[i0 + j * KH_MOE_LT] : 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const unsigned i = (unsigned)(i0 + j * KH_MOE_LT), b = i / (unsigned)E, e = i - b * (unsigned)E;
      if (!c[j]) continue;
      atomicAdd(&tot[e], c[j]);
      if (b < blockIdx.x) atomicAdd(&pre[e], c[j]);
    }
  }
  __syncthreads();
  // rows and tiles in front of each expert: a scan, one expert a thread
  const int c = tid < E ? tot[tid] : 0, nt = (c + a.bm - 1) / a.bm;
  part[0][0][tid] = c;
  part[0][1][tid] = nt;
  int from = 0;
  for (int d = 1; d < E; d <<= 1, from ^= 1) {
    __syncthreads();
    for (int q = 0; q < 2; ++q)
      part[from ^ 1][q][tid] = part[from][q][tid] + (tid >= d ? part[from][q][tid - d] : 0);
  }
  __syncthreads();
  const int row = part[from][0][tid] - c, til = part[from][1][tid] - nt;
  if (tid < E) pre[tid] += row;
  if (blockIdx.x == 0) {
    if (tid == E - 1) *a.n_tiles = til + nt;
    const int u = (c + 15) / 16;  // tile q: an equal number of 16-row units, one more in the first ones
    for (int q = 0; q < nt; ++q) {
      const int r0 = 16 * (q * (u / nt) + (q < u % nt ? q : u % nt));
      const int r1 = r0 + 16 * (u / nt + (q < u % nt ? 1 : 0));
      a.tiles[til + q] = LgTile{tid, row + r0, (r1 < c ? r1 : c) - r0, 0};
    }
  }
  __syncthreads();
  const int i1 = (int)(blockIdx.x + 1) * KH_MOE_RT * a.top, n = a.T * a.top;
  for (int i = i1 - KH_MOE_RT * a.top + tid; i < i1 && i < n; i += KH_MOE_LT) {
    const int e = a.id[i];
    int p = -1;
    if (e < E) {
      p = pre[e] + a.slot[i];
      a.rows[p] = i / a.top;
    }
    a.slot[i] = p;
  }
}
}  // namespace khm
