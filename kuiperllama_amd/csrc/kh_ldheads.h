// kh_ldheads.h — attention of one decoded token over grouped heads, as workgroups of the launch that reads the experts
// (kh_ldecode.h, k_ld_mid): in a parallel block neither needs the other, and a launch of its own is a chain of round trips on a
// few CUs.  Gusorax 1024 x 8 in fp32, 24 ... 64 keys: 9.4 us of experts and 9.3 of attention a layer were two launches and are
// one of 9.8; 64 steps 11 960 -> 9 270 us.
//
// Workgroup = 256 threads = one split of the visible keys of one sequence for up to four query heads of one key / value head,
// on the vector units: four heads' products per element read keep up with what one CU can pull (31 ... 40 bytes a ns).
//   scores    16 lanes per key, 16 bytes of it each (fp32: twice), 64 keys in flight
//   softmax   wave w has head w: a lane per key, running maximum and sum over the tiles of 64
//   values    16 bytes of a row per thread, all four heads; the rows of a wave meet by lane swaps, the waves in LDS
// The newest key and value come from the projected row, not from the cache row that another workgroup of the launch is writing;
// they are rounded as that one is.  Everything else is fp32.  Older keys come from the cache: no two tokens of a launch that also
// writes cache rows are one sequence's.  Where several of a prompt's tokens take the last layer together, a launch of the cache rows
// alone comes first (kh_hybrid_step.hip, `mates`).
// A layer has a fixed number of splits, and how long they are follows from the position: a sequence's bits are its own.  The
// last split of a group to arrive merges them all, in their order (kh_attn.h::attn_publish_barrier has the hand-over).
#pragma once
#include "kh_attn.h"
#include "kh_heads.h"

namespace khm {

#define KH_LDH_SPLITS 16   // splits of a group, at most (a power of two)
#define KH_LDH_WGS 128     // workgroups of a sequence, at most
#define KH_LDH_DIM 128     // key and value size that a thread's registers are laid out for

struct LdHeads {
  const float* qn;    // [dkp] query norm weight, scale not folded in (nullptr: no norm)
  const float* bias;  // as HeadsArgs::bias
  float* part;        // [B G chunks][nsplit][4][LDH_PART]
  float* out;         // [B][ldo], heads dvr apart
  int32_t* cnt;       // [B G chunks] tickets, zero between launches
  int nwg;            // workgroups: B G chunks nsplit (0: no such attention in this launch)
  int per, chunks;    // query heads of a key / value head, groups of four of them
  int nsplit, nbias, sink, g_off, ldo, fenced;
  KeySpan span;
  float scale2;       // scale * log2(e)
};
constexpr int kLdhPart = KH_LDH_DIM + 4;  // o, m, l of one head in one split
constexpr size_t kLdhLds = (4 * KH_LDH_DIM + 4 * 64 + 64 * 4 + 16 + 16 * KH_LDH_DIM) * 4;

// Workgroups of a sequence stand in front of the experts' in any case, most of them to leave at once while the sequence is short,
// and a split's tiles of 64 keys are a chain: so 128 workgroups a sequence, and this route for as many visible keys as its splits
// take 256 of each, in bf16 with less than 16 splits (more than 8 groups of four heads) 128.  Four layers of width 1024 with 7 of
// 32 experts of 512, heads of 128 over visible keys of that bound, us a step in launches of its own / so, one and four sequences:
//   keys                          30                       300                      1000                    4000
//   8 heads on 2, bf16     127 / 101  177 / 137     126 / 110  174 / 139     123 / 112  175 / 141    136 / 134  202 / 160
//   32 on 8, fp32          175 / 143  242 / 223     178 / 144  251 / 227     177 / 145  282 / 232    208 / 180  392 / 292
//   64 on 16, bf16         184 / 142  237 / 210     173 / 149  242 / 212     171 / 162  277 / 207
// In layers without experts, where it stands alone in its launch, 10-18 % less at 30 keys, as much at 3000 and in bf16 2-7 % more at
// 4000 keys of one sequence (8 on 2 130 / 138, 4 on 4 130 / 134).
// Beyond: 64 on 16 as 256 workgroups a sequence 230 / 250 at 30 keys, four sequences; in bf16 with 256 keys a split, one
// sequence at the last of them 163 / 168 (32 on 16, eight splits), 171 / 182 (32 on 32, four); 128 heads of 64 on 128 as one split,
// 4000 keys 262 / 528 and 616 / 977.
__host__ __device__ inline int ldh_splits(int groups) {
  int n = KH_LDH_SPLITS;
  while (n > 1 && n * groups > KH_LDH_WGS) n >>= 1;
  return n;
}
// Does a layer's attention run this way?  keys: the most that any position sees.
inline bool ldh_fits(int keys, int groups, int dkp, int dvp, size_t elem) {
  const int splits = ldh_splits(groups), each = elem == 2 && splits < KH_LDH_SPLITS ? 128 : 256;
  return keys <= each * splits && dkp <= KH_LDH_DIM && dvp <= KH_LDH_DIM;
}
// keys of a split: at least 32 KB of a group's keys and values of 128, in whole steps of 16
template <class T>
__host__ __device__ __forceinline__ int ldh_split_len(int n_keys, int nsplit) {
  const int per = ((n_keys + nsplit - 1) / nsplit + 15) & ~15, least = 128 / (int)sizeof(T);
  return per > least ? per : least;
}

template <class T>
__device__ __forceinline__ void ld_heads(const LdHeads& a, const HeadRow& r, const float* raw0, int ldr, const T* cache0,
                                         size_t slot_elems, const int32_t* pos_of, const int32_t* slot_of, int wg, char* smem) {
  typedef typename Tile<T>::frag frag;
  constexpr int E = Tile<T>::N, J = KH_LDH_DIM / (16 * E), KI = 4;  // 16-byte pieces of a key per lane; keys per lane and tile
  constexpr int LV = KH_LDH_DIM / E, VP = 256 / LV, NP = 64 / VP;   // lanes of a value row; rows of a pass; passes of a tile
  float* qs = (float*)smem;             // [4][128]
  float* sc = qs + 4 * KH_LDH_DIM;      // [4][64]
  float* ps = sc + 4 * 64;              // [64][4]
  float* fs = ps + 64 * 4;              // [4], ticket
  float* red = fs + 16;                 // [4 waves][4][128]
  const int tid = (int)threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int u = wg / a.nsplit, z = wg - u * a.nsplit, gc = r.G * a.chunks, q = u / gc, g = (u - q * gc) / a.chunks;
  const int h0 = (u - q * gc - g * a.chunks) * 4;
  const int pos = pos_of[q], slot = slot_of[q];
  const float* raw = raw0 + (size_t)q * ldr;
  // ---- what does not wait for the position: the wave's query head, its gate
  const int hw = h0 + wave, head = g * a.per + (hw < a.per ? hw : a.per - 1);
  float qx[2], qw[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int i = 64 * j + lane;
    qx[j] = i < r.dk && hw < a.per ? raw[(size_t)head * r.dkr + i] : 0.f;
    qw[j] = a.qn && i < r.dkp ? a.qn[i] : 1.f;
  }
  float2 gate{0.f, 0.f};
  if (a.g_off >= 0 && 2 * lane < r.dvr) gate = *(const float2*)(raw + a.g_off + (size_t)head * r.dvr + 2 * lane);
  const int k_first = a.span.first(pos), n_keys = pos + 1 - k_first;
  const int len = ldh_split_len<T>(n_keys, a.nsplit), nact = (n_keys + len - 1) / len;
  if (z >= nact) return;  // uniform
  const int k_lo = k_first + z * len, k_hi = k_lo + len < pos + 1 ? k_lo + len : pos + 1;
  // ---- the newest key and value as projected
  const int grp = tid >> 4, l16 = tid & 15, vrow = tid / LV, vc = (tid % LV) * E, row_e = r.dkp + r.dvp;
  float nk[J][E], nv[E];
#pragma unroll
  for (int j = 0; j < J; ++j)
#pragma unroll
    for (int e = 0; e < E; ++e) nk[j][e] = 0.f;
#pragma unroll
  for (int e = 0; e < E; ++e) nv[e] = 0.f;
  if (k_hi == pos + 1) {  // uniform
    const float *k = raw + r.k_off + (size_t)g * r.dkr, *v = raw + r.v_off + (size_t)g * r.dvr;
    float s = 0.f, w[J][E];
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int i = 16 * E * j + E * l16 + e;
        nk[j][e] = i < r.dk ? k[i] : 0.f;
        w[j][e] = r.kn && i < r.dkp ? r.kn[i] : 1.f;
        s = __builtin_fmaf(nk[j][e], nk[j][e], s);
      }
#pragma unroll
    for (int e = 0; e < E; ++e) nv[e] = vc + e < r.dv ? (float)(T)v[vc + e] : 0.f;
    s = group_sum<16>(s);
    const float rs = r.kn ? 1.0f / sqrtf(s / (float)r.dk + r.eps) : 1.f;
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
      for (int e = 0; e < E; ++e) nk[j][e] = (float)(T)(nk[j][e] * rs * w[j][e]);
  }
  {  // the query head: norm and scale, into LDS
    const float s = wave_sum(__builtin_fmaf(qx[0], qx[0], qx[1] * qx[1]));
    const float f = a.qn ? a.scale2 / sqrtf(s / (float)r.dk + r.eps) : a.scale2;
#pragma unroll
    for (int j = 0; j < 2; ++j) qs[wave * KH_LDH_DIM + 64 * j + lane] = qx[j] * f * qw[j];
  }
  __syncthreads();
  f32x4 qr[4][2];  // the lane's 8 elements of every head
#pragma unroll
  for (int h = 0; h < 4; ++h)
#pragma unroll
    for (int i = 0; i < 2; ++i)
      qr[h][i] = *(const f32x4*)(qs + h * KH_LDH_DIM + (J == 2 ? 64 * i + 4 * l16 : 8 * l16 + 4 * i));
  const T* cache = cache0 + (size_t)slot * slot_elems + (size_t)g * row_e;
  const unsigned step = (unsigned)(r.G * row_e);
  const int r0 = k_lo % r.ring;
  auto row_of = [&](int key) __attribute__((always_inline)) {  // (a key's distance from the first is below the span, and that the ring's)
    const int x = r0 + (key - k_lo);
    return cache + (size_t)((unsigned)(x < r.ring ? x : x - r.ring) * step);
  };
  float m = -1e30f, l = 0.f;  // finite: scores of -inf keep weights of zero
  float acc[4][E];
#pragma unroll
  for (int h = 0; h < 4; ++h)
#pragma unroll
    for (int e = 0; e < E; ++e) acc[h][e] = 0.f;
  for (int k0 = k_lo; k0 < k_hi; k0 += 64) {
    const int n = k_hi - k0 < 64 ? k_hi - k0 : 64;  // uniform
    frag kf[KI][J], vf[NP];
    float bs[KI];
#pragma unroll
    for (int i = 0; i < KI; ++i) {
      bs[i] = 0.f;
      if (16 * i >= n) continue;
      int key = k0 + 16 * i + grp;
      key = key < k_hi ? key : k_hi - 1;
      const T* p = row_of(key);
#pragma unroll
      for (int j = 0; j < J; ++j) {
        const int c = 16 * E * j + E * l16;
        kf[i][j] = *(const frag*)(p + (c < r.dkp ? c : 0));
      }
      if (a.bias && l16 < 4) {
        const int hh = h0 + l16 < a.per ? h0 + l16 : a.per - 1, d = pos - key;
        bs[i] = a.bias[(size_t)(g * a.per + hh) * a.nbias + (d < a.nbias - 1 ? d : a.nbias - 1)];
      }
    }
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      if (p * VP >= n) continue;
      int key = k0 + p * VP + vrow;
      key = key < k_hi ? key : k_hi - 1;
      vf[p] = *(const frag*)(row_of(key) + r.dkp + (vc < r.dvp ? vc : 0));
    }
#pragma unroll
    for (int i = 0; i < KI; ++i) {
      if (16 * i >= n) continue;
      const bool newest = k0 + 16 * i + grp >= pos;
      float s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < J; ++j)
#pragma unroll
        for (int e = 0; e < E; ++e) {
          const float x = newest ? nk[j][e] : (16 * E * j + E * l16 < r.dkp ? (float)kf[i][j][e] : 0.f);
#pragma unroll
          for (int h = 0; h < 4; ++h) s[h] = __builtin_fmaf(x, qr[h][J == 2 ? j : e >> 2][e & 3], s[h]);
        }
#pragma unroll
      for (int h = 0; h < 4; ++h) s[h] = group_sum<16>(s[h]);
      const float mine = l16 == 0 ? s[0] : l16 == 1 ? s[1] : l16 == 2 ? s[2] : s[3];
      if (l16 < 4) sc[l16 * 64 + 16 * i + grp] = mine + bs[i];
    }
    __syncthreads();
    {
      const float s = lane < n ? sc[wave * 64 + lane] : -INFINITY;
      const float mx = fmaxf(m, wave_max(s)), f = __builtin_amdgcn_exp2f(m - mx), p = __builtin_amdgcn_exp2f(s - mx);
      l = __builtin_fmaf(l, f, wave_sum(p));
      m = mx;
      ps[lane * 4 + wave] = p;
      if (lane == 0) fs[wave] = f;
    }
    __syncthreads();
    if (k0 != k_lo) {
#pragma unroll
      for (int h = 0; h < 4; ++h)
#pragma unroll
        for (int e = 0; e < E; ++e) acc[h][e] *= fs[h];
    }
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      if (p * VP >= n) continue;
      const bool newest = k0 + p * VP + vrow >= pos;  // and those behind it, whose weight is zero
      const f32x4 w = *(const f32x4*)(ps + (p * VP + vrow) * 4);
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const float x = newest ? nv[e] : (float)vf[p][e];
#pragma unroll
        for (int h = 0; h < 4; ++h) acc[h][e] = __builtin_fmaf(w[h], x, acc[h][e]);
      }
    }
  }
  // ---- the rows of a wave, then the waves
#pragma unroll
  for (int h = 0; h < 4; ++h)
#pragma unroll
    for (int e = 0; e < E; ++e) {
      if (LV <= 16) acc[h][e] = xor16_sum(acc[h][e]);
      acc[h][e] = xor32_sum(acc[h][e]);
    }
  if (lane < LV) {
#pragma unroll
    for (int h = 0; h < 4; ++h)
#pragma unroll
      for (int e = 0; e < E; e += 4)
        *(f32x4*)(red + (wave * 4 + h) * KH_LDH_DIM + vc + e) = f32x4{acc[h][e], acc[h][e + 1], acc[h][e + 2], acc[h][e + 3]};
  }
  __syncthreads();
  float2 o{0.f, 0.f};  // columns 2 lane, 2 lane + 1 of head h0 + wave
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    const float2 x = *(const float2*)(red + (w * 4 + wave) * KH_LDH_DIM + 2 * lane);
    o.x += x.x;
    o.y += x.y;
  }
  if (nact > 1) {
    float* part = a.part + ((size_t)u * a.nsplit * 4 + wave) * kLdhPart;  // the head in split 0; splits 4 kLdhPart apart
    {
      float* p = part + (size_t)z * 4 * kLdhPart;
      auto put = [](float* d, float x, float y) __attribute__((always_inline)) {
        const unsigned long long v = (unsigned long long)__float_as_uint(x) | (unsigned long long)__float_as_uint(y) << 32;
        __hip_atomic_store((unsigned long long*)d, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      };
      put(p + 2 * lane, o.x, o.y);
      if (lane == 0) put(p + KH_LDH_DIM, m, l);
    }
    attn_publish_barrier(a.fenced != 0);
    if (tid == 0) *(int*)(fs + 8) = __hip_atomic_fetch_add(a.cnt + u, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (*(const int*)(fs + 8) != nact - 1) return;  // uniform: not the last to arrive
    attn_acquire(a.fenced != 0);
    float2 ov[KH_LDH_SPLITS], ml[KH_LDH_SPLITS];
#pragma unroll
    for (int s = 0; s < KH_LDH_SPLITS; ++s) {  // all requested before the first is used; those behind the last repeat it
      const float* p = part + (size_t)(s < nact ? s : nact - 1) * 4 * kLdhPart;
      ov[s] = ld_agent_f2(p + 2 * lane);
      ml[s] = ld_agent_f2(p + KH_LDH_DIM);
    }
    m = ml[0].x;
#pragma unroll
    for (int s = 1; s < KH_LDH_SPLITS; ++s) m = fmaxf(m, ml[s].x);
    l = 0.f;
    o = float2{0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KH_LDH_SPLITS; ++s) {
      const float f = s < nact ? __builtin_amdgcn_exp2f(ml[s].x - m) : 0.f;
      l = __builtin_fmaf(ml[s].y, f, l);
      o.x = __builtin_fmaf(ov[s].x, f, o.x);
      o.y = __builtin_fmaf(ov[s].y, f, o.y);
    }
    if (tid == 0) __hip_atomic_store(a.cnt + u, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if (a.sink) {  // one more term exp(0) without a value
    const float mx = fmaxf(m, 0.f), f = __builtin_amdgcn_exp2f(m - mx);
    l = __builtin_fmaf(l, f, __builtin_amdgcn_exp2f(-mx));
    o.x *= f;
    o.y *= f;
  }
  if (hw >= a.per || 2 * lane >= r.dvr) return;
  const float inv = 1.0f / l;
  o.x *= inv;
  o.y *= inv;
  if (a.g_off >= 0) {
    o.x *= sigmoid1(gate.x);
    o.y *= sigmoid1(gate.y);
  }
  *(float2*)(a.out + (size_t)q * a.ldo + (size_t)head * r.dvr + 2 * lane) = o;
}
}  // namespace khm
