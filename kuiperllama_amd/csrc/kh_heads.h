// kh_heads.h — attention over cached keys and values with grouped heads (query head h reads key / value head h / (H / G)):
// per-head RMS norms of queries and keys, a learned bias by distance, sliding windows, chunks, a sink, an output gate.
// Everything but the kernel's tile sizes is a parameter.
//
// A cache row holds, key / value head by head, [key (dkp) | value (dvp)], both padded to 64 elements with zeros.  A run
// keeps `ring` rows per sequence: position p lies in row p % ring (ring = the cache length where every key stays
// visible; for windows and chunks the span of one query plus the tokens of one pass).
//
// k_heads_attn: workgroup = 4 waves = WR x MR tiles of 16 query rows x CP column parts (WR CP = 4) of the values of ONE
//   key / value head; a query row is a (token, query head of the group) pair, so the group's heads share each staged key
//   tile.  Tiles of KT cache rows go straight to LDS (LDS-DMA, a ring of NST stages).  S^T = K Q^T: a lane ends with the scores
//   of ONE query row per tile of 16, so the running max / sum are lane scalars plus two cross-row swaps, and P^T is
//   already the second operand of O^T = V^T P^T, whose first operand comes from the same LDS rows (lat_col).
//   Queries are read as projected and normalised in registers; scale and log2(e) are folded in with the norm weights.
// Scores, weights and sums are fp32; queries and P are rounded to the storage type for their products.
#pragma once
#include "kh_latent.h"

namespace khm {

// Keys position `pos` sees: [first(pos), pos].  0: no limit of that kind.
struct KeySpan {
  int window;  // at most that many keys, itself included
  int chunk;   // only keys of its own chunk, counted from position 0 of the sequence
  __host__ __device__ __forceinline__ int first(int pos) const {
    int f = chunk > 0 ? pos - pos % chunk : 0;
    if (window > 0 && pos - window + 1 > f) f = pos - window + 1;
    return f;
  }
};

// ---- cache rows: one wave per (token, key / value head) ----------------------------------------------------------------
struct HeadRow {
  const float* kn;  // [dkp] norm weight behind the keys' RMS norm (nullptr: no norm)
  int G, dk, dv, dkr, dvr, dkp, dvp, k_off, v_off, ring;  // k_off, v_off: first key / value column of a projected row
  float eps;
};
template <class R, class T>
__device__ __forceinline__ void heads_cache_row(const HeadRow& a, const R* raw, T* cache, int pos, int g, int lane) {
  constexpr int N = 4;  // 64 N >= the largest padded head
  const R *k = raw + a.k_off + (size_t)g * a.dkr, *v = raw + a.v_off + (size_t)g * a.dvr;
  float x[N], w[N], y[N], s = 0.f;
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const int i = 64 * j + lane;
    x[j] = i < a.dk ? (float)k[i] : 0.f;
    y[j] = i < a.dv ? (float)v[i] : 0.f;
    w[j] = a.kn && i < a.dkp ? a.kn[i] : 1.f;
    s = __builtin_fmaf(x[j], x[j], s);
  }
  const float rs = a.kn ? 1.0f / sqrtf(wave_sum(s) / (float)a.dk + a.eps) : 1.f;
  T* row = cache + ((size_t)(pos % a.ring) * a.G + g) * (a.dkp + a.dvp);
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const int i = 64 * j + lane;
    if (i < a.dkp) row[i] = (T)(x[j] * rs * w[j]);
    if (i < a.dvp) row[a.dkp + i] = (T)y[j];
  }
}
template <class T>
struct HeadRowsArgs {
  HeadRow r;
  const T* raw;  // [tokens][ldr]
  T* cache;      // + slot * slot_elems
  size_t slot_elems;
  int ldr, T_all;
  PassTabs p;
};
// grid (tokens G / 4)
template <class T>
__global__ __launch_bounds__(256) void k_heads_rows(const HeadRowsArgs<T> a) {
  const int i = blockIdx.x * 4 + (threadIdx.x >> 6), t = i / a.r.G, g = i - t * a.r.G;
  if (t >= a.T_all) return;
  heads_cache_row(a.r, a.raw + (size_t)t * a.ldr, a.cache + (size_t)a.p.seg_slot[a.p.seg[t]] * a.slot_elems, a.p.pos[t], g,
                  threadIdx.x & 63);
}

// ---- attention -------------------------------------------------------------------------------------------------
struct HeadsArgs {
  const void* raw;       // [T][ldr] projected rows: query heads dkr apart from column 0; gate logits dvr apart from g_off
  int raw_f32;           // the rows are fp32 (else the storage type)
  int g_off;             // -1: no output gate (it is applied where the result is written: with one split)
  const float* qn;       // [dkp] query norm weight (nullptr: no norm)
  const void* cache;     // + slot * slot_elems + row * G (dkp + dvp)
  size_t slot_elems;
  const float* bias;     // [H][nbias] by distance, in units of log2(e); the last entry holds for everything beyond.  nullptr: none
  void* out;             // [T][ldo], heads dvr apart (one split): T, or fp32
  int out_f32;
  float* part;           // splits > 1: [T H][splits][dvp + 4]: o (unnormalised), m, l.  One token per segment then
  const LatTile* tiles;  // nullptr: one token per segment, ceil((H / G) / rows of a tile) workgroups each
  int H, G, dk, dkr, dkp, dvr, dvp, ldr, ldo, ring, nsplit, nbias, bias_lds;
  int sink;              // the softmax denominator has one more term exp(0) without a value
  KeySpan span;
  float eps, scale2;     // scale * log2(e)
  PassTabs p;
};

#define KH_HEADS_MAX_DIM 256
#define KH_HEADS_BIAS_LDS (32 * 1024)  // the largest distance table that is copied to LDS, behind the stages
constexpr int kHeadsLds = 160 * 1024;  // of a workgroup: the stages of all sets of waves and the table
// a tile holds 64 bytes of keys a column: 32 in bf16, 16 in fp32
constexpr int heads_tile_bytes(int dkp, int dvp) { return 64 * (dkp + dvp); }
// stages of a key tile of tb bytes, ks sets of them: three of small tiles, where the largest table still fits beside them
constexpr int heads_stages(int tb, int ks) { return tb <= 24 * 1024 && 3 * ks * tb + KH_HEADS_BIAS_LDS <= kHeadsLds ? 3 : 2; }
constexpr bool heads_table_lds(size_t table) { return table <= KH_HEADS_BIAS_LDS; }
constexpr size_t heads_lds(int tb, int ks, size_t table) {
  return (size_t)ks * heads_stages(tb, ks) * tb + (heads_table_lds(table) ? table : 0);
}

// KN, KV: key and value size in units of 64.  CP = 4: 16 rows per workgroup; CP = 1: 64 MR rows.  KS: sets of four waves; set k
// takes key tiles k, k + KS, ... of the same rows, and the sets are merged at the end through LDS.  A tile of 32 keys is a
// serial chain (keys from LDS, scores, maximum, exponentials, values: 1.1 us for 0.1 us of products), so a wave needs another
// one on its SIMD; where the rows of a launch make one workgroup per CU, KS = 2 is where it comes from.  KS = 4: a decoded
// token whose keys nobody else shares (heads_one_split), the tiles of a workgroup side by side, or such a launch of rows in bf16.
// Two waves per SIMD where the accumulators allow it: within 256 registers the compiler keeps them where the rescaling can
// reach them (beyond, it moves them between two register files in every tile).
template <class T, int KN, int KV, int CP, int MR, int KS>
__global__ __launch_bounds__(256 * KS, KN + KV > 4 && KS == 1 ? 1 : 2) void k_heads_attn(const HeadsArgs a) {
  typedef Tile<T> TL;
  typedef typename TL::frag frag;
  constexpr int E = TL::N, KT = 4 * E, NS = KT / 16, ES = (int)sizeof(T);
  constexpr int DK = 64 * KN, DV = 64 * KV, ROW = DK + DV, CB = ROW / E;
  constexpr int NQ = DK / (4 * E), NT = DV / 16 / CP, NL = ROW / 64;
  constexpr int TB = heads_tile_bytes(DK, DV), NST = heads_stages(TB, KS), WR = 4 / CP, ROWS = 16 * MR * WR;
  constexpr bool LATE = KS == 4 && CP == 1;  // values behind the softmax: four waves on a SIMD have 128 registers
  constexpr int BOX = 4 * MR * NT * 1024 + 2048 * MR;  // what a set of four waves hands over
  static_assert((KS - 1) * BOX <= KS * NST * TB, "fits the stages");
  static_assert(TB == KT * ROW * ES, "a tile");
  static_assert(heads_lds(TB, KS, KH_HEADS_BIAS_LDS) <= kHeadsLds, "fits a CU with the largest table");
  extern __shared__ __attribute__((aligned(1024))) char smem_raw[];
  const int lane = threadIdx.x & 63, wave8 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wave = wave8 & 3, ks = KS == 1 ? 0 : wave8 >> 2;
  const int fr = lane & 15, fh = lane >> 4, wr = wave % WR, wc = wave / WR;
  const int g = blockIdx.x, per = a.H / a.G;
  LatTile tl;
  int n_rows, row0;
  if (a.tiles) {
    // longest key ranges first; a launch of at most two workgroups per CU pairs the longest with the shortest instead
    const int nt = (int)gridDim.y, half = (nt + 1) >> 1, y = (int)blockIdx.y;
    tl = a.tiles[nt * a.G <= 512 && y >= half ? nt - 1 - (y - half) : y];
    n_rows = a.p.seg_n[tl.seg] * per;
    row0 = a.p.seg_row0[tl.seg];
  } else {
    const int nt = (per + ROWS - 1) / ROWS;
    tl.seg = (int)blockIdx.y / nt;
    tl.r0 = ((int)blockIdx.y - tl.seg * nt) * ROWS;
    n_rows = per;
    row0 = tl.seg;
  }
  const int pos0 = a.p.seg_pos0[tl.seg];
  const char* cache = (const char*)((const T*)a.cache + (size_t)a.p.seg_slot[tl.seg] * a.slot_elems + (size_t)g * ROW);
  // the lane's query rows
  int head[MR], tok[MR], my_pos[MR];
  bool live[MR];
#pragma unroll
  for (int q = 0; q < MR; ++q) {
    int r = tl.r0 + (wr * MR + q) * 16 + fr;
    live[q] = r < n_rows;
    if (!live[q]) r = n_rows - 1;
    tok[q] = r / per;
    head[q] = g * per + r - tok[q] * per;
    my_pos[q] = pos0 + tok[q];
  }
  auto pos_of = [&](int r) __attribute__((always_inline)) { return pos0 + (r < n_rows ? r : n_rows - 1) / per; };
  // positions of the first and last row of the wave; keys [k_lo, k_hi) of the workgroup
  const int p_lo = pos_of(tl.r0 + wr * MR * 16), p_hi = pos_of(tl.r0 + (wr + 1) * MR * 16 - 1);
  const int w_first = a.span.first(p_lo), w_full = a.span.first(p_hi);  // some row sees from, every row sees from
  const int n_keys = pos_of(tl.r0 + ROWS - 1) + 1;
  int k_lo = a.span.first(pos_of(tl.r0)), k_hi = n_keys;
  if (a.nsplit > 1) {
    const int len = lat_split_len(n_keys - k_lo, a.nsplit);
    k_lo += (int)blockIdx.z * len;
    if (k_lo >= n_keys) return;  // uniform; the merge does not read this split
    k_hi = k_lo + len < n_keys ? k_lo + len : n_keys;
  }
  int my_first[MR];
#pragma unroll
  for (int q = 0; q < MR; ++q) my_first[q] = a.span.first(my_pos[q]);
  // ---- queries as they lie, requested ahead of all that depends on the position
  float qx[MR][NQ][E];
#pragma unroll
  for (int q = 0; q < MR; ++q) {
    const size_t at = (size_t)(row0 + tok[q]) * a.ldr + (size_t)head[q] * a.dkr;
#pragma unroll
    for (int b = 0; b < NQ; ++b) {
      const int e0 = 4 * E * b + E * fh;  // dkr is a multiple of 16: a fragment is inside or outside as a whole
      if (a.raw_f32) {
#pragma unroll
        for (int i = 0; i < E; i += 4) {
          const f32x4 v = e0 < a.dkr ? *(const f32x4*)((const float*)a.raw + at + e0 + i) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int j = 0; j < 4; ++j) qx[q][b][i + j] = v[j];
        }
      } else {
        const bool in = e0 < a.dkr;
        const frag v = *(const frag*)((const T*)a.raw + at + (in ? e0 : 0));
#pragma unroll
        for (int i = 0; i < E; ++i) qx[q][b][i] = in ? (float)v[i] : 0.f;
      }
    }
  }
  // ---- staging: request j of a wave covers chunks (4 j + wave) 64 .. of the tile; slot s of row r holds chunk s ^ (r & 7)
  int kr[NL];
  unsigned kc[NL];
#pragma unroll
  for (int j = 0; j < NL; ++j) {
    const int c = (4 * j + wave) * 64 + lane;
    kr[j] = c / CB;
    kc[j] = (unsigned)(((c - kr[j] * CB) ^ (kr[j] & 7)) << 4);
  }
  const unsigned lds0 = (unsigned)__builtin_amdgcn_readfirstlane((int)kh_lds_addr(smem_raw)) + 1024u * wave + (unsigned)(ks * NST * TB);
  const unsigned row_b = (unsigned)(a.G * ROW * ES);
  int fill_row = (k_lo + ks * KT) % a.ring;  // cache row of the next tile to request
  auto issue = [&](int slot, int k0) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < NL; ++j) {
      const int k = k0 + kr[j] < n_keys ? kr[j] : n_keys - 1 - k0;  // rows behind the sequence's last may not be backed
      int r = fill_row + k;
      r = r < a.ring ? r : r - a.ring;
      dma_x4_keep(cache, (unsigned)r * row_b + kc[j], lds0 + (unsigned)(slot * TB + 4096 * j));
    }
    fill_row += KS * KT;
    if (fill_row >= a.ring) fill_row -= a.ring;
  };
  constexpr int DK0 = KS * KT;  // from one tile of a wave to its next
#pragma unroll
  for (int i = 0; i < NST - 1; ++i)
    if (k_lo + ks * KT + i * DK0 < k_hi) issue(i, k_lo + ks * KT + i * DK0);
  // ---- queries: norm and scale in registers (a row's elements lie in the four lanes fr, fr + 16, ...)
  frag fq[MR][NQ];
#pragma unroll
  for (int q = 0; q < MR; ++q) {
    float s = 0.f;
#pragma unroll
    for (int b = 0; b < NQ; ++b)
#pragma unroll
      for (int i = 0; i < E; ++i) s = __builtin_fmaf(qx[q][b][i], qx[q][b][i], s);
    s = xor16_sum(s);
    s = xor32_sum(s);
    const float f = a.qn ? a.scale2 / sqrtf(s / (float)a.dk + a.eps) : a.scale2;
#pragma unroll
    for (int b = 0; b < NQ; ++b)
#pragma unroll
      for (int i = 0; i < E; i += 4) {
        const f32x4 w = a.qn ? *(const f32x4*)(a.qn + 4 * E * b + E * fh + i) : f32x4{1.f, 1.f, 1.f, 1.f};
#pragma unroll
        for (int j = 0; j < 4; ++j) fq[q][b][i + j] = (T)(qx[q][b][i + j] * f * w[j]);
      }
  }
  // ---- distance bias: the group's rows of the table to LDS when a key of this workgroup is near enough to need them
  float* tab = (float*)(smem_raw + KS * NST * TB);
  float far[MR];
#pragma unroll
  for (int q = 0; q < MR; ++q) far[q] = a.bias ? a.bias[(size_t)head[q] * a.nbias + a.nbias - 1] : 0.f;
  if (a.bias && a.bias_lds && pos_of(tl.r0) - (k_hi - 1) < a.nbias - 1)
    for (int i = threadIdx.x; i < per * a.nbias; i += 256 * KS) tab[i] = a.bias[(size_t)g * per * a.nbias + i];
  // a decoded token's gate logits, ahead of their use
  constexpr bool EARLY = CP == 4 && KS > 1;
  f32x4 zg[EARLY ? NT : 1];
  if constexpr (EARLY) {
    if (a.g_off >= 0 && a.raw_f32 && ks == 0) {
      const float* z = (const float*)a.raw + (size_t)(row0 + tok[0]) * a.ldr + a.g_off + (size_t)head[0] * a.dvr;
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        const int c = (wc * NT + n) * 16 + 4 * fh;
        zg[n] = *(const f32x4*)(z + (c < a.dvr ? c : 0));
      }
    }
  }
  float m[MR], l[MR];
  f32x4 o[MR][NT];
#pragma unroll
  for (int q = 0; q < MR; ++q) {
    const bool sinks = a.sink && (a.nsplit == 1 || blockIdx.z == 0) && ks == 0;
    m[q] = sinks ? 0.f : -1e30f;  // finite: a row without a visible key yet keeps weights of zero, not NaN
    l[q] = sinks && fh == 0 ? 1.f : 0.f;
#pragma unroll
    for (int n = 0; n < NT; ++n) o[q][n] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  int slot = -1, fill = NST - 2;
  for (int kb = k_lo; kb < k_hi; kb += DK0) {
    const int k0 = kb + ks * KT;
    slot = slot + 1 == NST ? 0 : slot + 1;
    fill = fill + 1 == NST ? 0 : fill + 1;
    // this stage has landed when only the younger NST - 2 stages are outstanding
    if (k0 + (NST - 2) * DK0 < k_hi) wait_vm<(NST - 2) * NL>();
    else wait_vm<0>();
    __syncthreads();
    if (k0 + (NST - 1) * DK0 < k_hi) issue(fill, k0 + (NST - 1) * DK0);
    // nothing in this tile for the wave (barriers stay uniform)
    if (k0 > p_hi || k0 + KT <= w_first || (KS > 1 && k0 >= k_hi)) continue;
    const char* Kt = smem_raw + (ks * NST + slot) * TB;
    f32x4 s[MR][NS];
#pragma unroll
    for (int q = 0; q < MR; ++q)
#pragma unroll
      for (int n = 0; n < NS; ++n) s[q][n] = f32x4{0.f, 0.f, 0.f, 0.f};
    frag fk[NQ][NS];
#pragma unroll
    for (int b = 0; b < NQ; ++b)
#pragma unroll
      for (int n = 0; n < NS; ++n) {
        const int k = n * 16 + fr;
        fk[b][n] = *(const frag*)(Kt + ((size_t)k * CB + ((4 * b + fh) ^ (k & 7))) * 16);
      }
    frag fv[NT];  // requested with the keys: they arrive under the scores and the softmax
#pragma unroll
    for (int n = 0; n < (LATE ? 0 : NT); ++n) fv[n] = lat_col<CB>(Kt, DK + (wc * NT + n) * 16, lane, T());
#pragma unroll
    for (int b = 0; b < NQ; ++b)
#pragma unroll
      for (int n = 0; n < NS; ++n)
#pragma unroll
        for (int q = 0; q < MR; ++q) s[q][n] = TL::mma(fk[b][n], fq[q][b], s[q][n]);
    // lane: keys k0 + 16 n + 4 fh + i of its rows
    frag p[MR];
    const bool edge = k0 + KT - 1 > p_lo || k0 < w_full || k0 + KT > k_hi;
    // (by the tile's last key, not its last row, as where the table is copied: or a wave would read what was not)
    const bool near = a.bias && p_lo - ((k0 + KT < k_hi ? k0 + KT : k_hi) - 1) < a.nbias - 1;
#pragma unroll
    for (int q = 0; q < MR; ++q) {
      if (near) {  // two loads of known address space, not one of a selected address
        const int d0 = my_pos[q] - k0 - 4 * fh;
        auto add = [&](const float* row) __attribute__((always_inline)) {
#pragma unroll
          for (int n = 0; n < NS; ++n)
#pragma unroll
            for (int i = 0; i < 4; ++i) s[q][n][i] += row[min(max(d0 - 16 * n - i, 0), a.nbias - 1)];
        };
        if (a.bias_lds) add(tab + (head[q] - g * per) * a.nbias);
        else add(a.bias + (size_t)head[q] * a.nbias);
      }
      if (edge) {
#pragma unroll
        for (int n = 0; n < NS; ++n)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int k = k0 + 16 * n + 4 * fh + i;
            s[q][n][i] = k <= my_pos[q] && k >= my_first[q] && k < k_hi ? s[q][n][i] : -INFINITY;
          }
      }
      const float add = near ? 0.f : far[q];  // the same for every key of a far tile: joins the maximum
      float mx = s[q][0][0];
#pragma unroll
      for (int n = 0; n < NS; ++n)
#pragma unroll
        for (int i = 0; i < 4; ++i) mx = fmaxf(mx, s[q][n][i]);
      mx += add;
      // the running maximum rarely moves after the first tiles: rescale only when some row's does
      if (__any(mx > m[q])) {
        mx = fmaxf(mx, m[q]);
        mx = xor16_max(mx);
        mx = xor32_max(mx);
        const float f = __builtin_amdgcn_exp2f(m[q] - mx);
        m[q] = mx;
        l[q] *= f;
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
          for (int i = 0; i < 4; ++i) o[q][n][i] *= f;
      }
      const float base = m[q] - add;
      float sum = 0.f;
#pragma unroll
      for (int n = 0; n < NS; ++n)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float e = __builtin_amdgcn_exp2f(s[q][n][i] - base);
          sum += e;
          p[q][4 * n + i] = (T)e;
        }
      l[q] += sum;
    }
    if constexpr (LATE) {
      asm volatile("" ::: "memory");
#pragma unroll
      for (int n = 0; n < NT; ++n) fv[n] = lat_col<CB>(Kt, DK + (wc * NT + n) * 16, lane, T());
    }
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int q = 0; q < MR; ++q) o[q][n] = TL::mma(fv[n], p[q], o[q][n]);
  }
#pragma unroll
  for (int q = 0; q < MR; ++q) {
    l[q] = xor16_sum(l[q]);
    l[q] = xor32_sum(l[q]);
  }
  if (KS > 1) {  // the sets of waves hold the same rows and columns lane by lane
    __syncthreads();
    auto box = [&](int set) __attribute__((always_inline)) { return (f32x4*)(smem_raw + (set - 1) * BOX) + wave * MR * NT * 64 + lane; };
    auto ml = [&](int set) __attribute__((always_inline)) {
      return (float*)(smem_raw + (set - 1) * BOX + 4 * MR * NT * 1024) + wave * MR * 128 + lane;
    };
    if (ks) {
#pragma unroll
      for (int q = 0; q < MR; ++q) {
#pragma unroll
        for (int n = 0; n < NT; ++n) box(ks)[(q * NT + n) * 64] = o[q][n];
        ml(ks)[q * 128] = m[q];
        ml(ks)[q * 128 + 64] = l[q];
      }
    }
    __syncthreads();
    if (ks) return;
#pragma unroll
    for (int set = 1; set < KS; ++set)
#pragma unroll
      for (int q = 0; q < MR; ++q) {
        const float m1 = ml(set)[q * 128], l1 = ml(set)[q * 128 + 64], mx = fmaxf(m[q], m1);
        const float f0 = __builtin_amdgcn_exp2f(m[q] - mx), f1 = __builtin_amdgcn_exp2f(m1 - mx);
        m[q] = mx;
        l[q] = __builtin_fmaf(l1, f1, l[q] * f0);
#pragma unroll
        for (int n = 0; n < NT; ++n) {
          const f32x4 b = box(set)[(q * NT + n) * 64];
#pragma unroll
          for (int i = 0; i < 4; ++i) o[q][n][i] = __builtin_fmaf(b[i], f1, o[q][n][i] * f0);
        }
      }
  }
#pragma unroll
  for (int q = 0; q < MR; ++q) {
    const float sum = l[q];
    if (!live[q]) continue;
    if (a.nsplit == 1) {
      const float inv = 1.0f / sum;
      const size_t t = (size_t)(row0 + tok[q]);
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        const int c = (wc * NT + n) * 16 + 4 * fh;
        if (c >= a.dvr) continue;
        f32x4 v;
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = o[q][n][i] * inv;
        if (a.g_off >= 0) {
          const size_t at = t * a.ldr + a.g_off + (size_t)head[q] * a.dvr + c;
          f32x4 z;
          if (EARLY && a.raw_f32) z = zg[EARLY ? n : 0];
          else z = a.raw_f32 ? *(const f32x4*)((const float*)a.raw + at) : quad_f((const T*)a.raw + at);
#pragma unroll
          for (int i = 0; i < 4; ++i) v[i] *= sigmoid1(z[i]);
        }
        const size_t to = t * a.ldo + (size_t)head[q] * a.dvr + c;
        if (a.out_f32) *(f32x4*)((float*)a.out + to) = v;
        else *(typename TL::quad*)((T*)a.out + to) = to_quad<T>(v);
      }
    } else {
      float* pt = a.part + (((size_t)(row0 + tok[q]) * a.H + head[q]) * a.nsplit + blockIdx.z) * (size_t)(DV + 4);
#pragma unroll
      for (int n = 0; n < NT; ++n) *(f32x4*)(pt + (wc * NT + n) * 16 + 4 * fh) = o[q][n];
      if (wc == 0 && fh == 0) {
        pt[DV] = m[q];
        pt[DV + 1] = sum;
      }
    }
  }
}

// One token per sequence over at most `keys` keys: is a group one workgroup, without splits and the launch that merges them?
// Where its keys and values are 64 KB, two microseconds of what one CU can pull; the merge costs three (8 heads of 128 on 2
// groups in fp32, 24 ... 64 keys: 6.7 + 4.7 -> 9.0 us a layer; Gusorax 1024 x 8, 24 + 40 tokens 12 255 -> 11 950).
__host__ __device__ inline bool heads_one_split(int keys, int dkp, int dvp, size_t elem) { return (size_t)keys * (dkp + dvp) * elem <= 64 * 1024; }
// rows of a workgroup's tile: 16, 64 or, for bf16 heads of up to 128, 128 (two row tiles per wave share every operand)
static inline bool heads_wide_rows(int dkp, int dvp, size_t elem) { return elem == 2 && dkp <= 128 && dvp <= 128; }
template <class T>
int heads_attn_launch(hipStream_t s, HeadsArgs a, int ntiles, int rows);
extern template int heads_attn_launch<bf16>(hipStream_t, HeadsArgs, int, int);
extern template int heads_attn_launch<float>(hipStream_t, HeadsArgs, int, int);
}  // namespace khm
