// kh_heads.hip — launcher and instantiations of the attention over grouped heads (kh_heads.h).
#include <vector>

#include "kh_heads.h"

namespace khm {

template <class T>
int heads_attn_launch(hipStream_t s, HeadsArgs a, int ntiles, int rows) {
  if (a.dkp % 64 || a.dvp % 64 || a.dkp > KH_HEADS_MAX_DIM || a.dvp > KH_HEADS_MAX_DIM || a.dkr > a.dkp || a.dvr > a.dvp ||
      a.dkr % 16 || a.dvr % 16 || a.ldr % 16 || a.G <= 0 || a.H % a.G || a.ring <= 0 || a.nsplit < 1 || ntiles <= 0)
    return KH_ERR_INTERNAL;
  const size_t table = (size_t)(a.H / a.G) * a.nbias * sizeof(float);
  a.bias_lds = a.bias && heads_table_lds(table);
  auto go = [&](auto kern, size_t stage, int ks) -> int {
    const size_t lds = heads_lds((int)stage, ks, a.bias ? table : 0);
    if (lds > 64 * 1024) {
      struct Done { int dev; const void* fn; size_t lds; };
      static thread_local std::vector<Done> done;
      int dev = 0;
      (void)hipGetDevice(&dev);
      bool hit = false;
      for (const auto& d : done) hit = hit || (d.dev == dev && d.fn == (const void*)kern && d.lds >= lds);
      if (!hit) {
        const hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return (int)e;
        done.push_back({dev, (const void*)kern, lds});
      }
    }
    hipLaunchKernelGGL(kern, dim3(a.G, ntiles, a.nsplit), dim3(256 * ks), lds, s, a);
    return KH_OK;
  };
  auto by_rows = [&](auto kn, auto kv) -> int {
    constexpr int KN = decltype(kn)::value, KV = decltype(kv)::value;
    const size_t stage = heads_tile_bytes(a.dkp, a.dvp);
    if constexpr (KN + KV <= 4)  // one token per sequence and one split: four sets of waves, a key tile each
      if (rows == 16 && !a.tiles && a.nsplit == 1) return go(k_heads_attn<T, KN, KV, 4, 1, 4>, stage, 4);
    if (rows == 16) return go(k_heads_attn<T, KN, KV, 4, 1, 1>, stage, 1);
    // at most one workgroup per CU: two sets of waves, which share the keys (1100 tokens of 2 x 4 heads of 128, 138 workgroups:
    // 37.2 -> 27.6 us; four sets on tiles of 32 rows 25.9, at twice the key traffic), or four in bf16, where heads of 128 leave
    // the registers (27.9 -> 25.1 in another session; in fp32 they spill) and what the sets hand over fits the stages.  Keys and
    // values of more than 256 elements together need the registers of a wave alone on its SIMD.
    if constexpr (KN + KV <= 4)
      if (rows == 64 && a.tiles && (long)ntiles * a.G <= 256) {
        if constexpr (sizeof(T) == 2 && KN == 2 && KV == 2) return go(k_heads_attn<T, KN, KV, 1, 1, 4>, stage, 4);
        else return go(k_heads_attn<T, KN, KV, 1, 1, 2>, stage, 2);
      }
    if (rows == 64) return go(k_heads_attn<T, KN, KV, 1, 1, 1>, stage, 1);
    if constexpr (sizeof(T) == 2 && KN <= 2 && KV <= 2)
      if (rows == 128) return go(k_heads_attn<T, KN, KV, 1, 2, 1>, stage, 1);
    return KH_ERR_INTERNAL;
  };
  auto by_value = [&](auto kn) -> int {
    switch (a.dvp / 64) {
      case 1: return by_rows(kn, std::integral_constant<int, 1>());
      case 2: return by_rows(kn, std::integral_constant<int, 2>());
      case 3: return by_rows(kn, std::integral_constant<int, 3>());
      default: return by_rows(kn, std::integral_constant<int, 4>());
    }
  };
  switch (a.dkp / 64) {
    case 1: return by_value(std::integral_constant<int, 1>());
    case 2: return by_value(std::integral_constant<int, 2>());
    case 3: return by_value(std::integral_constant<int, 3>());
    default: return by_value(std::integral_constant<int, 4>());
  }
}
template int heads_attn_launch<bf16>(hipStream_t, HeadsArgs, int, int);
template int heads_attn_launch<float>(hipStream_t, HeadsArgs, int, int);

}  // namespace khm

extern "C" int kh_plan_heads_lds(int32_t key, int32_t value, int32_t sets, int32_t table, int32_t* bytes) {
  using namespace khm;
  if (!bytes || key <= 0 || value <= 0 || table < 0 || (sets != 1 && sets != 2 && sets != 4)) return KH_ERR_INVALID_ARG;
  const int kp = (key + 63) / 64 * 64, vp = (value + 63) / 64 * 64;
  if (kp > KH_HEADS_MAX_DIM || vp > KH_HEADS_MAX_DIM || (sets > 1 && kp + vp > KH_HEADS_MAX_DIM)) return KH_ERR_UNSUPPORTED;
  *bytes = (int32_t)heads_lds(heads_tile_bytes(kp, vp), sets, (size_t)table);
  return KH_OK;
}
