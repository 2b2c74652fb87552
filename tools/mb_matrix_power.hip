// What the power limit leaves of the matrix rate: the stage loop of a 128 x 128 tile of the pair GEMMs (csrc/kh_pair.h), one ingredient
// after the other, on zeros and on random numbers.  512 workgroups of four waves, two a CU, 64 KB of LDS each.
//   hipcc --offload-arch=gfx950 -Xclang -target-feature -Xclang -packed-fp32-ops -O3 -o mb_matrix_power tools/mb_matrix_power.hip
// Prints us a launch, the clock it ran at, the matrix rate, and what a CU reads from LDS and requests into it.
#include <hip/hip_runtime.h>
#include <stdio.h>

#include <vector>
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

enum { BARRIER = 1, REQUESTS = 2, PRIO = 4 };

__device__ __forceinline__ void request16(const char* base, unsigned off, unsigned lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(lds) : "memory", "m0");
}
__device__ __forceinline__ void wait_requests() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// A stage: READS fragments from LDS, MATS matrix instructions, VALUS fused multiply-adds; with REQUESTS eight of 1 KB a wave into
// the other half of the LDS.  src holds span + 64 KB; a wave's requests cover 8 KB from a multiple of 8 KB below span.
template <int READS, int MATS, int VALUS, int F>
__global__ __launch_bounds__(256, 2) void k_stages(float* out, long* clk, const char* src, int stages, unsigned span) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  constexpr int NF = READS > 0 ? READS : 4;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), fr = lane & 15, fh = lane >> 4;
  for (int i = threadIdx.x; i < 65536 / 4; i += 256) ((float*)smem)[i] = ((const float*)src)[i];
  __syncthreads();
  f32x4 acc[16];
  for (auto& a : acc) a = f32x4{0, 0, 0, 0};
  f16x8 x[NF];
  for (int j = 0; j < NF; ++j) x[j] = ((const f16x8*)smem)[j * 64 + lane];
  float v[8];
  for (int i = 0; i < 8; ++i) v[i] = lane * 1e-3f + i;
  unsigned off = (unsigned)((blockIdx.x * 4 + wave) * 8192u) % span + lane * 16;
  const unsigned lds = (unsigned)(unsigned long)(__attribute__((address_space(3))) char*)smem + wave * 1024;
  const long c0 = clock64(), w0 = wall_clock64();
  for (int it = 0; it < stages; ++it) {
    int half = (it & 1) * 32768;
    asm volatile("" : "+s"(half));
    if (F & REQUESTS) wait_requests();
    if (F & BARRIER) __syncthreads();
    if (F & REQUESTS) {
#pragma unroll
      for (int j = 0; j < 8; ++j) request16(src, off + j * 1024u, __builtin_amdgcn_readfirstlane(lds + (half ^ 32768) + j * 4096));
      off += 256 * 32768u;
      off = off >= span ? off - span : off;
    }
#pragma unroll
    for (int j = 0; j < READS; ++j) {
      const int r = (j >> 1) * 16 + fr, swz = ((r & 2) << 1) | ((r & 4) ? 3 : 0);
      x[j] = *(const f16x8*)(smem + half + ((r * 128) & 32767) + ((((j & 1) * 4 + fh) ^ swz) << 4));
    }
    if (READS) __builtin_amdgcn_sched_barrier(0);
    if (F & PRIO) __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int j = 0; j < MATS; ++j)
      acc[j & 15] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x[READS ? j % NF : j & 3], x[READS ? (j * 7 + 3) % NF : (j + 1) & 3], acc[j & 15], 0, 0, 0);
#pragma unroll
    for (int j = 0; j < VALUS; ++j) v[j & 7] = __builtin_fmaf(v[j & 7], 1.0001f, 0.5f);
    if (F & PRIO) __builtin_amdgcn_s_setprio(0);
  }
  wait_requests();
  const long c1 = clock64(), w1 = wall_clock64();
  float s = 0;
  for (auto& a : acc) s += a[0];
  for (float e : v) s += e;
  out[blockIdx.x * 256 + threadIdx.x] = s;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    clk[0] = c1 - c0;
    clk[1] = w1 - w0;
  }
}

#define CK(x)                                                          \
  do {                                                                 \
    const hipError_t e_ = (x);                                         \
    if (e_ != hipSuccess) {                                            \
      fprintf(stderr, "%s: %s\n", #x, hipGetErrorString(e_));          \
      return 1;                                                        \
    }                                                                  \
  } while (0)

static float* g_out;
static long* g_clk;

template <int READS, int MATS, int VALUS, int F>
int go(const char* name, const char* src, unsigned span, int stages = 3000) {
  auto kern = k_stages<READS, MATS, VALUS, F>;
  CK(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, 65536));
  hipEvent_t a, b;
  CK(hipEventCreate(&a));
  CK(hipEventCreate(&b));
  float ms = 0;
  for (int r = 0; r < 4; ++r) {
    CK(hipEventRecord(a));
    hipLaunchKernelGGL(kern, dim3(512), dim3(256), 65536, 0, g_out, g_clk, src, stages, span);
    CK(hipGetLastError());
    CK(hipEventRecord(b));
    CK(hipEventSynchronize(b));
    CK(hipEventElapsedTime(&ms, a, b));
  }
  long c[2];
  CK(hipMemcpy(c, g_clk, 16, hipMemcpyDeviceToHost));
  const double us = ms * 1e3;
  printf("%-52s %8.1f us  %.2f GHz  %.2f PFLOP/s  LDS %3.0f B/ns a CU  requests %3.0f\n", name, us, (double)c[0] / c[1] * 0.1,
         512.0 * 4 * MATS * 16384.0 * stages / (us * 1e-6) / 1e15, 2.0 * 4 * READS * 1024.0 * stages / (us * 1e3),
         F & REQUESTS ? 2.0 * 32768 * stages / (us * 1e3) : 0.0);
  fflush(stdout);
  return 0;
}

int main() {
  const unsigned l2 = 16u << 20, cache = 128u << 20, hbm = 512u << 20;
  char *rnd, *zero;
  CK(hipMalloc(&g_out, 512 * 256 * 4));
  CK(hipMalloc(&g_clk, 64));
  CK(hipMalloc(&rnd, (size_t)hbm + 65536));
  CK(hipMalloc(&zero, (size_t)l2 + 65536));
  CK(hipMemset(zero, 0, (size_t)l2 + 65536));
  std::vector<_Float16> h(((size_t)hbm + 65536) / 2);
  unsigned s = 1;
  for (auto& e : h) {
    s = s * 1664525u + 1013904223u;
    e = (_Float16)(((int)(s >> 8) % 20001 - 10000) * 1e-4f);
  }
  CK(hipMemcpy(rnd, h.data(), h.size() * 2, hipMemcpyHostToDevice));
  return go<0, 48, 0, 0>("48 matrix instructions a stage, zeros", zero, l2) || go<0, 48, 0, 0>("the same, random numbers", rnd, l2) ||
         go<20, 48, 0, 0>("with 20 fragments from LDS, zeros", zero, l2) || go<20, 48, 0, 0>("the same, random numbers", rnd, l2) ||
         go<20, 48, 80, 0>("and 80 vector instructions (the split)", rnd, l2) || go<20, 48, 80, BARRIER>("and a barrier", rnd, l2) ||
         go<20, 48, 80, BARRIER | REQUESTS | PRIO>("and requests of 32 KB, from 16 MB", rnd, l2) ||
         go<20, 48, 80, BARRIER | REQUESTS | PRIO>("the same, from 128 MB", rnd, cache) ||
         go<20, 48, 80, BARRIER | REQUESTS | PRIO>("the same, from 512 MB", rnd, hbm, 1000) ||
         go<0, 0, 0, BARRIER | REQUESTS>("requests alone, from 16 MB", rnd, l2) ||
         go<0, 0, 0, BARRIER | REQUESTS>("requests alone, from 128 MB", rnd, cache) ||
         go<0, 0, 0, BARRIER | REQUESTS>("requests alone, from 512 MB", rnd, hbm, 1000);
}
