// Streaming-read rate of 16-byte global loads by cache policy bits (gfx950): plain, nt, sc1, sc0 sc1, sc1 nt,
// sc0 sc1 nt.  512 workgroups x 256 threads (two per CU, like the decode kernel), 8 loads in flight per lane,
// two 512 MiB buffers alternated (no Infinity-Cache reuse), steady state (each policy runs ~40 ms first).
// hipcc --offload-arch=gfx950 -Xclang -target-feature -Xclang -packed-fp32-ops -O3 tools/loadpolicy_bench.hip -o tools/loadpolicy_bench
// Measured (MI355X, 512 workgroups): plain 6.21, nt 6.89, sc1 6.20, sc0 sc1 6.19, sc1 nt 6.88, sc0 sc1 nt 6.85, sc0 nt 6.87 TB/s
// (768 / 2048 workgroups: the same picture, 6.1 vs 6.7-6.9): only the nt bit matters; ~6.9 TB/s = 86 % of the 8 TB/s
// spec is the streaming-read ceiling, and the decode kernel's steady 6.55 TB/s is 95 % of it.
#include <hip/hip_runtime.h>
#include <stdio.h>
#include <stdlib.h>
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;
#define CK(x) do { hipError_t e = (x); if (e != hipSuccess) { printf("%s: %s\n", #x, hipGetErrorString(e)); exit(1); } } while (0)

#define LOADP(dst, ptr, POL) asm volatile("global_load_dwordx4 %0, %1, off " POL : "=v"(dst) : "v"(ptr) : "memory")

template <int P>
__global__ __launch_bounds__(256) void rd(const u32x4* __restrict__ p, size_t n_per_wg, unsigned* sink) {
  const u32x4* base = p + (size_t)blockIdx.x * n_per_wg;
  u32x4 acc = {0, 0, 0, 0};
  for (size_t i = threadIdx.x; i + 7 * 256 < n_per_wg; i += 256 * 8) {
    u32x4 v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const u32x4* q = base + i + (size_t)j * 256;
      if (P == 0) LOADP(v[j], q, "");
      if (P == 1) LOADP(v[j], q, "nt");
      if (P == 2) LOADP(v[j], q, "sc1");
      if (P == 3) LOADP(v[j], q, "sc0 sc1");
      if (P == 4) LOADP(v[j], q, "sc1 nt");
      if (P == 5) LOADP(v[j], q, "sc0 sc1 nt");
      if (P == 6) LOADP(v[j], q, "sc0 nt");
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
    for (int j = 0; j < 8; ++j) acc ^= v[j];
  }
  if ((acc.x ^ acc.y ^ acc.z ^ acc.w) == 0x12345678u) sink[0] = 1;
}

template <int P> float run(const u32x4* a, const u32x4* b, size_t n_per_wg, unsigned* sink, int wgs) {
  hipEvent_t e0, e1; CK(hipEventCreate(&e0)); CK(hipEventCreate(&e1));
  for (int i = 0; i < 400; ++i) hipLaunchKernelGGL(rd<P>, dim3(wgs), dim3(256), 0, 0, (i & 1) ? a : b, n_per_wg, sink);
  CK(hipDeviceSynchronize());
  CK(hipEventRecord(e0));
  for (int i = 0; i < 200; ++i) hipLaunchKernelGGL(rd<P>, dim3(wgs), dim3(256), 0, 0, (i & 1) ? a : b, n_per_wg, sink);
  CK(hipEventRecord(e1)); CK(hipEventSynchronize(e1));
  float ms; CK(hipEventElapsedTime(&ms, e0, e1));
  return ms / 200 * 1e3f;
}

int main() {
  const size_t bytes = 512ull << 20;
  unsigned char *a, *b; unsigned* sink;
  CK(hipMalloc(&a, bytes)); CK(hipMalloc(&b, bytes)); CK(hipMalloc(&sink, 4));
  CK(hipMemset(a, 1, bytes)); CK(hipMemset(b, 2, bytes));
  const char* names[7] = {"plain", "nt", "sc1", "sc0 sc1", "sc1 nt", "sc0 sc1 nt", "sc0 nt"};
  for (int wgs : {512, 768, 2048}) {
    const size_t n_per_wg = bytes / 16 / wgs;
    float us[7];
    us[0] = run<0>((const u32x4*)a, (const u32x4*)b, n_per_wg, sink, wgs);
    us[1] = run<1>((const u32x4*)a, (const u32x4*)b, n_per_wg, sink, wgs);
    us[2] = run<2>((const u32x4*)a, (const u32x4*)b, n_per_wg, sink, wgs);
    us[3] = run<3>((const u32x4*)a, (const u32x4*)b, n_per_wg, sink, wgs);
    us[4] = run<4>((const u32x4*)a, (const u32x4*)b, n_per_wg, sink, wgs);
    us[5] = run<5>((const u32x4*)a, (const u32x4*)b, n_per_wg, sink, wgs);
    us[6] = run<6>((const u32x4*)a, (const u32x4*)b, n_per_wg, sink, wgs);
    for (int p = 0; p < 7; ++p) printf("wgs=%4d %-11s %7.1f us  %.2f TB/s\n", wgs, names[p], us[p], bytes / us[p] / 1e6);
  }
  return 0;
}
