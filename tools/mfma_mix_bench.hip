// What the matrix cores take beside the rest of the prefill kernel's tile loop (prefill_fa_tile.cuh), on one CU and on all of them:
//   hipcc --offload-arch=gfx950 -Xclang -target-feature -Xclang -packed-fp32-ops -O3 tools/mfma_mix_bench.hip -o tools/mfma_mix_bench && tools/mfma_mix_bench
// A loop of 16 slots, each a v_mfma_f32_32x32x16_bf16 (32 cycles of a SIMD's matrix core) and, by MODE, an LDS fragment of 16 bytes a lane for
// its A operand (four slots ahead) and the softmax of two scores (2 fma, 2 exp2, 2 add, 1 pack).  One workgroup of four waves (one per SIMD) or
// of eight on one CU, then 256 of them.
// On one CU two waves per SIMD take 15.4 ns per MFMA, 13.6 of them the MFMA's own 32 cycles: the vector work of one wave hides under the
// MFMA of the other.  With all CUs running MFMA alone takes 21 .. 23 ns, 32 cycles at 1.4 .. 1.5 GHz instead of 2.35, and the whole mix 26.4 ..
// 27.4: the chip is at its power limit, and what is left to gain there is less work, not another order of it.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <utility>

typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) unsigned u32x4;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;

#define CHECK(e)                                                                       \
  do {                                                                                 \
    if ((e) != hipSuccess) { printf("%s failed\n", #e); return 1; }                    \
  } while (0)

template <int... I, typename F>
__device__ __forceinline__ void static_for_(std::integer_sequence<int, I...>, F&& f) { (f(std::integral_constant<int, I>{}), ...); }
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) { static_for_(std::make_integer_sequence<int, N>{}, f); }
__device__ __forceinline__ f32x16 mfma(u32x4 a, u32x4 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ uint32_t pack(float a, float b) {
  const bf16x2 r = {(__bf16)a, (__bf16)b};
  return __builtin_bit_cast(uint32_t, r);
}

// MODE bits: 1 MFMAs in one dependent chain (else four), 2 LDS fragments, 4 fma + add + pack, 8 exp2, 16 no MFMA
template <int MODE>
__global__ __launch_bounds__(512) void mix_kernel(const float* in, float* out, int iters) {
  __shared__ __attribute__((aligned(1024))) uint8_t lds[65536];
  const int lane = threadIdx.x & 63;
  for (int i = threadIdx.x; i < 65536 / 4; i += blockDim.x) ((float*)lds)[i] = in[i & 1023];
  __syncthreads();
  f32x16 acc[4], s = {0};
  u32x4 a, b[4];
  for (int i = 0; i < 4; ++i)
    for (int r = 0; r < 16; ++r) acc[i][r] = in[lane + r];
  for (int r = 0; r < 16; ++r) s[r] = in[lane * 2 + r];
  for (int j = 0; j < 4; ++j) {
    a[j] = __float_as_uint(in[lane + j]);
    for (int i = 0; i < 4; ++i) b[i][j] = __float_as_uint(in[lane + 7 * j + i]);
  }
  uint32_t rd = (lane & 31) * 256 + (((lane >> 5) ^ (lane & 15)) << 4);   // at most 8176 + 16 bytes, + 7 x 4096 below
  u32x4 f[4] = {a, a, a, a};
  float sum = 0.f;
  const float scale = in[5], top = in[6];
  for (int it = 0; it < iters; ++it) {
    static_for<16>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      constexpr int ai = (MODE & 1) ? i / 8 : i % 4;
      const u32x4 fr = (MODE & 2) ? f[i % 4] : a;
      if (MODE & 2) f[i % 4] = *reinterpret_cast<const u32x4*>(lds + rd + ((i & 7) << 12));
      if (!(MODE & 16)) acc[ai] = mfma(fr, b[i % 4], acc[ai]);
      if (MODE & 12) {
        float e0 = s[i], e1 = s[(i + 1) & 15];
        if (MODE & 4) { e0 = fmaf(e0, scale, -top); e1 = fmaf(e1, scale, -top); }
        if (MODE & 8) { e0 = __builtin_amdgcn_exp2f(e0); e1 = __builtin_amdgcn_exp2f(e1); }
        if (MODE & 4) { sum += e0; sum += e1; }
        const uint32_t w = pack(e0, e1);
        asm volatile("" ::"v"(w));
      }
      __builtin_amdgcn_sched_barrier(0);
    });
    if (MODE & 2) asm volatile("" : "+v"(rd));
    if (MODE & 12) asm volatile("" : "+v"(s));
  }
  float r = sum;
  for (int i = 0; i < 4; ++i)
    for (int j = 0; j < 16; ++j) r += acc[i][j];
  out[blockIdx.x * blockDim.x + threadIdx.x] = r;
}

template <int MODE>
int run(const char* name, const float* in, float* out) {
  for (int threads : {256, 512})
    for (int wgs : {1, 256}) {
      const int iters = 4000;
      hipEvent_t e0, e1;
      CHECK(hipEventCreate(&e0));
      CHECK(hipEventCreate(&e1));
      hipLaunchKernelGGL((mix_kernel<MODE>), dim3(wgs), dim3(threads), 0, 0, in, out, iters);
      CHECK(hipEventRecord(e0));
      hipLaunchKernelGGL((mix_kernel<MODE>), dim3(wgs), dim3(threads), 0, 0, in, out, iters);
      CHECK(hipEventRecord(e1));
      CHECK(hipEventSynchronize(e1));
      float ms;
      CHECK(hipEventElapsedTime(&ms, e0, e1));
      printf("%-34s waves per SIMD %d  workgroups %3d  %6.1f ns a slot, %5.1f ns per MFMA of a SIMD\n", name, threads / 256, wgs, ms * 1e6 / (iters * 16),
             ms * 1e6 / (iters * 16) / (threads / 256));
      fflush(stdout);
    }
  return 0;
}

int main() {
  float *in, *out;
  CHECK(hipMalloc(&in, 8192));
  CHECK(hipMalloc(&out, 256 * 512 * sizeof(float)));
  static float h[2048];
  for (int i = 0; i < 2048; ++i) h[i] = ((i * 37) % 101 - 50) * 0.01f;
  CHECK(hipMemcpy(in, h, sizeof(h), hipMemcpyHostToDevice));
  int bad = run<0>("MFMA, four chains", in, out);
  bad |= run<1>("MFMA, one chain", in, out);
  bad |= run<16 + 12>("softmax alone", in, out);
  bad |= run<12>("MFMA + softmax", in, out);
  bad |= run<2>("MFMA + LDS", in, out);
  bad |= run<14>("MFMA + LDS + softmax", in, out);
  bad |= run<15>("one chain + LDS + softmax", in, out);
  return bad;
}
