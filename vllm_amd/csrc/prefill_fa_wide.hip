// The tile kernel's four-wave form (head sizes 136 .. 256), in a file of its own: one wave per SIMD has 512 registers, of which
// vector instructions reach the first 256.  By default the compiler then puts every MFMA result into the other half and copies S^T
// back for the softmax (64 .. 128 copies a tile); built with -amdgpu-mfma-vgpr-form (Makefile) it keeps them where they are used
// (us, head 256, 16 / 8 heads: flash fp8 1 x 4000 201 -> 183, 16-bit 201 -> 192; x layout fp8 2000 over 2000 182 -> 178, 200 fresh 24.5 -> 22.3,
// 16-bit 100 over 1000 40.5 -> 37.2).
#include "prefill_fa_tile.cuh"

namespace va {

template <typename T, bool FP8, bool PREFIX>
static void launch(const FaParams& p, dim3 grid, hipStream_t st) {
#define FA_WIDE(CAP_, S_) hipLaunchKernelGGL((fa::fa_fwd_kernel<T, FP8, PREFIX, 256, 4, CAP_, S_>), grid, dim3(256), 0, st, p)
  if constexpr (!PREFIX) {
    if (p.softcap > 0.f) {
      if (p.num_segments > 1) FA_WIDE(true, true); else FA_WIDE(true, false);
      return;
    }
  }
  if (p.num_segments > 1) FA_WIDE(false, true); else FA_WIDE(false, false);
#undef FA_WIDE
}

void launch_fa_wide(const FaParams& p, int dtype, bool fp8, dim3 grid, hipStream_t st) {
#define FA_WIDE(T_)                                                                                     \
  do {                                                                                                  \
    if (p.prefix) { if (fp8) launch<T_, true, true>(p, grid, st); else launch<T_, false, true>(p, grid, st); } \
    else { if (fp8) launch<T_, true, false>(p, grid, st); else launch<T_, false, false>(p, grid, st); }  \
  } while (0)
  if (dtype == VLLM_AMD_BF16) FA_WIDE(bf16_t); else FA_WIDE(f16_t);
#undef FA_WIDE
}

}  // namespace va

#ifdef VA_PROBES
extern "C" int vllm_amd_probe_fa_wide_stamps(unsigned long long* dst, int nwg) {
  return hipMemcpyFromSymbol(dst, HIP_SYMBOL(va::fa::g_fa_stamps), (size_t)nwg * 8 * 8 * 8) == hipSuccess ? 0 : -3;
}
#endif
