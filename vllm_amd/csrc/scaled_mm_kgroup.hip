// fp8 scaled GEMM for gfx950, the mid-M range (a single round of 128 x 128 tiles): two K groups and loader waves.
//
//   out[M,N] = ((sa (.) A[M,K]) . (sb (.) W[N,K]^T)).to(out_t) (+ bias)      K % 128 == 0
//
// What bounded the tile kernel before it (scaled_mm_large.hip, 128 x 128, two K blocks per barrier): all eight waves issued
// their share of the LDS-DMA behind the barrier (a CU takes one 1 KiB load per ~16 cycles: 32 loads = 512 cycles per K block
// in which the issuing waves stand still), then all read fragments, then all multiplied: ~1280 cycles per K block for 512
// cycles of MFMA.  Here the three kinds of work belong to different waves of a SIMD and run at the same time:
//   * waves 0-3 and 4-7 are two K groups, each owning the whole tile as 2 x 2 waves of 64 x 64 outputs: group g takes the
//     K blocks g, g + 2, ..  In an interval (barrier to barrier) one group reads the fragments of a block -- 16 KiB per wave, a
//     third less LDS traffic per MFMA than 64 x 32 wave tiles -- while the other multiplies the block before: 16 MFMAs back
//     to back, nothing else;
//   * waves 8-11, one per SIMD, issue all loads (8 per interval each) and are the only ones that wait for them.  The ring
//     holds five K blocks (160 KiB: the whole LDS); three are in flight.
// The groups' sums meet at the end through LDS.  Per interval: MFMA 586, fragment reads 513, load issue 560 cycles, ~800 with
// the barrier's skew (stamps at 509 x 8192 -> 7168).  us, weights from HBM: 509 x 8192 -> 7168 49.5 -> 39.4, 509 x 3584 -> 8192
// 25.3 -> 22.1, 1024 x 14336 -> 4096 80.8 -> 66.8, 256 x 8192 -> 10240 54.0 -> 41.2.
//
// LDS image of a K block: [rows][128 B], 16-byte chunks XOR-swizzled by f(row), applied to the per-lane SOURCE address (LDS-DMA
// writes lane-linearly) and to the read address.  The reads are inline asm because hipcc puts s_waitcnt vmcnt(0) in front of
// LDS loads it sees behind LDS-DMA; the asm block waits for its own reads.
#include "common.cuh"

namespace va {
namespace mmk {

typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) int i32x4;
typedef __attribute__((ext_vector_type(8))) int i32x8;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;

struct Params {
  const uint8_t *a, *b;
  const float *sa, *sb;
  const void* bias;
  void* out;
  int M, N, K;
  int64_t lda, ldb, ldc;
  int asn, bsn;
};

constexpr int BM = 128, BN = 128, LBK = 128;

__device__ __forceinline__ int swz(int row) { return ((row >> 1) & 1) | (((row >> 2) & 1) << 2); }
__device__ __forceinline__ i32x8 cat8(i32x4 lo, i32x4 hi) { return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7); }
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p;
}
template <int N> __device__ __forceinline__ void wait_vm() {
  static_assert(N <= 63, "vmcnt has 6 bits");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// the fragments of a wave's 64 activation rows and 64 weight rows: 16 rows are 2 KiB apart
__device__ __forceinline__ void read_frags(uint32_t a0, uint32_t a1, uint32_t w0, uint32_t w1, i32x8 (&af)[4], i32x8 (&wf)[4]) {
  i32x4 x[16];
  asm volatile("ds_read_b128 %0, %18\n\tds_read_b128 %1, %19\n\t"
               "ds_read_b128 %2, %18 offset:2048\n\tds_read_b128 %3, %19 offset:2048\n\t"
               "ds_read_b128 %4, %18 offset:4096\n\tds_read_b128 %5, %19 offset:4096\n\t"
               "ds_read_b128 %6, %18 offset:6144\n\tds_read_b128 %7, %19 offset:6144\n\t"
               "ds_read_b128 %8, %16\n\tds_read_b128 %9, %17\n\t"
               "ds_read_b128 %10, %16 offset:2048\n\tds_read_b128 %11, %17 offset:2048\n\t"
               "ds_read_b128 %12, %16 offset:4096\n\tds_read_b128 %13, %17 offset:4096\n\t"
               "ds_read_b128 %14, %16 offset:6144\n\tds_read_b128 %15, %17 offset:6144\n\t"
               "s_waitcnt lgkmcnt(0)"
               : "=&v"(x[0]), "=&v"(x[1]), "=&v"(x[2]), "=&v"(x[3]), "=&v"(x[4]), "=&v"(x[5]), "=&v"(x[6]), "=&v"(x[7]),
                 "=&v"(x[8]), "=&v"(x[9]), "=&v"(x[10]), "=&v"(x[11]), "=&v"(x[12]), "=&v"(x[13]), "=&v"(x[14]), "=&v"(x[15])
               : "v"(a0), "v"(a1), "v"(w0), "v"(w1)
               : "memory");
#pragma unroll
  for (int i = 0; i < 4; ++i) { wf[i] = cat8(x[2 * i], x[2 * i + 1]); af[i] = cat8(x[8 + 2 * i], x[9 + 2 * i]); }
}

template <typename out_t>
__global__ __launch_bounds__(768) void scaled_mm_kgroup_kernel(const Params p) {
  constexpr int R = 5;                                     // ring slots (K blocks)
  constexpr int A_BYTES = BM * LBK, STAGE = (BM + BN) * LBK;
  constexpr int L = (BM + BN) / 32, AL = BM / 32;          // load instructions per loader wave and K block, of which activations
  constexpr int MT = 4, NT = BN / 32;                      // MFMA tiles per wave
  static_assert(R * STAGE <= 160 * 1024 && (R - 2) * L <= 63, "");
  __shared__ __attribute__((aligned(1024))) uint8_t lds[R * STAGE];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = wave >> 2, wm = (wave >> 1) & 1, wn = wave & 1;   // (waves 0 .. 7)
  const int c16 = lane & 15, g4 = lane >> 4;
  const int M = p.M, N = p.N, nb = p.K / LBK;

  const int tiles_m = (M + BM - 1) / BM;
  int wg = blockIdx.x;
  {
    // hardware workgroup i runs on XCD i % 8: every XCD gets a contiguous run of tiles (m fastest), so that the tiles
    // that share a weight panel share an L2
    const int q = gridDim.x / 8, r = gridDim.x % 8, xcd = wg % 8, idx = wg / 8;
    wg = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + idx;
  }
  const int m0 = (wg % tiles_m) * BM, n0 = (wg / tiles_m) * BN;

  // LDS of the epilogue, over the ring: exchanged sums, the output tile, scales and bias
  constexpr int XB = NT * 2 * 1024;    // exchange bytes per wave
  constexpr int ROWB = 2 * BN, CPR = BN / 8, RPI = 64 / CPR;
  uint8_t* const tile = lds + 8 * XB;  // [BM rows][2 BN bytes], 16-byte chunks XOR-swizzled by the row
  float* const sal = reinterpret_cast<float*>(lds + 8 * XB + BM * ROWB);   // [BM] row scales, [BN] column scales, [BN] bias
  float *const sbl = sal + BM, *const bil = sbl + BN;
  static_assert(8 * XB + BM * ROWB + 4 * (BM + 2 * BN) <= R * STAGE, "");

  if (wave >= 8) {
    // ---- loader waves: round i, wave w: rows [32 i + 8 (w - 8), +8), lane -> (row lane >> 3, 16-byte chunk (lane & 7) ^ swz(row)).
    // Rows past the edge: any valid row (their outputs are never stored).
    __builtin_amdgcn_s_setprio(2);      // (the loads are the longest chain)
    const int t = tid - 512;
    const float sa_t = p.sa[p.asn == 1 ? 0 : min(m0 + (t & (BM - 1)), M - 1)];
    const float sb_t = p.sb[p.bsn == 1 ? 0 : min(n0 + (t & (BN - 1)), N - 1)];
    const float bi_t = p.bias != nullptr ? to_f32(((const out_t*)p.bias)[min(n0 + (t & (BN - 1)), N - 1)]) : 0.f;
    uint32_t off[L];
#pragma unroll
    for (int i = 0; i < L; ++i) {
      const int row = 32 * (i < AL ? i : i - AL) + 8 * (wave - 8) + (lane >> 3);
      const uint32_t ch = (uint32_t)(((lane & 7) ^ swz(row)) << 4);
      off[i] = i < AL ? (uint32_t)min(m0 + row, M - 1) * (uint32_t)p.lda + ch : (uint32_t)min(n0 + row, N - 1) * (uint32_t)p.ldb + ch;
    }
    auto issue = [&](int slot, int kb) __attribute__((always_inline)) {
      uint8_t* base = lds + slot * STAGE + 8 * (wave - 8) * LBK;
      const uint8_t *ag = p.a + (int64_t)kb * LBK, *bg = p.b + (int64_t)kb * LBK;
#pragma unroll
      for (int i = 0; i < L; ++i)
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)((i < AL ? ag : bg) + off[i]),
                                         (__attribute__((address_space(3))) void*)(base + 32 * i * LBK), 16, 0, 0);
    };
#pragma unroll
    for (int i = 0; i < R - 1; ++i)
      if (i < nb) issue(i, i);
    // Interval b: K block b has landed, the slot of block b - 1, read in the interval before, is refilled.  Blocks
    // b + 1 .. b + R - 2 stay in flight.
    int prev = R - 1, b = 0;
    for (; b < nb - (R - 1); ++b) {
      wait_vm<(R - 2) * L>();
      __builtin_amdgcn_s_barrier();
      issue(prev, b + R - 1);
      prev = prev + 1 == R ? 0 : prev + 1;
    }
    for (; b < nb; ++b) {               // nothing left to issue: nb - 1 - b K blocks behind b
      const int later = nb - 1 - b;
      if (later == 3) wait_vm<3 * L>();
      else if (later == 2) wait_vm<2 * L>();
      else if (later == 1) wait_vm<L>();
      else wait_vm<0>();
      __builtin_amdgcn_s_barrier();
    }
    __builtin_amdgcn_s_barrier();       // nb + 1 intervals
    if (t < BM) sal[t] = sa_t;
    if (t < BN) { sbl[t] = sb_t; bil[t] = bi_t; }
    __syncthreads();                    // the two of the epilogue
    __syncthreads();
    return;
  }

  const uint32_t ch0 = ((2 * g4) ^ swz(c16)) << 4, ch1 = ((2 * g4 + 1) ^ swz(c16)) << 4;
  const uint32_t a_rd = lds_addr(lds) + (64 * wm + c16) * LBK, w_rd = lds_addr(lds) + A_BYTES + ((BN / 2) * wn + c16) * LBK;

  f32x4 acc[NT][MT];
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};

  // group g takes the K blocks g, g + 2, ..: fragments read in the interval of the block, multiplied in the next one
  int cur = 0;
  auto sync = [&]() __attribute__((always_inline)) {
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  if (grp == 1) {
    sync();
    cur = 1;
  }
  const int mine = (nb - grp + 1) / 2;
  for (int k = 0; k < mine; ++k) {
    sync();
    i32x8 af[MT], wf[NT];
    const uint32_t so = cur * STAGE;
    read_frags(a_rd + so + ch0, a_rd + so + ch1, w_rd + so + ch0, w_rd + so + ch1, af, wf);
    cur = cur + 2 >= R ? cur + 2 - R : cur + 2;
    sync();
#pragma unroll
    for (int j = 0; j < MT; ++j)
#pragma unroll
      for (int i = 0; i < NT; ++i)
        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wf[i], af[j], acc[i][j], 0, 0, 0, 0x7f7f7f7f, 0, 0x7f7f7f7f);
    __builtin_amdgcn_sched_barrier(0);
  }
  if (((nb ^ grp) & 1) == 0) sync();   // nb + 1 intervals for either group

  // ---- epilogue: lane holds C^T[n = 16 i + 4 g4 + r][m = 16 j + c16].  Each group finishes half of the wave tile's rows:
  // group 0 gives its sums of j = 2, 3 away and takes group 1's of j = 0, 1.  (The group is a constant inside: a selected
  // index would put the accumulators into scratch memory.)
  auto combine = [&](auto gc) __attribute__((always_inline)) {
    constexpr int G = decltype(gc)::value;
    const int q = 2 * wm + wn;         // position of the wave tile
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        *reinterpret_cast<f32x4*>(lds + (G * 4 + q) * XB + ((i * 2 + j) * 64 + lane) * 16) = acc[i][2 * (1 - G) + j];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int row = 64 * wm + 16 * (2 * G + j) + c16;
      const float sav = sal[row];
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        const f32x4 other = *reinterpret_cast<const f32x4*>(lds + ((1 - G) * 4 + q) * XB + ((i * 2 + j) * 64 + lane) * 16);
        const int col = (BN / 2) * wn + 16 * i + 4 * g4;
        const f32x4 sbv = *reinterpret_cast<const f32x4*>(sbl + col), biv = *reinterpret_cast<const f32x4*>(bil + col);
        const f32x4 v = acc[i][2 * G + j] + other;
        struct alignas(8) V4 { out_t e[4]; } pk;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          pk.e[r] = from_f32<out_t>((v[r] * sav) * sbv[r]);
          if (p.bias != nullptr) pk.e[r] = from_f32<out_t>(to_f32(pk.e[r]) + biv[r]);
        }
        const int c8 = (BN / 8) * wn + 4 * i + g4;   // 8-byte chunk within the row
        *reinterpret_cast<V4*>(tile + row * ROWB + ((c8 ^ (2 * (row & 7))) << 3)) = pk;
      }
    }
    __syncthreads();
  };
  if (grp == 0) combine(std::integral_constant<int, 0>{});
  else combine(std::integral_constant<int, 1>{});
  out_t* const out = (out_t*)p.out;
#pragma unroll
  for (int i = 0; i < BM / (RPI * 8); ++i) {
    const int row = RPI * (wave * (BM / (RPI * 8)) + i) + lane / CPR, ch = lane % CPR;
    const u32x4 v = *reinterpret_cast<const u32x4*>(tile + row * ROWB + ((ch ^ (row & 7)) << 4));
    if (m0 + row < M && n0 + 8 * ch < N) *reinterpret_cast<u32x4*>(out + (int64_t)(m0 + row) * p.ldc + n0 + 8 * ch) = v;
  }
}

}  // namespace mmk

// Single rounds of 128 x 128 tiles, 160 .. 256 of them.  Against the kernels of scaled_mm_large.hip that served these shapes
// (the same tile with both waves of a SIMD in step, from 190 tiles on; 128 x 64 tiles below), weights from HBM, 145 shapes of
// K 1024 .. 14336, N 1280 .. 28672, M 72 .. 3200 with that many tiles (profiles/gemm_kgroup.txt): 0.99 .. 1.10 x at K 1024,
// 1.02 .. 1.24 at 2048, 1.02 .. 1.33 at 4096, 1.05 .. 1.37 at 8192, 1.05 .. 1.44 at 14336.  Below 160 tiles the smaller tiles fill more CUs (144 tiles: 0.96 .. 1.24 x, 128: 0.71 .. 0.77), above 256
// two workgroups of the smaller rings share a CU (320 and 448 tiles: 0.81 .. 1.03).
bool scaled_mm_kgroup_pays(int M, int N, int K) {
  const int64_t tiles = (int64_t)ceil_div(M, mmk::BM) * ceil_div(N, mmk::BN);
  return M > 64 && tiles >= 160 && tiles <= 256;
}

// Caller guarantees K % 128 == 0, K >= 256, 16-byte aligned operands, scaled_mm_large_fits() (32-bit offsets) and 16-byte
// aligned output rows (ldc % 8 == 0, N % 8 == 0, out 16-byte aligned).
int launch_scaled_mm_kgroup(void* out, const void* a, const void* b, const float* a_scales, const float* b_scales,
                            const void* bias, int M, int N, int K, int64_t lda, int64_t ldb, int64_t ldc, int asn, int bsn,
                            int out_dtype, hipStream_t st) {
  const mmk::Params p{(const uint8_t*)a, (const uint8_t*)b, a_scales, b_scales, bias, out, M, N, K, lda, ldb, ldc, asn, bsn};
  const dim3 grid(ceil_div(M, mmk::BM) * ceil_div(N, mmk::BN));
  if (out_dtype == VLLM_AMD_BF16) hipLaunchKernelGGL((mmk::scaled_mm_kgroup_kernel<bf16_t>), grid, dim3(768), 0, st, p);
  else hipLaunchKernelGGL((mmk::scaled_mm_kgroup_kernel<f16_t>), grid, dim3(768), 0, st, p);
  return VLLM_AMD_OK;
}

}  // namespace va
