// fp8 scaled GEMM for gfx950, few rows: the decode step's projections, bound by the weight stream (N x K bytes of HBM).
//
//   out[M,N] = ((sa (.) A[M,K]) . (sb (.) W[N,K]^T)).to(out_t) (+ bias)      K % 128 == 0
//
// A workgroup owns 16 NT output columns and MT blocks of 16 rows -- all of them, or one of several groups of rows where the column
// tiles alone leave CUs idle (stream_rows) --; its waves split K (wave w takes the 128-byte
// K blocks w, w + NW, ...) and every wave runs a pipeline of its own: a wave-private ring in LDS, filled with
// global_load_lds 16 bytes per lane, no barrier until the partial sums are combined at the end of a tile.  What bounded
// the forms before it (us at M 16: 14336 -> 4096 19.1, here 12.7; 4096 -> 28672 28.3, here 21.6; M 1: 15.8 / 28.8, here 11.0 / 20.8 =
// 5.3 / 5.6 TB/s):
//   * a load instruction that fetches 16 rows x 64 bytes (the MFMA operand order, straight into registers) costs the
//     CU's address path as much as one that fetches 8 whole 128-byte lines is worth twice over: 38 against 91 GB/s per
//     CU.  So the loads take whole lines, 8 rows x 128 bytes per instruction, and the operand order comes from LDS;
//   * the 64 x 32 tile kernel staged 64 activation rows whatever M was, behind one barrier per group of K blocks, and
//     left half the CUs idle at N 4096;
//   * every workgroup reads the same activations: workgroups that walk K in the same order hit the same L2 channel at
//     the same time (rows a power of two apart), so each starts at another K block of its list (up to 13 %).
// The weights are read once: non-temporal.  The activations come from L2 through the same address path, which is
// what limits M 32 .. 64 (per K block and workgroup 2 NT line groups of weights, 2 MT of activations):
//   * NT = 2 where 32-column tiles still give enough workgroups (a weight line then shares its activations with
//     another one): 4096 -> 6144 at M 16 7.7 -> 6.8 us; below that many tiles NT = 1;
//   * RESIDENT: where a workgroup has several tiles or K is short, a wave loads the activations of its K blocks once
//     and keeps them in registers (KBW x MT blocks); the ring then carries weights only (against all through the
//     ring: 4096 -> 28672 at M 32 24.3 -> 21.9 us, 8192 -> 28672 47.1 -> 41.7).
// Workgroups are persistent: the next tile's weights are in flight while a tile's partial sums are combined.
//
// LDS image of a block (16 rows x 128 bytes): 16-byte chunks XOR-swizzled by f(row), applied to the per-lane SOURCE
// address (LDS-DMA writes lane-linearly) and to the read address: conflict-free ds_read_b128.  The reads are inline
// asm because hipcc puts s_waitcnt vmcnt(0) -- the whole ring -- in front of LDS loads it sees behind LDS-DMA; every
// asm block waits for its own reads.
#include "common.cuh"

namespace va {
namespace mms {

typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) int i32x4;
typedef __attribute__((ext_vector_type(8))) int i32x8;

struct Params {
  const uint8_t *a, *b;
  const float *sa, *sb;
  const void* bias;
  void* out;
  int M, N, K;
  int64_t lda, ldb, ldc;
  int asn, bsn, ntiles;
  int groups;   // of 16 MT rows
  int vec;   // 8-byte aligned output rows, N % 4 == 0
};

__device__ __forceinline__ int swz(int row) { return ((row >> 1) & 1) | (((row >> 2) & 1) << 2); }
__device__ __forceinline__ i32x8 cat8(i32x4 lo, i32x4 hi) { return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7); }
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p;
}
template <int N> __device__ __forceinline__ void wait_vm() {
  static_assert(N <= 63, "vmcnt has 6 bits");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
template <int OFF> __device__ __forceinline__ void read2(uint32_t p0, uint32_t p1, i32x4& a, i32x4& b) {
  asm volatile("ds_read_b128 %0, %2 offset:%4\n\tds_read_b128 %1, %3 offset:%4\n\ts_waitcnt lgkmcnt(0)"
               : "=&v"(a), "=&v"(b) : "v"(p0), "v"(p1), "n"(OFF) : "memory");
}
template <int OFF> __device__ __forceinline__ void read4(uint32_t p0, uint32_t p1, i32x4& a, i32x4& b, i32x4& c, i32x4& d) {
  asm volatile("ds_read_b128 %0, %4 offset:%6\n\tds_read_b128 %1, %5 offset:%6\n\t"
               "ds_read_b128 %2, %4 offset:%7\n\tds_read_b128 %3, %5 offset:%7\n\ts_waitcnt lgkmcnt(0)"
               : "=&v"(a), "=&v"(b), "=&v"(c), "=&v"(d) : "v"(p0), "v"(p1), "n"(OFF), "n"(OFF + 2048) : "memory");
}
// F consecutive blocks (2 KiB apart) in MFMA operand order
template <int F, int OFF = 0> __device__ __forceinline__ void read_blocks(uint32_t p0, uint32_t p1, i32x8* f) {
  i32x4 a, b, c, d;
  if constexpr (F >= 2) {
    read4<OFF>(p0, p1, a, b, c, d);
    f[0] = cat8(a, b);
    f[1] = cat8(c, d);
    if constexpr (F > 2) read_blocks<F - 2, OFF + 4096>(p0, p1, f + 2);
  } else {
    read2<OFF>(p0, p1, a, b);
    f[0] = cat8(a, b);
  }
}
// one block in whole-line order (rows r8, r8 + 8 of the lane) -> LDS image
template <int OFF> __device__ __forceinline__ void write2(uint32_t p0, uint32_t p1, i32x4 a, i32x4 b) {
  asm volatile("ds_write_b128 %0, %2 offset:%4\n\tds_write_b128 %1, %3 offset:%5"
               ::"v"(p0), "v"(p1), "v"(a), "v"(b), "n"(OFF), "n"(OFF + 1024) : "memory");
}
template <int F, int OFF = 0> __device__ __forceinline__ void write_blocks(uint32_t p0, uint32_t p1, const i32x4* raw) {
  write2<OFF>(p0, p1, raw[0], raw[1]);
  if constexpr (F > 1) write_blocks<F - 1, OFF + 2048>(p0, p1, raw + 2);
}

constexpr int MAXT = 16;   // tiles per workgroup (their column scales sit in LDS)

// KBW = 0: weights and activations both travel through the ring (D stages of NT + MT blocks per wave).  KBW > 0
// (RESIDENT): a wave has at most KBW K blocks and keeps their activations in registers; ring stages of NT blocks.
// GROUPS: p.groups of 16 MT rows, one column tile per workgroup; else M <= 16 MT.
template <typename out_t, int MT, int NT, int NW, int D, int KBW, bool GROUPS>
__global__ __launch_bounds__(64 * NW) void scaled_mm_stream_kernel(const Params p_) {
  Params p = p_;
  int wg = blockIdx.x;
  if constexpr (GROUPS) {
    // Hardware workgroup i runs on XCD i % 8: all groups of a column tile on one XCD, one after the other, so that its weights leave
    // HBM once (with the groups as grid.y, 33 .. 48 rows of N 2192 took as long as two passes over the weights).
    const int idx = wg >> 3, grp = idx % p.groups;
    wg = (wg & 7) + 8 * (idx / p.groups);
    if (wg >= p.ntiles) return;
    const int m0 = grp * 16 * MT;
    p.a += (int64_t)m0 * p.lda;
    p.out = (out_t*)p.out + (int64_t)m0 * p.ldc;
    if (p.asn != 1) p.sa += m0;
    p.M = min(p.M - m0, 16 * MT);
  }
  constexpr bool RES = KBW > 0;
  constexpr int F = RES ? NT : NT + MT;            // blocks per ring stage
  constexpr int STAGE = F * 2048, L = 2 * F;       // bytes, load instructions per stage
  constexpr int RINGB = NW * D * STAGE, REDB = NW * MT * NT * 1024, ASCR = RES ? NW * MT * 2048 : 0;
  constexpr int SBL = (MAXT * 16 * NT + 64 * NW - 1) / (64 * NW);
  // partial sums: two buffers (one barrier per tile) where they fit
  constexpr int SCB = 16 * MT * 4 + SBL * 64 * NW * 4;
  constexpr int NRED = RINGB + SCB + (2 * REDB > ASCR ? 2 * REDB : ASCR) <= 160 * 1024 ? 2 : 1;
  constexpr int POOL = NRED * REDB > ASCR ? NRED * REDB : ASCR;   // (the activations' way into registers ends before the first sum)
  static_assert(RINGB + POOL + SCB <= 160 * 1024, "");
  __shared__ __attribute__((aligned(1024))) uint8_t ring[RINGB];
  __shared__ __attribute__((aligned(1024))) uint8_t pool[POOL];
  __shared__ __attribute__((aligned(16))) float sal[16 * MT], sbl[SBL * 64 * NW];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c16 = lane & 15, g4 = lane >> 4, r8 = lane >> 3;
  const int M = p.M, N = p.N, G = GROUPS ? p.ntiles : (int)gridDim.x;
  const int nkb = p.K / 128;
  const int spt = (nkb - wave + NW - 1) / NW;            // K blocks of this wave (0: it only takes part in the sums)
  const int mytiles = (p.ntiles - wg + G - 1) / G;
  const int T = spt * mytiles;
  // start of this workgroup's walk through the wave's K blocks (workgroups of an XCD: wg >> 3 apart)
  const int rot = spt > 0 ? (wg >> 3) % spt : 0;
  const int ik0 = wave + NW * rot;

  const uint32_t wc0 = ((lane & 7) ^ swz(r8)) << 4, wc1 = ((lane & 7) ^ swz(r8 + 8)) << 4;
  uint32_t aoff[2 * MT];   // activation rows r8 + 8 h (clamped): LDS-DMA carries the swizzle in the source address
#pragma unroll
  for (int h = 0; h < 2 * MT; ++h) {
    const int row = 8 * h + r8;
    aoff[h] = (uint32_t)(row < M ? row : M - 1) * (uint32_t)p.lda + (RES ? (uint32_t)((lane & 7) << 4) : ((h & 1) ? wc1 : wc0));
  }
  uint8_t* const myring = ring + wave * D * STAGE;
  auto issue = [&](int s, int tile, int kb) __attribute__((always_inline)) {
    uint8_t* st = myring + s * STAGE;
    const uint8_t* wb = p.b + (int64_t)kb * 128;
#pragma unroll
    for (int h = 0; h < 2 * NT; ++h) {
      const int n = tile * 16 * NT + 8 * h + r8;
      const uint32_t off = (uint32_t)(n < N ? n : N - 1) * (uint32_t)p.ldb + ((h & 1) ? wc1 : wc0);
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(wb + off),
                                       (__attribute__((address_space(3))) void*)(st + h * 1024), 16, 0, 2);   // nt
    }
    if constexpr (!RES) {
      const uint8_t* ab = p.a + (int64_t)kb * 128;
#pragma unroll
      for (int h = 0; h < 2 * MT; ++h)
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(ab + aoff[h]),
                                         (__attribute__((address_space(3))) void*)(st + NT * 2048 + h * 1024), 16, 0, 0);
    }
  };
  int it = wg, ik = ik0, is = 0, issued = 0, left = spt;
  auto next = [&]() __attribute__((always_inline)) {
    issue(is, it, ik);
    is = is + 1 == D ? 0 : is + 1;
    ik += NW;
    if (ik >= nkb) ik = wave;
    if (--left == 0) { left = spt; ik = ik0; it += G; }
    ++issued;
  };

  // scales: loaded in front of everything else, stored to LDS in the first tile's epilogue
  const float sa0 = p.sa[p.asn == 1 ? 0 : ((int)threadIdx.x < M ? (int)threadIdx.x : M - 1)];
  float sb0[SBL];
#pragma unroll
  for (int i = 0; i < SBL; ++i) {
    const int x = threadIdx.x + i * 64 * NW;       // column x of the workgroup's tiles
    const int n = (wg + (x / (16 * NT)) * G) * 16 * NT + x % (16 * NT);
    sb0[i] = p.sb[p.bsn == 1 ? 0 : (n < N ? n : N - 1)];
  }

  const uint32_t rbase = lds_addr(myring);
  const uint32_t fo0 = c16 * 128 + (((2 * g4) ^ swz(c16)) << 4), fo1 = c16 * 128 + (((2 * g4 + 1) ^ swz(c16)) << 4);
  i32x8 ares[RES ? KBW : 1][MT];
  if constexpr (RES) {
    i32x4 raw[KBW][2 * MT];
#pragma unroll
    for (int k = 0; k < KBW; ++k) {   // (a wave with fewer K blocks loads its first again: no branch, see below)
      const int kr = k < spt ? (k + rot < spt ? k + rot : k + rot - spt) : 0, kb = wave + kr * NW;
      const uint8_t* ab = p.a + (int64_t)(kb < nkb ? kb : nkb - 1) * 128;
#pragma unroll
      for (int h = 0; h < 2 * MT; ++h) raw[k][h] = *reinterpret_cast<const i32x4*>(ab + aoff[h]);
    }
    // unconditional too (T < D: stages that no step reads), so that the compiler can count the loads behind raw[] and
    // does not wait for the whole ring
#pragma unroll
    for (int d = 0; d < D; ++d) {
      it = it < p.ntiles ? it : p.ntiles - 1;
      ik = ik < nkb ? ik : nkb - 1;
      next();
    }
    const uint32_t ab = lds_addr(pool + wave * MT * 2048);
#pragma unroll
    for (int k = 0; k < KBW; ++k) {
      write_blocks<MT>(ab + r8 * 128 + wc0, ab + r8 * 128 + wc1, raw[k]);   // (one wave's LDS operations stay in order)
      read_blocks<MT>(ab + fo0, ab + fo1, ares[k]);
    }
  } else {
#pragma unroll
    for (int d = 0; d < D; ++d)
      if (issued < T) next();
  }

  f32x4 acc[NT][MT];
  int cs = 0, done = 0;
  auto step = [&](int k) __attribute__((always_inline)) {
    // the stage's loads are older than those of the D - 1 stages behind it (a tile's output stores in between only make
    // the wait stricter)
    if (done + D <= T) wait_vm<(D - 1) * L>(); else wait_vm<0>();
    i32x8 f[F];
    read_blocks<F>(rbase + cs * STAGE + fo0, rbase + cs * STAGE + fo1, f);
    if (issued < T) next();   // refills the stage just read
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int j = 0; j < MT; ++j) {
        i32x8 av;
        if constexpr (RES) av = ares[k][j]; else av = f[NT + j];
        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(f[i], av, acc[i][j], 0, 0, 0, 0x7f7f7f7f, 0, 0x7f7f7f7f);
      }
    cs = cs + 1 == D ? 0 : cs + 1;
    ++done;
  };
  for (int t = 0; t < mytiles; ++t) {
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int j = 0; j < MT; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
    if constexpr (RES) {
#pragma unroll
      for (int k = 0; k < KBW; ++k)
        if (k < spt) step(k);
    } else {
      for (int k = 0; k < spt; ++k) step(0);
    }
    // ---- the waves' partial sums -> out.  lane holds C^T[n = 16 i + 4 g4 + r][m = 16 j + c16]
    uint8_t* const red = pool + (t & (NRED - 1)) * REDB;
    if ((RES && t == 0) || NRED == 1) __builtin_amdgcn_s_barrier();   // everyone is past its reads of the pool
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int j = 0; j < MT; ++j)
        *reinterpret_cast<f32x4*>(red + ((wave * MT * NT + j * NT + i) * 64 + lane) * 16) = acc[i][j];
    if (t == 0) {
      if (threadIdx.x < 16 * MT) sal[threadIdx.x] = sa0;
#pragma unroll
      for (int i = 0; i < SBL; ++i) sbl[threadIdx.x + i * 64 * NW] = sb0[i];
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
#pragma unroll
    for (int fr0 = 0; fr0 < MT * NT; fr0 += NW) {
      const int fr = fr0 + wave;
      if (fr >= MT * NT) break;
      const int fm = fr / NT, fn = fr % NT, m = fm * 16 + c16;
      f32x4 v = {0.f, 0.f, 0.f, 0.f};
      const uint32_t rb = lds_addr(red + (fr * 64 + lane) * 16);
      constexpr int WS = MT * NT * 1024;
#pragma unroll
      for (int w = 0; w < NW; w += 2) {
        i32x4 x, y;
        read2<0>(rb + w * WS, rb + (w + 1) * WS, x, y);
        v += __builtin_bit_cast(f32x4, x);
        v += __builtin_bit_cast(f32x4, y);
      }
      i32x4 sx, sy;
      read2<0>(lds_addr(&sbl[(t * NT + fn) * 16 + 4 * g4]), lds_addr(&sal[fm * 16 + (c16 & 12)]), sx, sy);
      const f32x4 sbv = __builtin_bit_cast(f32x4, sx), sa4 = __builtin_bit_cast(f32x4, sy);
      const float s01 = (c16 & 1) ? sa4[1] : sa4[0], s23 = (c16 & 1) ? sa4[3] : sa4[2];
      const float sav = (c16 & 2) ? s23 : s01;
      const int n = ((wg + t * G) * NT + fn) * 16 + 4 * g4;
      if (m < M && n < N) {
        struct alignas(8) V4 { out_t e[4]; } pk;
#pragma unroll
        for (int r = 0; r < 4; ++r) pk.e[r] = from_f32<out_t>((v[r] * sav) * sbv[r]);
        if (p.bias != nullptr) {
          const out_t* bias = (const out_t*)p.bias;
#pragma unroll
          for (int r = 0; r < 4; ++r) pk.e[r] = from_f32<out_t>(to_f32(pk.e[r]) + to_f32(bias[n + r < N ? n + r : N - 1]));
        }
        out_t* op = (out_t*)p.out + (int64_t)m * p.ldc + n;
        if (p.vec) {
          *reinterpret_cast<V4*>(op) = pk;
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (n + r < N) op[r] = pk.e[r];
        }
      }
    }
  }
  if constexpr (RES) wait_vm<0>();   // T < D: loads that no step waited for have landed before the LDS is given back
}

// Row groups: N up to 4096 has at most 256 column tiles of 16, and a workgroup that pulls 128 (16 MT + 16 NT) bytes per K block gets
// 70 GB/s of them while half the CUs are idle, 55 (16 x 16) .. 49 (32 x 32) in a full round.  So the smallest MT + NT with which all rows
// still make one round of workgroups: the weights go to several of them, through L2, and the activations to none twice.  us, all rows in
// one workgroup (M > 64: the tile kernels) -> groups: 8192 -> 1280 at M 32 9.3 -> 7.2, M 63 12.3 -> 9.1, M 94 12.0 -> 9.3; 15360 -> 1248
// at M 40 18.4 -> 11.0, M 81 20.4 -> 14.7; 4096 -> 1024 at M 64 7.7 -> 5.1; 8192 -> 2048 at M 64 12.6 -> 9.5; 4096 -> 4096 at M 63 8.2 ->
// 8.1; of 849 launches with N up to 4096 and M 9 .. 330 the 340 that it takes 0.78 (profiles/gemm_row_groups.txt).  A second round costs
// more than it spreads: 8192 -> 1280 at M 49 as 320 workgroups of 16 rows 10.4, as 160 of 32 8.7; and a round is 32 workgroups on each XCD,
// in whole column tiles: 12672 -> 2624 at M 44 as 82 x 3, 33 on two of them, 17.0 -> 24.7.  32 rows x 32 columns only above M 48 (48 rows x
// 16 in one group there: 0.94 of it).
// 32 columns pull no less than all rows in one workgroup do, only with more of them: up to M 64 that takes K 1280 (16 rows; 1024 -> 2560 at
// M 40 4.2 -> 4.4, 1536 -> 2192 at M 44 4.8 -> 4.6) or 2048 (32 rows; 512 -> 3504 at M 50 3.9 -> 4.2, 1280 -> 3280 at M 56 5.0 -> 5.2,
// 2048 -> 4096 at M 64 6.3 -> 5.7).  The tile kernels above it, which three groups of 32 rows stand against, take four K blocks per barrier
// where K is a multiple of 512, and are ahead up to K 4096 (1536 -> 2560 at M 88 4.8 -> 5.2, 3584 -> 2560 at M 91 7.0 -> 7.6; 1280 -> 2560 at
// M 78 5.0 -> 4.8, 8192 -> 2560 at M 83 12.7 -> 11.4).  Over a long K the activations of a nearly empty last group cost more than it takes
// off the others: 16 rows from K 14336 on want K / 4096 in it (14336 -> 2192 at M 33 16.4 -> 17.6, 15616 -> 2192 at M 34 18.3 -> 18.9, M 36
// 18.1 -> 16.8), two groups of 32 rows 24 where a full round reads most (15360 -> 4096 at M 53 25.2 -> 26.4, M 62 24.8 -> 23.2; 20480 -> 3584 at
// M 49 30.7 -> 33.4; 14336 -> 3888 at M 54 22.7 -> 21.1) and three of them from K 20480 on 20 (20480 -> 2560 at M 75 27.9 -> 30.9, M 80 28.6 ->
// 29.8, M 91 29.9 -> 28.0; 16384 -> 2192 at M 65 22.0 -> 20.6).
// mt = 0: all rows in one workgroup.
struct Rows { int mt, nt; };
static Rows stream_rows(int M, int N, int K) {
  if (M <= 16 || N > 4096) return {0, 0};
  auto wgs = [&](int mt, int nt) { return (int64_t)ceil_div(ceil_div(N, 16 * nt), 8) * 8 * ceil_div(M, 16 * mt); };
  auto last = [&](int mt) { return (M - 1) % (16 * mt) + 1; };   // rows of the last group
  // (32 columns do not pay)
  const bool no12 = (M <= 64 && K < 1280) || (M <= 48 && K >= 14336 && last(1) * 4096 < K);
  const bool no22 = M <= 64 ? K < 2048 || ((int64_t)ceil_div(N, 32) * 2 * K > 3600000 && last(2) < 24)
                           : M <= 96 && wgs(2, 2) > 200 && ((K < 4096 && K % 512 == 0) || (K >= 20480 && last(2) < 20));
  if (wgs(1, 1) <= 256) return {1, 1};
  if (M <= 32) return {0, 0};
  if (wgs(2, 1) <= 256) return {2, 1};
  if (wgs(1, 2) <= 256) return no12 ? Rows{0, 0} : Rows{1, 2};
  if (M <= 48) return {0, 0};
  if (wgs(2, 2) <= 256 && wgs(2, 2) >= wgs(3, 1)) return no22 ? Rows{0, 0} : Rows{2, 2};
  if (wgs(3, 1) <= 256) return {3, 1};
  if (wgs(2, 2) <= 256) return no22 ? Rows{0, 0} : Rows{2, 2};
  return {0, 0};
}

template <typename out_t>
static void launch(const Params& p0, hipStream_t st) {
  Params p = p0;
  const int mt = ceil_div(p.M, 16), t32 = ceil_div(p.N, 32);
#define VA_STREAM(MT, NT, NW, D, KBW, GRID)                                                                   \
  do {                                                                                                        \
    p.ntiles = ceil_div(p.N, 16 * NT);                                                                        \
    int grid = p.ntiles < (GRID) ? p.ntiles : (GRID);                                                         \
    if (grid * MAXT < p.ntiles) grid = ceil_div(p.ntiles, MAXT);                                              \
    hipLaunchKernelGGL((scaled_mm_stream_kernel<out_t, MT, NT, NW, D, KBW, false>), dim3(grid), dim3(64 * NW), 0, st, p); \
  } while (0)
#define VA_STREAM_ROWS(MT, NT, NW, D)                                                                         \
  do {                                                                                                        \
    p.ntiles = ceil_div(p.N, 16 * NT);                                                                        \
    p.groups = ceil_div(p.M, 16 * MT);                                                                        \
    hipLaunchKernelGGL((scaled_mm_stream_kernel<out_t, MT, NT, NW, D, 0, true>), dim3(ceil_div(p.ntiles, 8) * 8 * p.groups), \
                       dim3(64 * NW), 0, st, p);                                                              \
  } while (0)
  const Rows rows = stream_rows(p.M, p.N, p.K);
  if (rows.mt > 0) {
    if (rows.mt == 1 && rows.nt == 1) VA_STREAM_ROWS(1, 1, 4, 3);
    else if (rows.mt == 2 && rows.nt == 1) VA_STREAM_ROWS(2, 1, 4, 2);
    else if (rows.mt == 1) VA_STREAM_ROWS(1, 2, 8, 2);
    else if (rows.mt == 2) VA_STREAM_ROWS(2, 2, 4, 2);
    else VA_STREAM_ROWS(3, 1, 4, 2);
    return;
  }
  // 32-column tiles from 160 of them on (N 5120): fewer, the 16-column ones fill the CUs better (N 4096 at M 16: 5.5 us
  // against 6.6; N 6144: 7.7 against 6.8).
  const bool wide = t32 >= 160, k4 = p.K <= 4 * 8 * 128, k8 = p.K <= 8 * 8 * 128;
  // Activations resident: more than one 32-column tile per CU and few enough K blocks per wave for the registers.
  if (t32 > 256 && mt == 1 && k8) VA_STREAM(1, 2, 8, 3, 8, 256);
  else if (t32 > 256 && mt == 2 && k4) VA_STREAM(2, 2, 8, 3, 4, 256);
  else if (t32 > 256 && mt == 2 && k8) VA_STREAM(2, 2, 8, 3, 8, 256);
  else if (t32 > 256 && mt == 3 && k4) VA_STREAM(3, 2, 8, 2, 4, 256);
  else if (t32 > 256 && mt == 4 && k4) VA_STREAM(4, 2, 8, 2, 4, 256);
  // (one workgroup of 8 waves per CU at M <= 16; the narrower rings of 4 waves let two share a CU)
  else if (wide && mt == 1) VA_STREAM(1, 2, 8, 2, 0, 256);
  else if (wide && mt == 2) VA_STREAM(2, 2, 4, 2, 0, 512);
  else if (wide && mt == 3) VA_STREAM(3, 2, 4, 2, 0, 256);
  else if (wide) VA_STREAM(4, 2, 4, 2, 0, 256);
  else if (mt == 1) VA_STREAM(1, 1, 4, 3, 0, 1024);
  else if (mt == 2) VA_STREAM(2, 1, 4, 2, 0, 1024);
  else if (mt == 3) VA_STREAM(3, 1, 4, 2, 0, 512);
  else VA_STREAM(4, 1, 4, 2, 0, 512);
#undef VA_STREAM_ROWS
#undef VA_STREAM
}

}  // namespace mms

// Whether launch_scaled_mm_stream is the better kernel (against the tile kernels, weights from HBM; us, tiles -> stream; all
// shapes: profiles/gemm_stream.txt).  M <= 32: up to 256 32-column tiles everywhere (0.98 .. 1.9 x).  With more, keeping the
// activations costs a workgroup a start of 4 .. 5 us that K has to earn back: M 17, 1024 -> 14336 6.0 -> 9.1, 2048 -> 10240
// 8.1 -> 9.3, 3072 -> 10240 10.7 -> 10.4, 4096 -> 28672 27.9 -> 21.0.
// M > 32: a 32-column tile's stage is 3 .. 4 blocks of activations to 2 of weights, and the tile kernels, which share them
// between more columns, win unless N is small (8192 -> 4096 at M 64 16.6 -> 13.5), a workgroup can keep them (4096 -> 28672
// 29.7 -> 25.9; but 64 x 64 tiles that just make one round need K 4096: 3584 -> 14336 at M 49 13.0 -> 14.4, 4096 -> 14336
// 15.5 -> 15.2) or M <= 48 leaves room (4096 -> 6144 8.7 -> 8.4, from K 3072 on: 2048 -> 8192 at M 48 6.3 -> 6.7); they keep
// 4096 -> 6144 (10.4 : 10.3) and 3584 -> 8192 (9.8 : 10.1) at M 64, and more than 256 tiles over K above 4096 (8192 -> 14336 at
// M 49, 64 27.9, 28.9 : 28.2, 30.9; not at M 33, 27.6 : 25.2).
bool scaled_mm_stream_pays(int M, int N, int K) {
  if (M > 64) return K >= 1024 && mms::stream_rows(M, N, K).mt > 0;
  const int t32 = ceil_div(N, 32), t64 = ceil_div(N, 64);
  if (t32 > 256 && (K < 3072 || (M > 32 && K < 4096 && t64 >= 190 && t64 <= 256))) return false;
  if (M <= 32 || t32 < 160) return true;
  return K <= 4096 ? K >= 3072 && (M <= 48 || t32 > 256) : t32 <= 256;
}

// 16 x rows and columns of a workgroup where the rows go in groups, 10 mt + nt; 0 where a workgroup takes all of them.
int scaled_mm_stream_groups(int M, int N, int K) {
  const mms::Rows r = mms::stream_rows(M, N, K);
  return 10 * r.mt + r.nt;
}

// The groups of rows are so small that nothing the tile kernels have for these shapes comes near, K slices included.
bool scaled_mm_stream_small(int M, int N, int K) {
  const mms::Rows r = mms::stream_rows(M, N, K);
  return r.mt > 0 && r.mt + r.nt <= 3;
}

// Caller guarantees M >= 1, above 64 scaled_mm_stream_pays(), K % 128 == 0, 16-byte aligned operands and scaled_mm_large_fits() (32-bit offsets).
int launch_scaled_mm_stream(void* out, const void* a, const void* b, const float* a_scales, const float* b_scales,
                            const void* bias, int M, int N, int K, int64_t lda, int64_t ldb, int64_t ldc, int asn, int bsn,
                            int out_dtype, hipStream_t st) {
  const int vec = ldc % 4 == 0 && N % 4 == 0 && (((uintptr_t)out) & 7) == 0;
  const mms::Params p{(const uint8_t*)a, (const uint8_t*)b, a_scales, b_scales, bias, out, M, N, K, lda, ldb, ldc, asn, bsn, 0, 1, vec};
  if (out_dtype == VLLM_AMD_BF16) mms::launch<bf16_t>(p, st);
  else mms::launch<f16_t>(p, st);
  return VLLM_AMD_OK;
}

}  // namespace va
