// Launches of the 256-row tile kernel (prefill_fa_tile.cuh), of a mixed step's chunks and decodes, and the merge of key segments.
#include "prefill_fa_tile.cuh"
#include "unified_decode_kernel.cuh"

#include <atomic>

namespace va {
namespace fa {

// A mixed step in one launch: the row blocks of the chunks first, behind them an eight-wave workgroup for every decode (sequence,
// kv head) pair, longest first.  Row blocks of a chunk differ in length and so do the chunks: a launch of their own ended on a
// few of them with most CUs idle (2000 tokens over 1500: 256 blocks of 24 .. 55 tiles), and the decode kernel, which waits for
// bytes and not for the matrix cores, stood in front of it.  us, two launches -> one (32 / 8 heads, fp8, cache write included),
// 2000 over 1500 among 63 decodes of up to 4096 keys 158 -> 144, of up to 1000 131 -> 114; 2 x 1000 fresh among 15 of 4000
// 70.6 -> 43.7; 6000 fresh among 63 of 4000 371 -> 354.
// (Tried, where the first of these took 148: two groups of four waves per workgroup 152; several kv heads per workgroup one after the
// other, 160.)
template <typename T, bool FP8>
__global__ __launch_bounds__(512) void fa_mixed_kernel(const FaParams p, const UniDecodeParams u, int gx, int gy, int nfa, int npairs, int first, int early, int sub_shift, int order) {
  constexpr int DL = ua_decode_lds<FP8, 128, 8>(), LDS = DL > fa_lds<128>() ? DL : fa_lds<128>();
  __shared__ __attribute__((aligned(1024))) uint8_t lds[LDS];
  // the decodes `pair` < early come behind the first `first` row blocks, the others behind all of them
  int id = blockIdx.x, pair = -1;
  if (id >= first) {
    if (id < first + early) pair = id - first;
    else id -= early;
  }
  if (pair < 0 && id >= nfa) pair = id - nfa + early;
  if (pair < 0) {
    if (id < gx * gy) fa_body<T, FP8, false, 128, 8, false, false, true>(p, lds, id, gy);
  } else {
    ua_decode_body<T, FP8, 128, 8, false, true>(u, (char*)lds, sub_shift, 0, order, pair, npairs, 0);
  }
}

// The last i of [0, n) for which le(i) holds (it holds for all i up to that one; 0 if it holds for none): 64 candidates per
// step, so that 64 sequences take one load and 4096 two, where a binary search chains 6 and 12.
template <typename F>
__device__ __forceinline__ int wave_last(int n, int lane, F&& le) {
  int lo = 0;
  while (n > 1) {
    const int step = (n + 63) >> 6, i = lane * step;
    const int m = (int)__popcll(__ballot(i < n && le(lo + (i < n ? i : 0))));   // (popcll is unsigned)
    const int c = m > 0 ? m - 1 : 0;
    lo += c * step;
    n = min(step, n - c * step);
  }
  return __builtin_amdgcn_readfirstlane(lo);
}

// Merge of a split launch: one wave per (token, q head).  Lane s holds segment s's maximum and sum; a half wave (D <= 128;
// the whole wave above) reads one partial row per step, four rows in flight.  Segments that saw nothing (maximum -inf) are
// not read.
template <typename T, int D>
__global__ __launch_bounds__(256) void fa_reduce_kernel(const FaParams p) {
  constexpr int LPR = D / 4, PAR = 64 / LPR;      // lanes per row, rows per step
  const int lane = threadIdx.x & 63;
  const int pair = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tok = pair / p.num_heads, head = pair % p.num_heads;
  if (tok >= p.num_tokens) return;
  const int nseg = p.num_segments, dr = p.head_size;
  const int64_t row = ((int64_t)tok * p.num_heads + head) * nseg;
  // (in front of the checks, not behind their loads; rows that nobody wrote are not used)
  float ms = lane < nseg ? p.segm_max[row + lane] : -INFINITY;
  float ls = lane < nseg ? p.segm_sum[row + lane] : 0.f;
  if (tok < p.cu_seqlens_q[0] || tok >= p.cu_seqlens_q[p.num_seqs]) return;
  int live = -1;
  if (p.skip_decode) {
    const int lo = wave_last(p.num_seqs, lane, [&](int i) { return p.cu_seqlens_q[i] <= tok; });
    if (p.cu_seqlens_q[lo + 1] - p.cu_seqlens_q[lo] == 1) {           // the decode kernel's token
      if (p.decode_segments <= 1) return;
      const int tiles = (p.seq_lens[lo] + 63) >> 6, per = (tiles + p.decode_segments - 1) / p.decode_segments;
      live = per > 0 ? (tiles + per - 1) / per : 0;
    }
  }
  if (live < 0) {
    const float last = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, ls), nseg - 1));
    live = last < 0.f ? (int)-last : nseg;
    if (live == 1) return;             // the only segment has written the output
  }
  if (lane >= live) { ms = -INFINITY; ls = 0.f; }
  const float mx = wave_max(ms);
  const float w = ms == -INFINITY ? 0.f : fast_exp2(ms - mx);
  const float l = wave_sum(ls * w);
  const int d = 4 * (lane % LPR), sub = lane / LPR;
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
  const float* base = p.segm_out + row * dr + (d < dr ? d : 0);
  for (int s0 = 0; s0 < live; s0 += 4 * PAR) {
    float4 part[4];
    float ws[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int s = s0 + u * PAR + sub;
      ws[u] = __shfl(w, s < live ? s : 0, 64);
      if (s >= live) ws[u] = 0.f;
      part[u] = ws[u] > 0.f ? *reinterpret_cast<const float4*>(base + (int64_t)s * dr) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      acc.x = fmaf(part[u].x, ws[u], acc.x);
      acc.y = fmaf(part[u].y, ws[u], acc.y);
      acc.z = fmaf(part[u].z, ws[u], acc.z);
      acc.w = fmaf(part[u].w, ws[u], acc.w);
    }
  }
  if constexpr (PAR == 2) {
    acc.x = sum_xor32(acc.x);
    acc.y = sum_xor32(acc.y);
    acc.z = sum_xor32(acc.z);
    acc.w = sum_xor32(acc.w);
  }
  if (sub != 0 || d >= dr) return;
  // (a row of NaN scores never raises its maximum from -inf: weight 0, but its sum is NaN, and so is the row, as unsplit)
  const float inv = l == 0.f ? 0.f : 1.0f / l;
  const int64_t oi = (int64_t)tok * p.o_stride_t + (int64_t)head * p.o_stride_h + d;
  if (p.out_scale == nullptr) {
    *reinterpret_cast<u32x2*>((T*)p.o + oi) = (u32x2){Mma<T>::pack2(acc.x * inv, acc.y * inv), Mma<T>::pack2(acc.z * inv, acc.w * inv)};
  } else {
    const float oinv = inv / *p.out_scale;
    auto cl = [](float y) { return fmaxf(-448.0f, fminf(y, 448.0f)); };
    *reinterpret_cast<uint32_t*>((uint8_t*)p.o + oi) = f32x4_to_fp8x4(cl(acc.x * oinv), cl(acc.y * oinv), cl(acc.z * oinv), cl(acc.w * oinv));
  }
}

}  // namespace fa

int g_pf_fa_stagger = 1;   // tuning "pf_fa_stagger": 0 = all eight waves stage at the bottom of the interval
std::atomic<int> g_pf_mixed_launches{0};   // get_tuning "pf_mixed_launches"
std::atomic<int> g_pf_cut_launches{0};     // get_tuning "pf_cut_launches": merges that took cut decodes along
int launch_unified_fa(const FaParams& given, int dtype, bool fp8, hipStream_t st, const UniDecodeParams* u) {
  FaParams p = given;
  const bool wide = p.head_size > 128;                 // 128-row workgroups of four waves
  const int tpb = p.tpb = (wide ? 128 : 256) / p.pack;
  const unsigned gx = p.blocks_per_seq > 0 ? (unsigned)(p.blocks_per_seq * p.num_seqs) : (unsigned)(p.num_tokens / tpb + p.num_seqs);
  const unsigned gy = (unsigned)(p.pack > 1 ? p.num_kv_heads : p.num_heads);
  const unsigned slots = p.num_segments > 1 ? (unsigned)p.seg_slots : 0u;
  p.halves = 128 % p.pack == 0;
  p.shares = fa_shares((int)gy, p.window, p.max_k);
  const unsigned per = p.shares ? p.shares : 1;   // (fa_find)
  const dim3 grid(((gx > slots ? gx : slots) + per - 1) / per * per, gy);
  int npairs = 0, sub_shift = 0, order = 0;
  if (u != nullptr) {
    npairs = unified_decode_pairs(*u);
    while ((16 << sub_shift) < u->block_size) ++sub_shift;
    if (pa_order_enabled() && u->num_seqs <= kLptMaxSeqs)   // longest first (unified_decode)
      for (order = 1; order < 30 && u->max_seq_len > 0 && (u->max_seq_len >> order) != 0;) ++order;
  }
  const unsigned nfa = (grid.x * grid.y + 7) / 8 * 8;   // (the ids behind them go round-robin over the XCDs too)
  // Fewer than 16 sequences have keys of at least twice the longest chunk's tokens here.  They may be a decode's: those do not come behind all
  // row blocks but behind the 24 of every XCD that start first (us, 32 / 8 heads, 2 x 1500 over 500 among 5 of 8000 99 -> 78, 3 x 1200 among one
  // of 16000 127 -> 98, 2 x 4000 among 10 of 10000 252 -> 233; 16-bit 126 -> 88, 181 -> 155, 291 -> 238).  They may as well be a chunk's own
  // context, and then the workgroups that find no decode keep a few row blocks waiting: 0.2 % on average, up to 2 us (64 / 8, 14 x 62 .. 130 over
  // 256 .. 678 54.0 -> 56.5); behind all row blocks that was no less.  With more sequences the longest may be a chunk's context, and what
  // starts late a row block: 64 / 8, 3 x 540 over 4000 among 40 of 2566 183 -> 200.
  const int first = nfa < 8 * 24 ? (int)nfa : 8 * 24, early = p.num_seqs < 16 ? npairs / 8 * 8 : 0;
#define FA_MIXED(T_, F_)                                                                                                  \
  hipLaunchKernelGGL((fa::fa_mixed_kernel<T_, F_>), dim3(nfa + (unsigned)npairs), dim3(512), 0, st, p, *u, (int)grid.x, \
                     (int)grid.y, (int)nfa, npairs, first, early, sub_shift, order)
#define FA_LAUNCH___(T_, F_, P_, D_, NW_, S_)                                                                            \
  do {                                                                                                                   \
    if (p.num_segments > 1) hipLaunchKernelGGL((fa::fa_fwd_kernel<T_, F_, P_, D_, NW_, S_, true>), grid, dim3(64 * NW_), 0, st, p); \
    else hipLaunchKernelGGL((fa::fa_fwd_kernel<T_, F_, P_, D_, NW_, S_, false>), grid, dim3(64 * NW_), 0, st, p);         \
  } while (0)
#define FA_LAUNCH__(T_, F_, P_, D_, NW_)                                                           \
  do {                                                                                             \
    if (!P_ && p.softcap > 0.f) FA_LAUNCH___(T_, F_, false, D_, NW_, true);                        \
    else FA_LAUNCH___(T_, F_, P_, D_, NW_, false);                                                 \
  } while (0)
#define FA_LAUNCH_(T_, F_, P_) FA_LAUNCH__(T_, F_, P_, 128, 8)
#define FA_LAUNCH(T_, F_)                                                   \
  do {                                                                      \
    if (p.prefix) FA_LAUNCH_(T_, F_, true); else FA_LAUNCH_(T_, F_, false); \
  } while (0)
  if (u != nullptr) {
    g_pf_mixed_launches.fetch_add(1, std::memory_order_relaxed);
    if (dtype == VLLM_AMD_BF16) { if (fp8) FA_MIXED(bf16_t, true); else FA_MIXED(bf16_t, false); }
    else { if (fp8) FA_MIXED(f16_t, true); else FA_MIXED(f16_t, false); }
  }
  else if (wide) launch_fa_wide(p, dtype, fp8, grid, st);
  else if (dtype == VLLM_AMD_BF16) { if (fp8) FA_LAUNCH(bf16_t, true); else FA_LAUNCH(bf16_t, false); }
  else { if (fp8) FA_LAUNCH(f16_t, true); else FA_LAUNCH(f16_t, false); }
  if (p.num_segments > 1) {
    if (p.decode_segments > 1) g_pf_cut_launches.fetch_add(1, std::memory_order_relaxed);
    const dim3 rgrid((unsigned)(((int64_t)p.num_tokens * p.num_heads + 3) / 4));
#define FA_REDUCE(T_)                                                                          \
  do {                                                                                         \
    if (wide) hipLaunchKernelGGL((fa::fa_reduce_kernel<T_, 256>), rgrid, dim3(256), 0, st, p); \
    else hipLaunchKernelGGL((fa::fa_reduce_kernel<T_, 128>), rgrid, dim3(256), 0, st, p);      \
  } while (0)
    if (dtype == VLLM_AMD_BF16) FA_REDUCE(bf16_t); else FA_REDUCE(f16_t);
#undef FA_REDUCE
  }
#undef FA_MIXED
#undef FA_LAUNCH
#undef FA_LAUNCH_
#undef FA_LAUNCH__
#undef FA_LAUNCH___
  return VLLM_AMD_OK;
}

}  // namespace va

// The order of a launch's row blocks: no device, no launch.
extern "C" int vllm_amd_prefill_order(int head_size, int group, int num_kv_heads, int num_seqs, int row_blocks, int chunks, int over, int cached,
                                      int decodes, int window, int max_seq_len) {
  if (group < 1 || num_kv_heads < 1) return 0;
  const int bm = head_size > 128 ? 128 : 256, pack = group > 1 && group <= 16 ? group : 1, gy = pack > 1 ? num_kv_heads : num_kv_heads * group;
  const bool most = 2 * over >= chunks, halves = 128 % pack == 0, pairs = va::fa_pairs(bm, halves, gy, row_blocks, decodes, window);
  const bool few = va::fa_few(va::fa_shares(gy, window, max_seq_len), gy, row_blocks, chunks, pairs, most, window);
  const int order = (pairs ? 1 : 0) | (few ? 2 : 0);
  if (pairs || num_seqs > 64 || chunks < 2 || !(few || gy % 8 == 0)) return order;
  if (halves && (few || (!most && va::fa_by_end(bm, bm / pack, gy, row_blocks, chunks, cached > 0)))) return order | 4;
  return order | (most && decodes == 0 ? 8 : 0);
}

#ifdef VA_PROBES
extern "C" int vllm_amd_probe_fa_stamps(unsigned long long* dst, int nwg) {
  return hipMemcpyFromSymbol(dst, HIP_SYMBOL(va::fa::g_fa_stamps), (size_t)nwg * 8 * 8 * 8) == hipSuccess ? 0 : -3;
}
#endif
