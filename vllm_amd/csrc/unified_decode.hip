// unified_attention, decode tokens (every sequence with a query of one token): launches of the kernel in
// unified_decode_kernel.cuh, and the merge of its key segments.
#include "unified_decode_kernel.cuh"

#include <algorithm>

namespace va {

extern int g_uni_decode;

namespace {

// (head 128 sits at the 168 registers of three workgroups per CU: 172 sequences x 80 fp8 keys, 1376 workgroups, 16.4 us against
// 19.6 at two)
template <typename T, bool FP8, int D, int NW, bool GEN>
__global__ __launch_bounds__(NW * 64, (D > 128 && !FP8 ? 1 : D == 128 ? 3 : 2)) void ua_decode_kernel(const UniDecodeParams p, int sub_shift, int xcd_group, int order) {
  __shared__ __attribute__((aligned(16))) char lds[ua_decode_lds<FP8, D, NW>()];
  ua_decode_body<T, FP8, D, NW, GEN, false>(p, lds, sub_shift, xcd_group, order, blockIdx.x, gridDim.x, blockIdx.y);
}

// Merge of the key segments of a split launch (reduce_segments,
// triton_unified_attention.py:499-586): one wave per (sequence, q head).  Lane s holds the max /
// sum of segment s (at most NS), the weights come from two 16-lane butterflies, and the NS partial
// rows are loaded back to back.  Bound by its memory round trips: the rows of token `seq` are requested
// together with the lengths that say which token and how many segments it is -- in a decode step of one
// token per sequence that is the token; if not, they are loaded again -- and rows that no segment wrote
// are left out afterwards.  us, two round trips -> one, with the main kernel and the cache write:
// 1 x 1000 fp8 12.0 -> 11.1, 8 x 3000 ragged of head 64 14.4 -> 13.6, 16 x 6000 ragged 31.8 -> 30.9.
template <typename T, int D, int NS>
__global__ __launch_bounds__(256) void ua_decode_reduce_kernel(const UniDecodeParams p) {
  constexpr int VPL = D / 64;   // outputs per lane
  const int lane = threadIdx.x & 63;
  const int pair = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (pair >= p.num_seqs * p.num_heads) return;
  const int seq = pair / p.num_heads, head = pair % p.num_heads;
  const int dr = p.head_size;
  const bool dval = VPL * lane < dr;
  typedef __attribute__((ext_vector_type(VPL))) float fv;
  fv part[NS];
  float ms, ls;
  auto load = [&](int tok) __attribute__((always_inline)) {
    const int64_t row = ((int64_t)tok * p.num_heads + head) * p.segm_stride;
    const int sl = lane < p.num_segments ? lane : 0;
    ms = p.segm_max[row + sl];
    ls = p.segm_sum[row + sl];
#pragma unroll
    for (int s2 = 0; s2 < NS; ++s2)
      part[s2] = *reinterpret_cast<const fv*>(p.segm_out + (row + min(s2, p.num_segments - 1)) * dr + (dval ? VPL * lane : 0));
  };
  const int guess = min(seq, p.num_tokens - 1);
  load(guess);
  const int qtok = p.cu_seqlens_q[seq];
  if (p.cu_seqlens_q[seq + 1] - qtok != 1) return;
  const int ntiles = (p.seq_lens[seq] + 63) >> 6;
  if (qtok != guess) load(qtok);
  const int tps = (ntiles + p.num_segments - 1) / p.num_segments;
  const int nseg = tps > 0 ? (ntiles + tps - 1) / tps : 0;   // segments the main kernel wrote
  float acc[VPL], l = 0.f;
#pragma unroll
  for (int j = 0; j < VPL; ++j) acc[j] = 0.f;
  if (nseg > 0) {
    ms = lane < nseg ? ms : -INFINITY;
    ls = lane < nseg ? ls : 0.f;
#pragma unroll
    for (int s2 = 0; s2 < NS; ++s2)
      part[s2] = s2 < nseg ? part[s2] : (fv)(0.f);
    float mx = ms;
    mx = row_max16(mx);
    const float w = ms == -INFINITY ? 0.f : fast_exp2(ms - mx);
    l = ls * w;
    l = row_sum16(l);
    l = __shfl(l, 0, 64);
#pragma unroll
    for (int s2 = 0; s2 < NS; ++s2) {
      const float ws = __shfl(w, s2, 64);
#pragma unroll
      for (int j = 0; j < VPL; ++j) acc[j] += part[s2][j] * ws;
    }
  }
  if (!dval) return;
  const float inv = l > 0.f ? 1.0f / l : 0.f;
  const int64_t oidx = (int64_t)qtok * p.o_stride_t + (int64_t)head * p.o_stride_h + VPL * lane;
  if (p.out_scale) {
    const float oi = inv * (1.0f / *p.out_scale);
#pragma unroll
    for (int j = 0; j < VPL; ++j) ((uint8_t*)p.out)[oidx + j] = f32_to_fp8(acc[j] * oi);
  } else {
#pragma unroll
    for (int j = 0; j < VPL; ++j) ((T*)p.out)[oidx + j] = from_f32<T>(acc[j] * inv);
  }
}

template <typename T, bool FP8, int D>
int launch(const UniDecodeParams& p) {
  constexpr int NW = 4;
  int sub_shift = 0;
  while ((16 << sub_shift) < p.block_size) ++sub_shift;
  const int chunks = (p.hp * (p.num_heads / p.num_kv_heads) + 15) / 16;
  const dim3 grid((unsigned)(p.num_seqs * (p.num_kv_heads / p.hp) * chunks), (unsigned)(p.num_segments > 1 ? p.num_segments : 1));
  const int xcd_group = g_uni_decode == 2 ? 1 : g_uni_decode == 3 ? 0 : (grid.x * grid.y >= 1024 ? 1 : 0);
  int order = 0;   // key bits of the longest-first order; tuning "pa_order" = 0 turns it off
  if (pa_order_enabled() && grid.y == 1 && grid.x > 256 && p.num_seqs <= kLptMaxSeqs &&
      (xcd_group ? p.num_seqs % 8 == 0 : grid.x <= 1024)) {
    int ml = p.max_seq_len > 0 ? p.max_seq_len : (1 << 29);
    if (p.window > 0 && p.window < ml) ml = p.window;   // a workgroup streams at most `window` keys
    order = 1;
    while (order < 30 && (ml >> order) != 0) ++order;
  }
  if (p.softcap > 0.f || p.window > 0 || p.alibi_slopes != nullptr)
    hipLaunchKernelGGL((ua_decode_kernel<T, FP8, D, NW, true>), grid, dim3(NW * 64), 0, p.stream, p, sub_shift, xcd_group, order);
  else
    hipLaunchKernelGGL((ua_decode_kernel<T, FP8, D, NW, false>), grid, dim3(NW * 64), 0, p.stream, p, sub_shift, xcd_group, order);
  VA_LAUNCH_CHECK("unified_attention decode launch");
  if (p.num_segments > 1 && p.merge) {
    const dim3 rgrid((unsigned)((p.num_seqs * p.num_heads + 3) / 4));
    if (p.num_segments <= 4) hipLaunchKernelGGL((ua_decode_reduce_kernel<T, D, 4>), rgrid, dim3(256), 0, p.stream, p);
    else if (p.num_segments <= 8) hipLaunchKernelGGL((ua_decode_reduce_kernel<T, D, 8>), rgrid, dim3(256), 0, p.stream, p);
    else hipLaunchKernelGGL((ua_decode_reduce_kernel<T, D, 16>), rgrid, dim3(256), 0, p.stream, p);
    VA_LAUNCH_CHECK("unified_attention decode merge launch");
  }
  return VLLM_AMD_OK;
}

}  // namespace

bool unified_decode_supported(const UniDecodeParams& p) {
  // head sizes up to 256 in whole 16-byte K chunks and 8-element output pieces (padded to 64 / 128 / 256)
  if (p.head_size < 8 || p.head_size > 256 || p.head_size % (p.fp8 ? 16 : 8) != 0) return false;
  // the 256-wide form's lanes own 16 consecutive d of a V row: whole lanes only (136, 152 .. stay with the tile kernel)
  if (p.head_size > 128 && p.head_size % 16 != 0) return false;
  if (p.block_size < 16 || (p.block_size & (p.block_size - 1)) != 0) return false;
  if (p.num_kv_heads <= 0 || p.num_heads % p.num_kv_heads != 0) return false;
  const int es = p.fp8 ? 1 : 2;
  const int vrow = (p.head_size <= 64 ? 4 : p.head_size <= 128 ? 8 : 16) * es;   // bytes of a V row one lane loads (4 .. 32)
  if (p.vc_slot_bytes % vrow || p.vc_block_bytes % vrow || p.vc_head_bytes % vrow) return false;
  if (p.kc_slot_bytes % 16 || p.kc_block_bytes % 16 || p.kc_head_bytes % 16) return false;
  if (p.q_stride_t % 8 || p.q_stride_h % 8 || (((uintptr_t)p.q) & 15)) return false;
  // one thread stores 8 consecutive outputs: 16 bytes (8 with an fp8 output)
  if (p.o_stride_t % 8 || p.o_stride_h % 8 || (((uintptr_t)p.out) & (p.out_scale ? 7 : 15))) return false;
  if (p.num_segments > 16 || (p.num_segments > 1 && (((uintptr_t)p.segm_out) & 15))) return false;
  return true;
}

int g_uni_hp = 0;   // tuning "uni_hp": 0 = heuristic, 1 = never pack kv heads, 2 / 4 = that many when possible

// kv heads taken per workgroup row (see the kernel): token-major caches whose (token, head) rows are shorter than 256
// bytes; the packed width must be one of the instantiations and the q heads of the packed groups fit the 16 columns
int unified_decode_heads_per_row(const UniDecodeParams& p) {
  if (g_uni_hp == 1 || p.num_kv_heads <= 0) return 1;
  const int es = p.fp8 ? 1 : 2, gq = p.num_heads / p.num_kv_heads;
  if (p.kc_head_bytes != (int64_t)p.head_size * es || p.vc_head_bytes != (int64_t)p.head_size * es) return 1;   // heads not adjacent
  if (p.head_size * es >= 256) return 1;                                                                         // long enough
  // rows of up to 128 elements first (largest packing), then the 256-wide form
  for (int pass = 0; pass < 2; ++pass)
  for (int hp = 4; hp >= 2; hp >>= 1) {
    const int w = p.head_size * hp;
    if ((w > 128) != (pass == 1)) continue;
    if ((w != 64 && w != 128 && w != 256) || gq * hp > 16 || p.num_kv_heads % hp != 0) continue;
    if (g_uni_hp > 1) { if (hp > g_uni_hp) continue; }
    else {
      // Measured (16q / 8kv and 8q / 4kv x 4096 tokens, fp8, tools/bench_uni_decode_d.py): rows of up to 128 elements
      // always gain -- head 64: 2 heads per row 92 -> 52 us at 64 sequences, 291 -> 180 at 256 (4 heads per row, the
      // 256-wide form: 59 / 184); head 128 x 2 in the 256-wide form (fp8: 32-token steps, two workgroups per CU):
      // 8 kv heads 102 -> 90 us at 64 sequences, 194 -> 171 at 128, 355 -> 353 at 256, 32.5 -> 32.1 at 16; 4 kv heads
      // 92.8 -> 87.1 at 128, 180 -> 164.5 at 256.  (w * es <= 256: a 16-bit cache never reaches the 256-wide form here.)
      if (w * es > 256) continue;
    }
    const int vrow = (w <= 64 ? 4 : w <= 128 ? 8 : 16) * es;
    if (p.vc_slot_bytes % vrow || p.vc_block_bytes % vrow || (p.vc_head_bytes * hp) % vrow) continue;
    return hp;
  }
  return 1;
}

int g_uni_seg = 0;   // tuning "uni_seg": 0 = heuristic, n = that many key segments (at most those there is scratch for)

int unified_decode_segments(const UniDecodeParams& p, int max_segments) {
  // Split over the keys (when the caller brought scratch).  With the chip counted as 512 slots (two workgroups per CU, as it was
  // fitted; rows of 128 fit three by now, of 64 four) a launch of full-length ones takes ceil(wgs n / 512) / n rounds, and every
  // workgroup pays ~4 us of prologue and merge next to ~25 ns per token of streaming: take the
  // smallest segment count within 5 % of the best estimate (513..1023 workgroups: ~1.3
  // rounds instead of 2); few sequences: as many segments of >= 256 tokens as allowed.
  const int max_k = p.max_seq_len, row = p.head_size * p.hp;
  const int wgs = unified_decode_pairs(p);
  if (max_segments <= 1 || max_k <= 0) return 1;
  if (g_uni_seg > 0) return std::min(g_uni_seg, std::min(max_segments, 16));
  int cap = (max_k + 255) / 256;
  if (cap > max_segments) cap = max_segments;
  if (cap > 16) cap = 16;
  const float ovh = 160.f / (float)max_k;
  // rows above 128 elements: 256 workgroups carry the bytes in flight of 512 narrow ones (16-bit cache: one workgroup
  // per CU; fp8: two of 32-token steps -- counting 512 slots there split 64 x 4096 in two: 93.8 against 89.9 us)
  const int slots = row > 128 ? 256 : 512;
  auto cost = [&](int n) { return (float)((wgs * n + slots - 1) / slots) / n * (1.f + n * ovh); };
  float best = 1e30f;
  for (int n = 1; n <= cap; ++n) best = cost(n) < best ? cost(n) : best;
  int nseg = cap;
  if (wgs * cap > slots)
    for (int n = 1; n <= cap; ++n)
      if (cost(n) <= best * 1.05f) { nseg = n; break; }
  // One piece all the same where what the cut gains does not pay for the merge behind it: 4.5 us and 4 ns for each workgroup.
  // A workgroup alone takes 2.5 ns + 1 ns per 43 bytes for a token, the chip 1 us per 6.2 MB -- the batch taken to be 0.6 full --
  // and both more where some of the 256 CUs have a workgroup more than others.  us, cut -> one piece (32 / 8 heads of 128, fp8):
  // 1 x 500 11.9 -> 9.9, 16 x 777 14.7 -> 13.6, 24 x 500 14.9 -> 11.3, 32 x 1000 ragged 17.9 -> 14.4, 48 x 3000 ragged 40.2 -> 33.8,
  // 96 x 1600 60.1 -> 53.6; 16-bit 32 x 500 19.0 -> 15.8.  Kept cut: 1 x 1600 11.8 (one piece 16.0), 8 x 3000 18.1 (24.2), 40 x 3000
  // 46.7 (51.8), 40 x 3000 ragged 34.3 (30.8).  Over 4625 batches (1 .. 1023 pairs, 257 .. 9000 tokens, head 64 .. 256, both caches;
  // tools/sweep_decode_plans.py, 237 of them in profiles/decode_plans.txt) 3.7 % below always cutting and 0.5 % above the cheaper
  // form on average; more than 2.5 % slower than the cut in 2.4 % of them, since the merge now costs 0.3 .. 1.1 us less than when the
  // price was fitted (4 x 1281 fp8 of 12 heads of 64 11.6 cut, 13.1 so).  Not where the longest sequence may take a workgroup more than
  // 24 us on an idle chip: among short ones it has to be cut.
  const double tb = 2.0 * row * (p.fp8 ? 1 : 2);
  auto us = [&](int n) {
    const int64_t tot = (int64_t)wgs * n;
    const double alone = (double)(((max_k + 63) / 64 + n - 1) / n) * 64 * (2.5e-3 + tb * 2.3e-5);
    const double stream = 0.6 * (double)wgs * max_k * tb / 6.2e6;
    const double over = tot >= 256 ? (double)((tot + 255) / 256 * 256) / (double)tot - 1.0 : 0.0;
    return (alone > stream ? alone : stream) * (1.0 + 1.6 * over * over) + (n > 1 ? 4.5 + 0.004 * (double)tot : 0.0);
  };
  return nseg > 1 && max_k * (2.5e-3 + tb * 1.2e-5) <= 24.0 && us(1) < 0.98 * us(nseg) ? 1 : nseg;
}

int unified_decode(const UniDecodeParams& p) {
  const int w = p.head_size * p.hp;   // (hp from unified_decode_heads_per_row, or 1)
#define L(T) \
  (w > 128 ? (p.fp8 ? launch<T, true, 256>(p) : launch<T, false, 256>(p))  \
   : w > 64 ? (p.fp8 ? launch<T, true, 128>(p) : launch<T, false, 128>(p)) \
                      : (p.fp8 ? launch<T, true, 64>(p) : launch<T, false, 64>(p)))
  return p.dtype == VLLM_AMD_F16 ? L(f16_t) : L(bf16_t);
#undef L
}

}  // namespace va
