// unified_attention (vllm/attention/ops/triton_unified_attention.py:52-272, 588-700) and context_attention_fwd
// (vllm/attention/ops/prefix_prefill.py:36-288, 726-913; the PREFIX instantiation below) with the causal + padding mask
// (unified: + sliding window, softcap): chunks that fill row blocks, at head sizes 72 .. 256, and -- split over the keys, head
// sizes 8 .. 256 -- any chunk of more than one token where few row blocks have long key ranges (fa_plan in
// prefill_attention.hip).  The matrix-core-bound case of prefill_attention.hip, re-built around what bounds that kernel (16 query rows per wave = one LDS fragment byte per
// 32 flops and ~300 VALU per 32 MFMAs; a 64-row tile restages every K / V tile for 64 rows).
//
//   * a workgroup = 8 waves = 256 tile rows; a wave owns 32 rows and computes with v_mfma_f32_32x32x16:
//     every K / V fragment read from LDS feeds 32 rows (half the LDS bytes per flop of the 16-row form), a K / V
//     tile is staged once per 256 rows (a quarter of the staging work per flop);
//   * rows are (token, q head of ONE kv head's GQA group) pairs, token-major, as the reference packs
//     BLOCK_M / num_queries_per_kv tokens (:612-613): K / V stream once per group;
//   * the transposed problem, as in the decode kernel:  S^T[n, m] = K[n, :] . Q[m, :]  (A = K rows from LDS,
//     B = Q^T from registers),  O^T[d, m] += V^T[d, n] . P^T[n, m]  (A = V^T by the transposing LDS read
//     ds_read_b64_tr_b16 from the row-major V tile, B = P^T).  A lane holds ONE query row (column m) of S^T:
//     row max and sum need one cross-half exchange, and the C layout of S^T (keys (r & 3) + 8 (r >> 2) + 4 hi of
//     a 32-key block) is the B layout of P^T once the contraction slots of the PV product are numbered the
//     same way -- the V^T fragment is simply read in that order.  P never leaves the registers;
//   * K / V tiles of 64 keys, double-buffered in LDS (64 KiB), one barrier per tile: registers hold tile t + 1
//     while tile t is computed; in interval t they are written to the other buffer (fp8 widened exactly on the way)
//     and the loads of tile t + 2 are issued -- by waves 0-3 behind their compute, by waves 4-7 in front of it, so
//     that one wave of every SIMD stages while its partner is in its MFMA sections;
//   * the running max is updated lazily: O and l are rescaled only when some row's tile max exceeds the
//     running max by more than 2^8 (the probabilities then reach at most 256, exact in the 16-bit formats'
//     exponent range; every row is normalised by its own sum at the end).
//
// fp8 cache: K / V are widened exactly (e4m3 is a subset of f16 / bf16), k_scale rides in the score scale,
// v_scale in the softmax exponent (one rounding fewer than the reference's (fp8 * scale).to(dtype)).
#pragma once
#include "mma.cuh"
#include "prefill_fa.cuh"

#include <float.h>
#include <type_traits>

namespace va {
namespace fa {

typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;
typedef __attribute__((ext_vector_type(2))) unsigned int u32x2;

template <typename T> struct Mma32;
template <> struct Mma32<bf16_t> {
  static __device__ __forceinline__ f32x16 mfma(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                   0, 0, 0);
  }
};
template <> struct Mma32<f16_t> {
  static __device__ __forceinline__ f32x16 mfma(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c,
                                                  0, 0, 0);
  }
};

constexpr int BN = 64;            // keys per tile
constexpr int KN = 2, VN = 2;     // K / V tiles in LDS (rings indexed by the tile number)
#ifndef FA_KRW
#define FA_KRW 8
#define FA_VRW 4
#endif
constexpr int KR128 = 8, VR128 = 4;   // fragment reads in flight: K reads, V^T fragments (two transposing reads each)
constexpr int KR256 = FA_KRW, VR256 = FA_VRW;
constexpr float THR = 8.f;        // lazy rescale threshold (log2 domain)
constexpr int ONE_SEG = 3;        // a row block of up to this many tiles is not split

// One v_maximum3_f32.  (fmaxf on MFMA results makes hipcc canonicalise every input first; inline asm must not read them
// at all: the wait states between an MFMA and a VALU read of its result are the compiler's to insert, it inserts none in
// front of an asm block, and the hardware does not wait -- the row maximum then came from a sum still being accumulated.)
__device__ __forceinline__ float max3(float a, float b, float c) {
  return __builtin_elementwise_maximum(__builtin_elementwise_maximum(a, b), c);
}
__device__ __forceinline__ u32x2 lds_tr16(const uint8_t* p) {
  typedef __attribute__((ext_vector_type(4))) short s16x4;
  const s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)p);
  return __builtin_bit_cast(u32x2, v);
}

// Sum of v over the lanes up to and with this one (DPP: rows of 16, then the rows' last lanes)
__device__ __forceinline__ int wave_scan(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);   // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);   // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);   // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);   // row_shr:8
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);   // row_bcast:15 into rows 1, 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);   // row_bcast:31 into rows 2, 3
  return v;
}

__device__ __forceinline__ int wave_max_i(int v) {   // (lanes without a source keep their own value)
  v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x111, 0xf, 0xf, false));
  v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x112, 0xf, 0xf, false));
  v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x114, 0xf, 0xf, false));
  v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x118, 0xf, 0xf, false));
  v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x142, 0xa, 0xf, false));
  v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x143, 0xc, 0xf, false));
  return __builtin_amdgcn_readlane(v, 63);
}

// -DVA_PROBES (tools/fa_stamps.py): shader-clock time per wave spent in each part of the tile loop, summed over
// the wave's tiles: 0 K ring fill + staging (LDS writes of tile t + 1, loads of t + 2), 2 S^T, 4 softmax + PV,
// 5 barrier, 6 tiles computed, 7 whole kernel
#ifdef VA_PROBES
static __device__ unsigned long long g_fa_stamps[2048 * 8 * 8];   // (one for each file that launches the kernel, with its reader)
#define FA_T(i)                                                   \
  do {                                                            \
    const unsigned long long now__ = __builtin_readcyclecounter(); \
    acc__[i] += now__ - last__;                                   \
    last__ = now__;                                               \
  } while (0)
#else
#define FA_T(i) do { } while (0)
#endif

// Where a workgroup works: row block `blk` of sequence `seq` (its first query token tok0, its lengths), grid row y, and in split
// launches the key segment `seg` of `segs`.  pair: not rows of one row block, but of the blk-th half block from the front and the
// blk-th from the back.
struct FaAt { bool some = false, pair = false; int seq, blk, y, seg, segs, tok0, qlen, seq_len; };

// hw: the workgroup's hardware id in a grid of gx x gy (of the launch's first gx gy workgroups: ids go round-robin over the XCDs),
// an upper bound of the row blocks there are (gx = num_tokens / tpb + num_seqs, or blocks_per_seq * num_seqs where the caller did
// not say how many query tokens there are; 1, 2 or 4 heads: gx gy a multiple of 8).
// MIXED: behind the row blocks the launch has a workgroup for every (decode, kv head).
template <bool PREFIX, bool SPLIT, bool MIXED, int BM>
__device__ __forceinline__ FaAt fa_find(const FaParams& p, int lane, int hw, int gy) {
  // ---- workgroup -> (row block of some sequence, head).  Hardware ids go round-robin over the XCDs: the
  // bijective remap gives every XCD a contiguous range of logical ids (row blocks fastest, then heads), so the
  // row blocks and heads that read the same K / V share an L2; later (longer) row blocks first.
  auto xcd_order = [hw](int nwg) __attribute__((always_inline)) {   // -1: more workgroups than work
    const int q8 = nwg / 8, r8 = nwg % 8, xcd = hw % 8, idx = hw / 8;
    return idx < q8 + (xcd < r8 ? 1 : 0) ? (xcd < r8 ? xcd * (q8 + 1) : r8 * (q8 + 1) + (xcd - r8) * q8) + idx : -1;
  };
  const int nseg = SPLIT ? p.num_segments : 1;
  const int tpb = p.tpb;                      // tokens per workgroup
  const int tsh = (tpb & (tpb - 1)) == 0 ? __builtin_ctz(tpb) : -1;   // (a division here is 1 % of a short row block)
  FaAt at;
  at.seg = 0;
  at.segs = 1;
  // The row blocks there really are, and in split launches seg_slots workgroups dealt out to them: as num_segments workgroups for
  // each block there may be, a launch spent 2.2 ns on each one of a sequence that the decode kernel takes (100 fresh tokens among
  // 60 decodes of 3000 keys, 32 / 8 heads: 4032 workgroups, whole step 86.7 us, now 75.1; 200 over 3800 among 100 of 700: 91.7
  // -> 66.0).  The work goes evenly over the XCDs: a few blocks too many on one of them double up on its CUs (512 over 7488,
  // 8 q / 1 kv head: 60 against 40 us), and so do those of a launch in whose grid every other workgroup is empty (32 chunks of 64
  // tokens over 6000 keys, one row block each, in a grid of 64 a head: 232 -> 180; 16 of 60 .. 100 over 1500 .. 3000 among 40 decodes
  // 119 -> 101).
  struct Seq { int tok0, qlen, len, blocks; };
  auto seq_at = [&](int i) __attribute__((always_inline)) {   // (lengths too: the found sequence's need no load of their own)
    Seq q = {0, 0, 0, 0};
    if (i < p.num_seqs) {
      q.tok0 = p.cu_seqlens_q[i];
      q.qlen = p.cu_seqlens_q[i + 1] - q.tok0;
      q.len = p.seq_lens[i];
      q.blocks = p.skip_decode && q.qlen == 1 ? 0 : tsh >= 0 ? (q.qlen + tpb - 1) >> tsh : (q.qlen + tpb - 1) / tpb;
    }
    return q;
  };
  Seq my = seq_at(lane);                                    // the first 64 sequences stay in registers
  int incl = wave_scan(my.blocks);
  int here = __builtin_amdgcn_readlane(incl, 63), total = here;
  const unsigned long long chunks = __ballot(my.blocks > 0);
  int nchunks = 0, nover = 0;   // sequences with row blocks, those of them over contexts at least twice as long
  if constexpr (!SPLIT) {
    nchunks = (int)__popcll(chunks);
    nover = (int)__popcll(__ballot(my.blocks > 0 && my.len >= 3 * my.qlen));
  }
  for (int i = 64; i < p.num_seqs; i += 64) {
    const Seq q = seq_at(i + lane);
    total += __builtin_amdgcn_readlane(wave_scan(q.blocks), 63);
    if constexpr (!SPLIT) {
      nchunks += (int)__popcll(__ballot(q.blocks > 0));
      nover += (int)__popcll(__ballot(q.blocks > 0 && q.len >= 3 * q.qlen));
    }
  }
  if (total == 0) return at;
  const int work = SPLIT ? max(total, min(p.seg_slots, total * nseg)) : total;   // per head
  // Most chunks are short ones over contexts at least twice as long: a sequence's blocks read the same keys, and belong together.
  // (Of all sequences: an engine's decodes come first, and of the first 64 alone none may be a chunk.)
  const bool over = !SPLIT && 2 * nover >= nchunks;
  // One round of workgroups ends with its longest one, and under the causal mask the rows of a block differ in length by up to the
  // chunk: each takes four waves' rows from the front of the chunk and four from its back, which all add up to the same.
  // (A SIMD's second wave is done early; the first one then walks on alone at 1.2 us a tile, two take 1.9.)
  // us, 32 / 8 heads, with the cache write: 2000 fresh tokens 69.5 -> 61.5, 1700 over 300 68 -> 60, 2000 over 1500 116 -> 107; 8 / 1
  // heads 6000 fresh 198 -> 172.  Beside more decodes than the same round has CUs for, those of short row blocks do not idle, and row blocks
  // of one length leave the decodes to the end (2000 over 1500 among 63 of up to 4096 keys 143 -> 152 us, 2048 fresh among 48 of 2000
  // 69 -> 81); up to that, 8 / 1 heads, 5000 fresh among 40 of 1000 138 -> 109, 2 x 3000 among 20 of 3000 87 -> 71.
  const int decodes = !MIXED ? 0 : p.num_seqs > 64 ? p.num_seqs : (int)__popcll(__ballot(my.qlen == 1));
  at.pair = !SPLIT && fa_pairs(BM, p.halves, gy, total, decodes, p.window);
  // 1, 2 or 4 heads, several rounds: every XCD takes its share of a head's blocks one by one.  In runs the long ones meet on the
  // first XCDs (8 / 1 heads, 10000 fresh tokens 483 -> 277 us, 3 x 5000 231 -> 155; 16 / 4, 6000 229 -> 184; head 256 8 / 2, 4460 + 3411
  // tokens 608 -> 453; window 7792 of 13000 914 -> 545).  Not in one round of several chunks, where blocks do not wait for each other and a run's share their
  // keys: 2 % on average over 50 steps that are not paired (head size 256, windows, groups that do not divide 128, beside decodes; 16 / 4, head 256,
  // 14 chunks of 61 .. 98 28.9 us in shares, 27.6 in runs); those of one chunk differ most in length, and shares spread them (6 / 1 heads, 9061
  // fresh 251 in runs, 237 in shares).
  const bool few = !SPLIT && fa_few(p.shares, gy, total, nchunks, at.pair, over, p.window);
  int gs;
  if (few) {
    const int per = p.shares, xcd = hw % 8;
    at.y = xcd / per;
    gs = hw / 8 * per + xcd % per;
    if (gs >= work) return at;
  } else {
    const int w = xcd_order(work * gy);
    if (w < 0) return at;
    at.y = w / work;
    gs = w - at.y * work;
  }
  auto take = [&](int l) __attribute__((always_inline)) {
    at.some = true;
    at.tok0 = __builtin_amdgcn_readlane(my.tok0, l);
    at.qlen = __builtin_amdgcn_readlane(my.qlen, l);
    at.seq_len = __builtin_amdgcn_readlane(my.len, l);
  };
  if constexpr (!SPLIT) {
    if (!at.pair && p.num_seqs <= 64 && (few || gy % 8 == 0) && nchunks > 1) {
      // Several chunks: an XCD's workgroups start in this order, and what it ends on should be short.  The row blocks in the order of
      // their last keys, those with most of them first, in 64 steps of the range: lane l counts the blocks of its step and the ones
      // before it.  What that costs are the keys: row blocks of other chunks run at the same time, and each chunk's keys are read for fewer
      // query tokens at once, 32 tpb / chunks of them on an XCD (us: 8 x 300 .. 500 over 250 .. 500, 256 tokens, 70 -> 66, 5 x 540 .. 900 fresh 61
      // -> 57, 16 / 8 heads 12 x 133 .. 587 96 -> 80; but 64 / 8 13 x 95 .. 154 fresh, 79 tokens, 35.0 -> 36.3).  By the last
      // keys / by sequence, up to two rounds 135 steps of 160 tokens and more 0.946 (three more than 2 % slower), 28 of 128 .. 159 0.979 (three, by up to
      // 3 %; 13 x 202 .. 336 fresh 42.5 -> 44.3), 16 of fewer 0.996 (five, by up to 5 %).  In more rounds what a launch ends on matters less, and the
      // blocks wait for keys that have left the L2: without a context 92 steps below 520 tokens 1.029 (by up to 12 %), 108 from 640 on, up to eight
      // rounds, 0.972 (four) -- three prompts for a group of 4 q heads, six for one of 2, twelve without (32 / 32, 3605 + 3260 309 -> 282, 16 / 8, 6 x
      // 735 .. 2825 181 -> 173, 32 / 8, 2606 + 2515 + 1572 168 -> 164, 3001 + 5003 317 -> 312) --, beyond eight rounds 0.992 of 11.  Over
      // contexts, whose keys every block reads, 0.997 of 80.  Above head size 128 a tile takes long enough for keys from anywhere (5 x 550 .. 917 fresh
      // 76 -> 68, 3 x 1200 .. 2000 143 -> 132).
      const bool cached = __ballot(my.blocks > 0 && my.len > my.qlen) != 0;
      if (p.halves && (few || (!over && fa_by_end(BM, tpb, gy, total, nchunks, cached)))) {
        const int sh = __builtin_ctz(tpb), ctx = my.len - my.qlen;
        const int top = wave_max_i(my.blocks > 0 ? ctx + (my.blocks << sh) : 0), low = -wave_max_i(my.blocks > 0 ? -ctx : -top);
        const int step = ((top - low) >> 6) + 1;
        // blocks of a sequence whose last key is beyond `end`
        auto beyond = [&](int end, int ctx_, int n) __attribute__((always_inline)) { return n - min(max((end - ctx_) >> sh, 0), n); };
        int upto = 0;
        const int end = top - (lane + 1) * step;
        for (unsigned long long m = chunks; m != 0; m &= m - 1) {
          const int j = __ffsll((long long)m) - 1;
          upto += beyond(end, __builtin_amdgcn_readlane(ctx, j), __builtin_amdgcn_readlane(my.blocks, j));
        }
        const int l = __builtin_amdgcn_readfirstlane(__ffsll((long long)__ballot(upto > gs)) - 1);
        const int r = gs - (l > 0 ? __builtin_amdgcn_readlane(upto, l - 1) : 0);
        const int before = beyond(top - l * step, ctx, my.blocks), n = beyond(top - (l + 1) * step, ctx, my.blocks) - before;
        const int sum = wave_scan(n);
        at.seq = __builtin_amdgcn_readfirstlane(__ffsll((long long)__ballot(r < sum)) - 1);
        at.blk = __builtin_amdgcn_readlane(my.blocks - 1 - before + (sum - n), at.seq) - r;
        take(at.seq);
        return at;
      }
      // Short chunks over long contexts: the row blocks of the longest sequence first (24 chunks of 150 .. 250 over 1500 .. 3000 tokens,
      // three rounds of workgroups: 266 -> 257 us, the flash layout 260 -> 250; 19 prompts of 745 .. 1242 without context, whose
      // blocks differ more than the prompts, 294 -> 302: they keep the order below).
      if (over && decodes == 0) {
        int before = 0;                        // blocks of longer sequences
        const uint32_t key = (uint32_t)my.len << 6 | (uint32_t)(63 - lane);   // (no two alike)
#pragma unroll 4
        for (int j = 0; j < p.num_seqs; ++j)
          before += (uint32_t)__builtin_amdgcn_readlane((int)key, j) > key ? __builtin_amdgcn_readlane(my.blocks, j) : 0;
        const unsigned long long mine = __ballot(before <= gs && gs < before + my.blocks);
        at.seq = __builtin_amdgcn_readfirstlane(__ffsll((long long)mine) - 1);
        at.blk = __builtin_amdgcn_readlane(my.blocks, at.seq) - 1 - (gs - __builtin_amdgcn_readlane(before, at.seq));
        take(at.seq);
        return at;
      }
    }
  }
  int b = gs;
  if constexpr (SPLIT) {
    at.seg = gs / total;
    b = gs - at.seg * total;                                // (a segment's row blocks are adjacent, they read the same K / V)
    at.segs = work / total;
    at.segs += b < work - at.segs * total ? 1 : 0;
  }
  b = total - 1 - b;                                        // later (longer) row blocks first
  for (int i = 0; i < p.num_seqs; i += 64) {
    if (i > 0) {
      my = seq_at(i + lane);
      incl = wave_scan(my.blocks);
      here = __builtin_amdgcn_readlane(incl, 63);
    }
    if (b < here) {
      const int l = __builtin_amdgcn_readfirstlane(__ffsll((long long)__ballot(b < incl)) - 1);
      at.seq = i + l;
      at.blk = b - __builtin_amdgcn_readlane(incl - my.blocks, l);
      take(l);
      break;
    }
    b -= here;
  }
  return at;
}

// PREFIX = context_attention_fwd (vllm/attention/ops/prefix_prefill.py:36-288, 726-913): the keys are the sequence's
// cached context -- K [block][kv head][D / x][BS][x] (x = 16 bytes), V [block][kv head][D][BS], every cached token
// visible -- followed by the new tokens' dense k / v (causal).  Context V is already V^T: its tile is staged as
// [d][token] (16-byte units XOR-swizzled by d >> 1) and the PV MFMA's A operand is one plain 16-byte read; the new
// tokens take the unified path's row-major image and transposing reads.  Dense k / v are never fp8.
//
// D_ = 128, NW_ = 8: head sizes 72 .. 128 (split over the keys: 8 .. 128), eight waves = 256 rows, two waves per SIMD.
// D_ = 256, NW_ = 4: head sizes 136 .. 256: O^T alone is 128 registers for a wave's 32 rows and Q^T 64, so a wave takes a
// whole SIMD's register file: four waves = 128 rows, one per SIMD, 32 KiB tiles (128 KiB of LDS), 32 + 32 MFMAs per tile.
// SOFTCAP (unified_attention): scores softcap * tanh(score / softcap) (triton_unified_attention.py:219-221): a pass of
// ~9 VALU per score between S^T and the softmax, in its own instantiation.
// SPLIT: num_segments > 1, in its own instantiation (the 256-wide forms have no register to spare).
template <int D_> constexpr int fa_lds() { return (KN + VN) * BN * 2 * D_; }   // 64 / 128 KiB
template <typename T, bool FP8, bool PREFIX, int D_, int NW_, bool SOFTCAP, bool SPLIT, bool MIXED = false>
__device__ __forceinline__ void fa_body(const FaParams& p, uint8_t* lds, int hw, int gy) {
  constexpr int NW = NW_, BM = 32 * NW, D = D_;
  constexpr int ROWB = 2 * D;       // bytes per LDS row (one key, D 16-bit values)
  constexpr int TILE = BN * ROWB;   // 16 / 32 KiB
  constexpr int K_OFF = 0, V_OFF = KN * TILE;
  constexpr int KS = D / 16, DB = D / 32;         // k-steps of S^T, d blocks of O^T
  constexpr int KR = D > 128 ? KR256 : KR128, VR = D > 128 ? VR256 : VR128;
  constexpr int PPK = D / 16;                     // 32-byte staging pieces per key
  constexpr int NTHR = 64 * NW, IPT = BN * PPK / NTHR, KSTEP = NTHR / PPK;   // staging items per thread, keys between them
  static_assert(IPT * NTHR == BN * PPK && (IPT == 1 || KSTEP % 16 == 0) && 4 * D == IPT * NTHR, "");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hi = lane >> 5;
  // ablations are compile-time (-DVA_FA_ABL=bits, tools/fa_stamps.sh; garbage results: 1 no exp2, 2 no staging after the first
  // tiles, 4 no S^T MFMAs, 8 no PV MFMAs): a run-time branch around every MFMA costs the schedule it is meant to measure
#ifndef VA_FA_ABL
#define VA_FA_ABL 0
#endif
  constexpr int abl = VA_FA_ABL;
#ifdef VA_PROBES
  unsigned long long acc__[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  const unsigned long long t_entry__ = __builtin_readcyclecounter();
  unsigned long long last__ = t_entry__;
#endif

  const FaAt at = fa_find<PREFIX, SPLIT, MIXED, BM>(p, lane, hw, gy);
  if (!at.some) return;
  const int nseg = SPLIT ? p.num_segments : 1;
  const int pack = p.pack, tpb = p.tpb;       // tokens per workgroup
  const int seq = at.seq, blk = at.blk, y = at.y, seg = at.seg, segs = at.segs, tok0 = at.tok0, qlen = at.qlen, seq_len = at.seq_len;
  const int ctx = seq_len - qlen;
  // first query token of this block
  const int tok_base = blk * tpb;
  // The rows of this wave: those of its half of the workgroup (waves 0-3 and 4-7, where the group divides into 128 rows) from row
  // hrow0 and token htok on
  const bool halves = NW == 8 && p.halves;
  const int htpb = halves ? tpb / 2 : tpb, hrow0 = halves && wave >= 4 ? 128 : 0;
  int htok = tok_base + hrow0 / pack, new_end = min(tok_base + tpb, qlen);
  if (at.pair) {
    const int front = blk * htpb, back = ((qlen + htpb - 1) / htpb - 1 - blk) * htpb;
    htok = wave < 4 ? back : (front < back ? front : qlen);   // (the middle half of an odd number: nothing for waves 4-7)
    new_end = min(back + htpb, qlen);
  }
  const int kvh = pack > 1 ? y : y / (p.num_heads / p.num_kv_heads);
  // head sizes up to 128 (multiples of 8; 16 with an fp8 cache) run padded to 128, above to 256: the columns d >= dr of Q, K and V are
  // staged as zeros from clamped addresses, the output columns are not stored
  const int dr = p.head_size;

  // ---- this lane's query row: tile row 32 wave + l32 -> (token, head) ----------------------------------------
  const int wrow = 32 * wave - hrow0, hrow = wrow + l32;
  const int rtok = htok + hrow / pack;
  const int rhead = pack > 1 ? kvh * pack + hrow % pack : y;
  const bool rok = hrow < htpb * pack && rtok < qlen;
  // last visible key: among the new-domain keys (UNI: every key, by position; PREFIX: the new tokens, by index) and
  // among the context keys (PREFIX)
  const int bound_new = rok ? (PREFIX ? rtok : ctx + rtok) : -1;
  const int bound_ctx = rok ? ctx - 1 : -1;

  // tiles: ctx_tiles of the context (PREFIX), then the new domain's
  const int ctx_tiles = PREFIX ? (ctx + BN - 1) / BN : 0;
  const int new_tiles = ((PREFIX ? new_end : ctx + new_end) + BN - 1) / BN;
  const int ntiles = ctx_tiles + new_tiles;
  const int window = PREFIX ? 0 : p.window;          // keys (position - window, position] are visible; 0 = all
  // (sliding window: the tiles left of the window of the workgroup's first row are not even staged)
  const int t_start = window > 0 ? max(ctx + tok_base - window + 1, 0) / BN : 0;
  // Split: this segment's share [t0, t1) of the block's tiles.  The host plans for the longest sequence it was told of -- of a
  // decode beside the chunks, or for the width of the block table -- so a block of up to ONE_SEG tiles is one segment, which
  // writes its output itself, segments without a tile leave here, and segment 0 tells the merge how many there are: -live in
  // the last place of the sums, which is free unless all num_segments are live.
  const int walk = ntiles - t_start;
  const int per = !SPLIT || segs == 1 || walk <= ONE_SEG ? max(walk, 1) : (walk + segs - 1) / segs;
  const int live = SPLIT ? max((walk + per - 1) / per, 1) : 1;
  const int t0 = t_start + seg * per, t1 = min(t0 + per, ntiles);
  if (seg >= live) return;
  // Q^T fragments (B operand of S^T): column m = this row, k = d = 16 ks + 8 hi + (0..7)
  u32x4 qf[KS];
  {
    const T* qp = (const T*)p.q + (int64_t)(tok0 + (rok ? rtok : 0)) * p.q_stride_t + (int64_t)(rok ? rhead : 0) * p.q_stride_h;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const bool dok = 16 * ks + 8 * hi < dr;   // padded head sizes: zero columns
      const u32x4 v = *reinterpret_cast<const u32x4*>(qp + (dok ? 16 * ks + 8 * hi : 0));
      qf[ks] = (rok && dok) ? v : (u32x4){0, 0, 0, 0};
    }
  }
  // wave-uniform: the tokens of the wave's rows
  const bool w_rows = wrow < htpb * pack && htok + wrow / pack < qlen;
  const int w_lo = (PREFIX ? 0 : ctx) + htok + wrow / pack;
  const int w_hi = (PREFIX ? 0 : ctx) + min(htok + (wrow + 31) / pack, min(htok + htpb, qlen) - 1);

  float kscale = 1.f, vscale = 1.f;
  if constexpr (FP8) { kscale = *p.k_scale; vscale = *p.v_scale; }
  const float sc2 = p.sm_scale * kLog2e;             // > 0 (host checks sm_scale)
  const float sc2k = sc2 * kscale;                   // fp8 keys: k_scale rides in the score scale
  const float vlog2 = FP8 ? log2f(vscale) : 0.f, vinv = FP8 ? 1.0f / vscale : 1.f;

  const int* bt = p.block_table + (int64_t)seq * p.bt_stride;
  const int last_page = PREFIX ? (ctx > 0 ? (ctx - 1) >> p.bs_shift : 0) : (seq_len - 1) >> p.bs_shift;

  // ---- staging: item = tid + NTHR i -> (key, two 8-column chunks ca and cb of its row), a wave's keys side by side ----------
  // Eight lanes write 16 bytes each per LDS cycle, to banks 128 bytes apart at most: chunk numbers that differ modulo 8.  As 2 piece
  // and 2 piece + 1 of one key every write took two cycles (SQ_LDS_BANK_CONFLICT: 256 cycles a tile).  PAIR (16 fp8 values of
  // a load are two neighbouring chunks): four pieces each of two keys, whose swizzles differ in the lowest bit; else the eight
  // lanes of a key write eight chunks in a row, and load 128 bytes in a row.
  constexpr bool PAIR = FP8;
  constexpr int WK = 64 / PPK;                                     // keys of a wave
  const int lkey = PAIR ? ((lane >> 2) & 1) | ((lane / (2 * PPK)) << 1) : lane / PPK;
  const int spiece = PAIR ? (lane & 3) | (((lane >> 3) & (PPK / 4 - 1)) << 2) : lane % PPK;
  const int wkey = WK * wave, skey = wkey + lkey;
  const int ca = PAIR ? 2 * spiece : spiece, cb = PAIR ? 2 * spiece + 1 : spiece + PPK;
  const bool pv0 = 8 * ca < dr, pv1 = 8 * cb < dr;                 // the thread's two chunks exist
  const int cal = pv0 ? ca : 0, cbl = pv1 ? cb : 0;                // clamped
  constexpr int NST = (FP8 && !PREFIX) ? 1 : 2;
  u32x4 kst[IPT][NST], vst[IPT][NST];
  // PREFIX, context V^T: item -> (d = item % D, tokens 16 vq .. of the tile with vq = item / D)
  auto vd_of = [&](int i) __attribute__((always_inline)) { return (tid + NTHR * i) % D; };
  auto vq_of = [&](int i) __attribute__((always_inline)) { return (tid + NTHR * i) / D; };
  // A wave's items are 64 / PPK = 8 (D = 256: 4) neighbouring keys and, for the context V^T, one group of 16 tokens: inside
  // one block of the cache (16 slots or more), so block ids and base addresses are wave-uniform -- scalar arithmetic -- and
  // a lane adds a 32-bit constant.  (Per-lane 64-bit products cost ~400 of the ~4100 cycles of a tile on every SIMD.)
  auto wvq_of = [&](int i) __attribute__((always_inline)) { return (64 * wave + NTHR * i) / D; };
  uint32_t koff, koff1 = 0, voff, voff1 = 0;                       // context / paged part: first and second 16 bytes
  uint32_t vtoff[IPT];
  if constexpr (PREFIX) {
    koff = (uint32_t)((((FP8 ? cal / 2 : cal) << p.bs_shift) + lkey) << 4);
    koff1 = FP8 ? 0 : (uint32_t)(((cbl << p.bs_shift) + lkey) << 4);
#pragma unroll
    for (int i = 0; i < IPT; ++i) vtoff[i] = (uint32_t)((min(vd_of(i), dr - 1) << p.bs_shift) * (FP8 ? 1 : 2));
    voff = 0;
  } else {
    koff = (uint32_t)lkey * (uint32_t)p.kc_slot_bytes + (FP8 ? 8 : 16) * cal;
    voff = (uint32_t)lkey * (uint32_t)p.vc_slot_bytes + (FP8 ? 8 : 16) * cal;
    koff1 = (uint32_t)lkey * (uint32_t)p.kc_slot_bytes + 16 * cbl;
    voff1 = (uint32_t)lkey * (uint32_t)p.vc_slot_bytes + 16 * cbl;
  }
  struct Blk { int k[IPT], v[IPT]; };
  auto load_blk = [&](int t) __attribute__((always_inline)) {
    Blk b;
#pragma unroll
    for (int i = 0; i < IPT; ++i) {
      b.k[i] = 0; b.v[i] = 0;
      if constexpr (PREFIX) {
        if (t < ctx_tiles) {
          b.k[i] = bt[min((t * BN + wkey + KSTEP * i) >> p.bs_shift, last_page)];
          b.v[i] = bt[min((t * BN + 16 * wvq_of(i)) >> p.bs_shift, last_page)];
        }
      } else {
        if (t < ntiles) b.k[i] = bt[min((t * BN + wkey + KSTEP * i) >> p.bs_shift, last_page)];
      }
    }
    return b;
  };
  auto ld16 = [](const void* ptr) __attribute__((always_inline)) { return *reinterpret_cast<const u32x4*>(ptr); };
  // (one branch per tile, not per item: hipcc copies the loaded registers at every join)
  auto issue_ctx = [&](int t, const Blk& blk) __attribute__((always_inline)) {
    const int bsm = (1 << p.bs_shift) - 1;
#pragma unroll
    for (int i = 0; i < IPT; ++i) {
      const int slot = (t * BN + wkey + KSTEP * i) & bsm, slot0 = (t * BN + 16 * wvq_of(i)) & bsm;
      const uint8_t* kb = p.k_cache + (int64_t)__builtin_amdgcn_readfirstlane(blk.k[i]) * p.kc_block_bytes + (int64_t)kvh * p.kc_head_bytes + (slot << 4);
      kst[i][0] = ld16(kb + koff);
      if constexpr (!FP8) kst[i][1] = ld16(kb + koff1);
      const uint8_t* vb = p.v_cache + (int64_t)__builtin_amdgcn_readfirstlane(blk.v[i]) * p.vc_block_bytes + (int64_t)kvh * p.vc_head_bytes + slot0 * (FP8 ? 1 : 2);
      vst[i][0] = ld16(vb + vtoff[i]);
      if constexpr (!FP8) vst[i][1] = ld16(vb + vtoff[i] + 16);
      // (dead until a tile of new tokens: said so, hipcc does not carry -- copy, wait for -- them around the loop)
      if constexpr (FP8) {
        kst[i][NST - 1] = __builtin_nondeterministic_value(kst[i][NST - 1]);
        vst[i][NST - 1] = __builtin_nondeterministic_value(vst[i][NST - 1]);
      }
    }
  };
  auto issue_new = [&](int t, auto fast_c) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < IPT; ++i) {
      if constexpr (decltype(fast_c)::value) {   // every row exists: a scalar base and a lane constant
        const int64_t row = tok0 + (t - ctx_tiles) * BN + wkey + KSTEP * i;
        const T* kb = (const T*)p.k_new + row * p.k_stride_t + (int64_t)kvh * p.k_stride_h;
        const T* vb = (const T*)p.v_new + row * p.v_stride_t + (int64_t)kvh * p.v_stride_h;
        const uint32_t ko = (uint32_t)lkey * (uint32_t)p.k_stride_t + 8 * ca, vo = (uint32_t)lkey * (uint32_t)p.v_stride_t + 8 * ca;
        kst[i][0] = ld16(kb + ko); kst[i][NST - 1] = ld16(kb + ko + 8 * (cb - ca));
        vst[i][0] = ld16(vb + vo); vst[i][NST - 1] = ld16(vb + vo + 8 * (cb - ca));
        continue;
      }
      const int64_t row = tok0 + min((t - ctx_tiles) * BN + skey + KSTEP * i, qlen - 1);
      const T* kr = (const T*)p.k_new + row * p.k_stride_t + (int64_t)kvh * p.k_stride_h;
      const T* vr = (const T*)p.v_new + row * p.v_stride_t + (int64_t)kvh * p.v_stride_h;
      kst[i][0] = ld16(kr + 8 * cal); kst[i][NST - 1] = ld16(kr + 8 * cbl);
      vst[i][0] = ld16(vr + 8 * cal); vst[i][NST - 1] = ld16(vr + 8 * cbl);
    }
  };
  auto issue_paged = [&](int t, const Blk& blk) __attribute__((always_inline)) {
    const int bsm = (1 << p.bs_shift) - 1;
#pragma unroll
    for (int i = 0; i < IPT; ++i) {
      const int slot = (t * BN + wkey + KSTEP * i) & bsm;
      const int64_t bid = __builtin_amdgcn_readfirstlane(blk.k[i]);
      const uint8_t* kr = p.k_cache + bid * p.kc_block_bytes + (int64_t)slot * p.kc_slot_bytes + (int64_t)kvh * p.kc_head_bytes;
      const uint8_t* vr = p.v_cache + bid * p.vc_block_bytes + (int64_t)slot * p.vc_slot_bytes + (int64_t)kvh * p.vc_head_bytes;
#pragma unroll
      for (int j = 0; j < NST; ++j) {
        kst[i][j] = ld16(kr + (j ? koff1 : koff));   // (fp8: one load; 16-bit: the second chunk 16 bytes on, if it exists)
        vst[i][j] = ld16(vr + (j ? voff1 : voff));
      }
    }
  };
  auto issue_loads = [&](int t, const Blk& blk) __attribute__((always_inline)) {
    if constexpr (!PREFIX) issue_paged(t, blk);
    else if (t < ctx_tiles) issue_ctx(t, blk);
    else issue_new(t, std::false_type{});
  };
  // K image: chunk ^= key & 15 (conflict-free ds_read_b128 of 32 keys x one chunk); V image: chunk ^= (key & 3) << 2 | (key & 1)
  // (the four keys of a transposing read land in four different 64-byte bank ranges; the lowest bit is for the writes); context
  // V^T image (PREFIX): rows of 128 bytes = 64 tokens of one d, 16-byte unit ^= (d >> 1) & 7 (16 rows x one unit: every bank once).
  // (the keys of a thread's items are KSTEP apart, a multiple of 16: one pair of swizzled chunk offsets for all)
  uint8_t* k_wr = lds + K_OFF + skey * ROWB;
  uint8_t* v_wr = lds + V_OFF + skey * ROWB;
  auto vswz = [](int key) __attribute__((always_inline)) { return ((key & 3) << 2) | (key & 1); };
  const int kc0 = (ca ^ (skey & 15)) << 4, kc1 = (cb ^ (skey & 15)) << 4;
  const int vc0 = (ca ^ vswz(skey)) << 4, vc1 = (cb ^ vswz(skey)) << 4;
  // PREFIX above head size 128: the offsets of a thread's first chunks (the second ones are at offset ^ CX), computed anew for
  // every tile from a thread id that hipcc cannot trace back.  Kept over the loop they are spilled, and their reloads wait for
  // the loads in flight (us, head 256: 32 x 128 tokens over 4096 16-bit 660 -> 538, fp8 440 -> 377; 2 x 2048 over 2048 fp8
  // 299 -> 290).
  constexpr bool WIDE = PREFIX && D > 128;
  constexpr int CX = PAIR ? 16 : 16 * PPK;
  struct WideAt { int k, v; };
  auto wide_at = [&](bool context) __attribute__((always_inline)) {
    WideAt a = {0, 0};
    if constexpr (WIDE) {
      int t_ = tid;
      asm volatile("" : "+v"(t_));
      const int key = PAIR ? (t_ / 64) * WK + (((t_ >> 2) & 1) | (((t_ & 63) / (2 * PPK)) << 1)) : t_ / PPK;   // (as skey and ca)
      const int chunk = PAIR ? 2 * ((t_ & 3) | (((t_ >> 3) & (PPK / 4 - 1)) << 2)) : t_ % PPK;
      const int kperm = (key & ~12) | ((key & 4) << 1) | ((key & 8) >> 1);   // (below)
      const int kr = context ? kperm : key;
      a.k = K_OFF + kr * ROWB + ((chunk ^ (kr & 15)) << 4);
      a.v = context ? V_OFF + t_ * 128 + (((t_ >> 1) & 7) << 4) : V_OFF + key * ROWB + ((chunk ^ vswz(key)) << 4);
    }
    return a;
  };
  auto u4 = [](u32x4 v) __attribute__((always_inline)) { return make_uint4(v[0], v[1], v[2], v[3]); };
  // Slots past the sequence hold stale bytes (possibly NaN): K and V rows of such keys are zeroed (their scores are 0 + the
  // mask's -inf, their probabilities 0, and 0 * NaN = NaN), and so are the padding columns.  whole: every key of the tile
  // exists and no column is padding, nothing to zero.  conv: the registers hold e4m3.
  auto write_row = [&](uint8_t* row, int c0, int c1, const u32x4 (&st)[NST], bool live, auto whole, auto conv_c) __attribute__((always_inline)) {
    u32x4 x0, x1;
    if constexpr (decltype(conv_c)::value) {
      uint4 lo, hi4;
      widen16<T>(u4(st[0]), lo, hi4);
      x0 = (u32x4){lo.x, lo.y, lo.z, lo.w};
      x1 = (u32x4){hi4.x, hi4.y, hi4.z, hi4.w};
    } else {
      x0 = st[0]; x1 = st[NST - 1];
    }
    if (!whole) {
      if (!live || !pv0) x0 = (u32x4){0, 0, 0, 0};
      if (!live || !pv1) x1 = (u32x4){0, 0, 0, 0};
    }
    *reinterpret_cast<u32x4*>(row + c0) = x0;
    *reinterpret_cast<u32x4*>(row + c1) = x1;
  };
  // rows of keys base + (0..63) of `keys` keys, K and V
  auto write_rows = [&](int t, int base, int keys, auto conv_c, auto whole) __attribute__((always_inline)) {
    const int kb_ = (t & (KN - 1)) * TILE, vb_ = (t & (VN - 1)) * TILE;
    const WideAt at = wide_at(false);
#pragma unroll
    for (int i = 0; i < IPT; ++i) {
      const bool live = base + skey + KSTEP * i < keys;
      if constexpr (WIDE) {
        write_row(lds + at.k + kb_ + KSTEP * i * ROWB, 0, (at.k ^ CX) - at.k, kst[i], live, whole, conv_c);
        write_row(lds + at.v + vb_ + KSTEP * i * ROWB, 0, (at.v ^ CX) - at.v, vst[i], live, whole, conv_c);
      } else {
        write_row(k_wr + kb_ + KSTEP * i * ROWB, kc0, kc1, kst[i], live, whole, conv_c);
        write_row(v_wr + vb_ + KSTEP * i * ROWB, vc0, vc1, vst[i], live, whole, conv_c);
      }
    }
  };
  // Context tiles: LDS row i of K is key i with bits 2 and 3 swapped.  S^T row (r & 3) + 8 (r >> 2) + 4 hi, which lane half hi
  // holds in register r, is then key 16 (r >> 3) + 8 hi + (r & 7): eight keys in a row per register group, so that a fragment
  // of V^T is one 16-byte read (two 8-byte ones before: head 128 2 .. 5 %, head 256 5 .. 23 % slower).
  const int kperm = (skey & ~12) | ((skey & 4) << 1) | ((skey & 8) >> 1);
  uint8_t* k_wr_ctx = lds + K_OFF + kperm * ROWB;
  const int kc0_ctx = (ca ^ (kperm & 15)) << 4, kc1_ctx = (cb ^ (kperm & 15)) << 4;
  auto write_ctx = [&](int t, auto whole) __attribute__((always_inline)) {
    const int kb_ = (t & (KN - 1)) * TILE, vb_ = (t & (VN - 1)) * TILE;
    const WideAt at = wide_at(true);
#pragma unroll
    for (int i = 0; i < IPT; ++i) {
      const bool live = t * BN + skey + KSTEP * i < ctx;
      if constexpr (WIDE) write_row(lds + at.k + kb_ + KSTEP * i * ROWB, 0, (at.k ^ CX) - at.k, kst[i], live, whole, std::integral_constant<bool, FP8>{});
      else write_row(k_wr_ctx + kb_ + KSTEP * i * ROWB, kc0_ctx, kc1_ctx, kst[i], live, whole, std::integral_constant<bool, FP8>{});
      // V^T: the item's 16 tokens of row vd = two 16-byte units
      const int vd = vd_of(i), vq = vq_of(i);
      const int valid = vd < dr ? ctx - (t * BN + 16 * vq) : 0;
      uint4 lo, hi4;
      if constexpr (FP8) {
        uint4 raw = u4(vst[i][0]);
        if (!whole) raw = mask_bytes(raw, valid);
        widen16<T>(raw, lo, hi4);
      } else {
        lo = u4(vst[i][0]);
        hi4 = u4(vst[i][NST - 1]);
        if (!whole) {
          lo = mask_halfs(lo, valid);
          hi4 = mask_halfs(hi4, valid - 8);
        }
      }
      if constexpr (WIDE) {      // (vd is the thread, vq is i)
        *reinterpret_cast<u32x4*>(lds + (at.v ^ (32 * i)) + vb_) = (u32x4){lo.x, lo.y, lo.z, lo.w};
        *reinterpret_cast<u32x4*>(lds + (at.v ^ (32 * i + 16)) + vb_) = (u32x4){hi4.x, hi4.y, hi4.z, hi4.w};
      } else {
        uint8_t* row = lds + V_OFF + vb_ + vd * 128;
        const int f = (vd >> 1) & 7;
        *reinterpret_cast<u32x4*>(row + (((2 * vq + 0) ^ f) << 4)) = (u32x4){lo.x, lo.y, lo.z, lo.w};
        *reinterpret_cast<u32x4*>(row + (((2 * vq + 1) ^ f) << 4)) = (u32x4){hi4.x, hi4.y, hi4.z, hi4.w};
      }
    }
  };
  auto write_tile = [&](int t) __attribute__((always_inline)) {
    if constexpr (!PREFIX) write_rows(t, t * BN, seq_len, std::integral_constant<bool, FP8>{}, false);
    else if (t < ctx_tiles) write_ctx(t, false);
    else write_rows(t, (t - ctx_tiles) * BN, qlen, std::false_type{}, false);
  };

  // ---- fragment read addresses (lane constants; buffer, key block and key group are immediates) ---------
  const uint8_t* k_rd[KS];   // K rows l32 (+ 32 kb), chunk 2 ks + hi
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) k_rd[ks] = lds + K_OFF + l32 * ROWB + (((2 * ks + hi) ^ (l32 & 15)) << 4);
  // transposing read: the 16 lanes of group G = lane >> 4 read keys 4 hi + (0..3) (+ 16 g16 + 8 e) x d
  // 32 db + 16 (G & 1) + (0..15); lane 4 q + pp of the group addresses key q, d 4 pp .. 4 pp + 3 and receives
  // d = 32 db + (lane & 31) of the four keys
  const uint8_t* v_rd[DB];
  {
    const int q = (lane & 15) >> 2, pp = lane & 3, g1 = (lane >> 4) & 1;
#pragma unroll
    for (int db = 0; db < DB; ++db)
      v_rd[db] = lds + V_OFF + (4 * hi + q) * ROWB + ((4 * (db ^ q) + 2 * g1 + ((pp >> 1) ^ (q & 1))) << 4) + 8 * (pp & 1);
  }

  // (D = 256: the same addresses from one offset each, XORed with the k-step / d block / unit at the read)
  const int k_off0 = K_OFF + l32 * ROWB + ((hi ^ (l32 & 15)) << 4);
  const int v_off0 = V_OFF + (4 * hi + ((lane & 15) >> 2)) * ROWB +
                     ((4 * ((lane & 15) >> 2) + 2 * ((lane >> 4) & 1) + (((lane & 3) >> 1) ^ ((lane >> 2) & 1))) << 4) + 8 * (lane & 1);
  // context V^T (PREFIX): row d = 32 db + l32, unit 2 g16 + hi = tokens 16 g16 + 8 hi .. + 7
  int vt_o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) vt_o[i] = V_OFF + l32 * 128 + (((2 * i + hi) ^ ((l32 >> 1) & 7)) << 4);

  float m_run = -INFINITY, l_run = 0.f;
  f32x16 o[DB];   // O^T[d = 32 db + (r & 3) + 8 (r >> 2) + 4 hi][this row]
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[db][r] = 0.f;

  // ---- one K / V tile --------------------------------------------------------------------------------------------
  // A wave's instruction stream is what bounds this kernel (in-kernel stamps, profiles/r03_prefill_fa.txt: with
  // every MFMA removed a tile still took 94 % of its time -- LDS fragment reads a fixed short distance ahead of
  // their use, then the softmax, then the next reads), so the three kinds of work are interleaved inside the
  // wave, and the sched_barriers keep hipcc from undoing it:
  //   * fragment reads run a ring ahead of the MFMAs that consume them (8 K reads, 4 V^T fragments); the K ring is
  //     filled right behind the barrier, IN FRONT of the staging work (LDS writes of tile t + 1, address
  //     arithmetic and loads of tile t + 2), the V^T ring in front of the serial part of the softmax;
  //   * S^T is computed key block by key block, the row maximum of block 0 is taken between the MFMAs of block 1;
  //   * the probabilities of key group g + 1 (exp2, row sum, pack: 7 VALU per MFMA) are computed between the
  //     four PV MFMAs of group g.
  // (all per-tile state is local to this lambda: declared outside the tile loop and assigned under `if (active)`
  // it would be live around the whole loop)
  auto compute = [&](int t, auto masked_c, auto vt_c) __attribute__((always_inline)) {
  constexpr bool MASKED = decltype(masked_c)::value;
  constexpr bool VT = decltype(vt_c)::value;               // a context tile of the PREFIX kernel
  constexpr bool TILE_FP8 = FP8 && (!PREFIX || VT);        // the tile's K / V were e4m3
  const float sct0 = TILE_FP8 ? sc2k : sc2;            // raw score -> log2 domain
  const float sct = SOFTCAP ? 1.f : sct0;                // (soft-capped scores are rewritten in the log2 domain)
  const int bound0 = VT ? bound_ctx - t * BN : bound_new - (t - ctx_tiles) * BN;
  f32x16 s[2];
  u32x4 pb[4];   // P^T fragments of key groups 16 g16 ..: slots 0-3 = keys 4 hi + (0..3), 4-7 = 8 + 4 hi + (0..3) (VT: 8 hi + (0..7))
  u32x4 kf[KR];
  const int kofs = (t & (KN - 1)) * TILE;
  const int vofs = (t & (VN - 1)) * TILE;
  auto k_read = [&](auto ic, int kofs) __attribute__((always_inline)) {
    constexpr int i = decltype(ic)::value;   // read i -> (key block i / KS, k-step i % KS)
    if constexpr (D > 128)   // one base offset, the k-step XORed in (the tile is 1 KiB aligned): 15 registers fewer
      return *reinterpret_cast<const u32x4*>(lds + ((k_off0 ^ ((i % KS) << 5)) + kofs + (i / KS) * 32 * ROWB));
    else
      return *reinterpret_cast<const u32x4*>(k_rd[i % KS] + kofs + (i / KS) * 32 * ROWB);
  };
  static_for<KR>([&](auto ic) { kf[decltype(ic)::value] = k_read(ic, kofs); });
  __builtin_amdgcn_sched_barrier(0);
  float mx = 0.f;   // running maximum of the tile's raw scores in this lane
  {
    static_for<2 * KS>([&](auto ic) {
      constexpr int i = decltype(ic)::value, kb = i / KS, ks = i % KS;
      const u32x4 f = kf[i % KR];
      if constexpr (i + KR < 2 * KS) kf[i % KR] = k_read(std::integral_constant<int, i + KR>{}, kofs);
      if constexpr (ks == 0) {
        // the accumulator starts at 0, or at -inf where the key is invisible to this row: the mask rides in the
        // MFMA's C operand (K rows past the sequence are staged as zeros, so nothing there is NaN or inf)
        f32x16 z;
        const int lim = bound0 - 32 * kb - (VT ? 8 : 4) * hi;
        const int lim_lo = window > 0 ? lim - window + 1 : -(1 << 30);   // sliding window: keys (bound - window, bound]
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int c = VT ? 16 * (r >> 3) + (r & 7) : (r & 3) + 8 * (r >> 2);
          z[r] = (!MASKED || (c <= lim && c >= lim_lo)) ? 0.f : -INFINITY;
        }
        s[kb] = Mma32<T>::mfma(f, qf[0], z);
      } else {
        if (!(abl & 4)) s[kb] = Mma32<T>::mfma(f, qf[ks], s[kb]);
      }
      if constexpr (kb == 1 && ks < 8 && !SOFTCAP) {   // block 0 is complete: its maximum, two scores per MFMA
        if constexpr (ks == 0) mx = max3(s[0][0], s[0][1], s[0][1]);
        else mx = max3(mx, s[0][2 * ks], s[0][2 * ks + 1]);
      }
      __builtin_amdgcn_sched_barrier(0);
    });
  }
  FA_T(2);
  u32x4 vf[VR];
  auto v_read = [&](auto ic, int vofs) __attribute__((always_inline)) {
    constexpr int i = decltype(ic)::value;   // MFMA i -> (key group i / DB, d block i % DB)
    if constexpr (VT) {
      const int oa = D > 128 ? (vt_o[0] ^ ((i / DB) << 5)) : vt_o[i / DB];
      return *reinterpret_cast<const u32x4*>(lds + oa + vofs + 4096 * (i % DB));
    } else {
      const uint8_t* vp = D > 128 ? lds + ((v_off0 ^ ((i % DB) << 6)) + vofs) : v_rd[i % DB] + vofs;
      const u32x2 va = lds_tr16(vp + (16 * (i / DB)) * ROWB);
      const u32x2 vb = lds_tr16(vp + (16 * (i / DB) + 8) * ROWB);
      return (u32x4){va[0], va[1], vb[0], vb[1]};
    }
  };
  {
    static_for<VR>([&](auto ic) { vf[decltype(ic)::value] = v_read(ic, vofs); });
    __builtin_amdgcn_sched_barrier(0);
    // lane holds S^T[key = 64 t + 32 kb + (r & 3) + 8 (r >> 2) + 4 hi][this row] (context tiles: 16 (r >> 3) + 8 hi + (r & 7))
    if constexpr (SOFTCAP) {
      // x = cap2 tanh(y), y = score / softcap, cap2 = softcap log2 e; tanh from one exp2 of -2 |y| and one rcp.  A
      // masked score (-inf) would come out as -cap2: kept at -inf.
      const float cap2 = p.softcap * kLog2e, c1 = sct0 / cap2;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float raw = s[kb][r];
          const float y = raw * c1;
          const float e2 = fast_exp2(-2.0f * kLog2e * fabsf(y));
          const float th = (1.0f - e2) * __builtin_amdgcn_rcpf(1.0f + e2);
          const float x = copysignf(cap2 * th, y);
          s[kb][r] = (MASKED && raw == -INFINITY) ? -INFINITY : x;
        }
      mx = max3(s[0][0], s[0][1], s[0][1]);
#pragma unroll
      for (int r = 2; r < 16; r += 2) mx = max3(mx, s[0][r], s[0][r + 1]);
    }
#pragma unroll
    for (int r = 0; r < 16; r += 2) mx = max3(mx, s[1][r], s[1][r + 1]);
    const float ms = max_xor32(mx) * sct;
    if (__any(ms > m_run + THR)) {
      const float m_new = fmaxf(m_run, ms);
      const float alpha = m_new == -INFINITY ? 1.f : fast_exp2(m_run - m_new);
      m_run = m_new;
      l_run *= alpha;
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[db][r] *= alpha;
    }
    // v_scale rides in the exponent: exp2(s - (m - log2 v_scale)) = p * v_scale
    const float msub = (m_run == -INFINITY ? 0.f : m_run) - (TILE_FP8 ? vlog2 : 0.f);
    float psum = 0.f;
    auto p_word = [&](auto gc, auto jc) __attribute__((always_inline)) {   // word j2 of pb[g16]: two probabilities
      constexpr int g16 = decltype(gc)::value, j2 = decltype(jc)::value, r0 = 8 * (g16 & 1) + 2 * j2;
      float e0 = fmaf(s[g16 >> 1][r0], sct, -msub), e1 = fmaf(s[g16 >> 1][r0 + 1], sct, -msub);
      if (!(abl & 1)) { e0 = fast_exp2(e0); e1 = fast_exp2(e1); }
      psum += e0;
      psum += e1;
      pb[g16][j2] = Mma<T>::pack2(e0, e1);
    };
    static_for<4>([&](auto jc) { p_word(std::integral_constant<int, 0>{}, jc); });
    __builtin_amdgcn_sched_barrier(0);
    // O^T += V^T . P^T
    static_for<4 * DB>([&](auto ic) {
      constexpr int i = decltype(ic)::value, g16 = i / DB, db = i % DB;
      const u32x4 f = vf[i % VR];
      if constexpr (i + VR < 4 * DB) vf[i % VR] = v_read(std::integral_constant<int, i + VR>{}, vofs);
      if (!(abl & 8) || i < 4) o[db] = Mma32<T>::mfma(f, pb[g16], o[db]);
      if constexpr (g16 + 1 < 4 && db < 4) p_word(std::integral_constant<int, g16 + 1>{}, std::integral_constant<int, db>{});
      __builtin_amdgcn_sched_barrier(0);
    });
    l_run += TILE_FP8 ? psum * vinv : psum;   // the sum in units of the unscaled probabilities
  }
  };

  // ---- pipeline ------------------------------------------------------------------------------------------------
  // Registers hold tile t + 1 (loads in flight) while tile t is computed from LDS buffer t & 1; in interval t they
  // are written to buffer (t + 1) & 1 -- last read for tile t - 1, before the barrier that ended interval t - 1 --
  // and the loads of tile t + 2 are issued.  One barrier per tile.
  if (t0 < t1) {
  Blk blk = load_blk(t0);
  issue_loads(t0, blk);
  blk = load_blk(t0 + 1);
  write_tile(t0);
  if (t0 + 1 < t1) issue_loads(t0 + 1, blk);
  blk = load_blk(t0 + 2);
  __syncthreads();
#ifdef VA_PROBES
  last__ = __builtin_readcyclecounter();
#endif
  // A wave's tiles come in three runs: interior tiles (every key visible to every row of the wave), masked
  // tiles (the diagonal and the sequence's last tile), tiles above its rows (staging only).  One loop per run:
  // with both compute copies behind a branch inside one loop hipcc spills 40 registers at the join.
  // STAGGER: the second wave of every SIMD (waves 4-7) does its share of the staging at the TOP of the interval,
  // the first one at the bottom: while one wave converts, writes and computes addresses, its partner is in its
  // MFMA sections (all eight waves in step leave the matrix pipe idle during the staging and collide in it
  // otherwise: in-kernel stamps showed tile time = MFMA time + everything else, no overlap at all).
  const bool stage_first = (p.stagger & 1) && NW == 8 && wave >= NW / 2;   // (one wave per SIMD: nothing to stagger)
  // ("pf_fa_stagger" bits 1 / 2, measurement: a static priority for waves 4-7 / 0-3)
  if ((p.stagger & 2) && wave >= NW / 2) __builtin_amdgcn_s_setprio(1);
  if ((p.stagger & 4) && wave < NW / 2) __builtin_amdgcn_s_setprio(1);
  // FAST: tiles t + 1 and t + 2 exist, are whole and belong to the run's domain: no branch in the staging.  (us with the
  // checks -> without: unified bf16 1 x 8192 521 -> 507, head 256 bf16 4 x 2048 + 2048 1297 -> 1139, fp8 64 x 128 + 4096
  // 1695 -> 1392; context_attention fp8 64 x 128 + 4096 738 -> 653, head 256 2170 instead of 3218: behind the checks hipcc
  // copied the loaded registers at every join, which waited for the loads just issued.)
  auto stage = [&](int t, auto fast_c, auto vt_c) __attribute__((always_inline)) {
    if (abl & 2) return;
    if constexpr (decltype(fast_c)::value) {
      if constexpr (!PREFIX) {
        write_rows(t + 1, 0, 0, std::integral_constant<bool, FP8>{}, std::true_type{});
        issue_paged(t + 2, blk);
      } else if constexpr (decltype(vt_c)::value) {
        write_ctx(t + 1, std::true_type{});
        issue_ctx(t + 2, blk);
      } else {
        write_rows(t + 1, 0, 0, std::false_type{}, std::true_type{});
        issue_new(t + 2, std::true_type{});
      }
    } else {
      if (t + 1 < t1) write_tile(t + 1);
      if (t + 2 < t1) issue_loads(t + 2, blk);
    }
    blk = load_blk(t + 3);
  };
  auto tile_loop = [&](int t_begin, int t_end, auto mode_c, auto vt_c, auto fast_c) __attribute__((always_inline)) {
    constexpr int MODE = decltype(mode_c)::value;
    t_end = min(t_end, t1);
    // (The place of the loop in the instruction cache's lines is worth up to 1.5 %, with the same instructions: one at the front of a line
    // and its successors behind it measured best of eight places.  Left to what stands in front, any change there moves it.)
    [[clang::code_align(64)]] for (int t = max(t_begin, t0); t < t_end; ++t) {
      asm volatile("s_nop 0");
      if (stage_first) stage(t, fast_c, vt_c);
      FA_T(1);
      if constexpr (MODE < 2) {
        compute(t, std::integral_constant<bool, MODE == 1>{}, vt_c);
        FA_T(4);
#ifdef VA_PROBES
        acc__[6] += 1;
#endif
      }
      // (behind the compute the fragment rings are dead: room for the conversion temporaries)
      if (!stage_first) stage(t, fast_c, vt_c);
      FA_T(0);
      __syncthreads();
      FA_T(5);
    }
  };
  constexpr std::integral_constant<int, 0> INTERIOR{};
  constexpr std::integral_constant<int, 1> MASKED_{};
  constexpr std::integral_constant<int, 2> SKIP{};
  // new-domain tiles u = t - ctx_tiles: interior while 64 u + 63 <= w_lo, computed while 64 u <= w_hi
  const int n2 = w_rows ? min(w_hi / BN + 1, new_tiles) : 0;
  const int n1 = w_rows ? min((w_lo + 1) / BN, n2) : 0;
  // interior tiles whose staging has nothing to check (stage()) run in loops of their own: [begin, fast_end), the tiles t with
  // t + 2 below `wholes`, the end of the whole tiles of the domain
  auto fast_end = [&](int begin, int end, int wholes) __attribute__((always_inline)) {
    const int e = min(min(wholes, t1) - 2, end);
    return dr == D && e - max(begin, t0) >= 4 ? e : begin;   // (fewer tiles do not pay for another cold copy of the loop)
  };
  if constexpr (PREFIX) {
    // context: whole tiles are interior, the last one (ctx % 64 tokens) is masked
    const int c2 = w_rows ? ctx_tiles : 0, c1 = w_rows ? ctx / BN : 0, cf = fast_end(0, c1, ctx / BN);
    tile_loop(0, cf, INTERIOR, std::true_type{}, std::true_type{});
    tile_loop(cf, c1, INTERIOR, std::true_type{}, std::false_type{});
    tile_loop(c1, c2, MASKED_, std::true_type{}, std::false_type{});
    tile_loop(c2, ctx_tiles, SKIP, std::true_type{}, std::false_type{});
    const int nf = fast_end(ctx_tiles, ctx_tiles + n1, ctx_tiles + qlen / BN);
    tile_loop(ctx_tiles, nf, INTERIOR, std::false_type{}, std::true_type{});
    tile_loop(nf, ctx_tiles + n1, INTERIOR, std::false_type{}, std::false_type{});
    tile_loop(ctx_tiles + n1, ctx_tiles + n2, MASKED_, std::false_type{}, std::false_type{});
    tile_loop(ctx_tiles + n2, ntiles, SKIP, std::false_type{}, std::false_type{});
  } else {
    // sliding window: tiles wholly left of every row's window are skipped (64 t + 63 <= w_lo - window), tiles that
    // some row sees only in part (64 t <= w_hi - window) are masked
    const int e2 = max(n2, t_start);
    const int l0 = (window > 0 && w_rows) ? max(w_lo - window + 1, 0) / BN : 0;
    const int l1 = (window > 0 && w_rows && w_hi >= window) ? (w_hi - window) / BN + 1 : 0;
    const int b0 = min(max(l0, t_start), e2), b1 = min(max(l1, b0), e2), b2 = min(max(n1, b1), e2);
    const int bf = fast_end(b1, b2, seq_len / BN);
    tile_loop(t_start, b0, SKIP, std::false_type{}, std::false_type{});
    tile_loop(b0, b1, MASKED_, std::false_type{}, std::false_type{});
    tile_loop(b1, bf, INTERIOR, std::false_type{}, std::true_type{});
    tile_loop(bf, b2, INTERIOR, std::false_type{}, std::false_type{});
    tile_loop(b2, e2, MASKED_, std::false_type{}, std::false_type{});
    // (waves without rows, too, with the checks: without them they get in the way of a single wave that has some, 160 tiles of one
    // query token 172 -> 184 us, and pairs gain nothing)
    tile_loop(e2, ntiles, SKIP, std::false_type{}, std::false_type{});
  }
  }   // t0 < t1

#ifdef VA_PROBES
  if (lane == 0 && hw < 2048) {
    acc__[7] = __builtin_readcyclecounter() - t_entry__;
    for (int i = 0; i < 8; ++i) g_fa_stamps[((size_t)hw * 8 + wave) * 8 + i] = acc__[i];
  }
#endif
  // ---- O^T / l -> out ------------------------------------------------------------------------------------------
  if (!rok) return;
  const float l = sum_xor32(l_run);
  if (SPLIT && seg == 0 && live < nseg && hi == 0)
    p.segm_sum[((int64_t)(tok0 + rtok) * p.num_heads + rhead + 1) * nseg - 1] = -(float)live;
  if (SPLIT && live > 1) {   // this segment's partial: O unnormalised, running maximum (log2 domain; -inf: nothing visible), sum
    const int64_t row = ((int64_t)(tok0 + rtok) * p.num_heads + rhead) * nseg + seg;
    if (hi == 0) {
      p.segm_max[row] = m_run;
      p.segm_sum[row] = l;
    }
    float* so = p.segm_out + row * dr + 4 * hi;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int rq = 0; rq < 4; ++rq)
        if (32 * db + 8 * rq + 4 * hi < dr)
          *reinterpret_cast<float4*>(so + 32 * db + 8 * rq) = make_float4(o[db][4 * rq], o[db][4 * rq + 1], o[db][4 * rq + 2], o[db][4 * rq + 3]);
    return;
  }
  const float inv = l > 0.f ? 1.0f / l : 0.f;
  if (p.out_scale == nullptr) {
    T* op = (T*)p.o + (int64_t)(tok0 + rtok) * p.o_stride_t + (int64_t)rhead * p.o_stride_h + 4 * hi;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int rq = 0; rq < 4; ++rq) {
        const u32x2 w = {Mma<T>::pack2(o[db][4 * rq] * inv, o[db][4 * rq + 1] * inv),
                         Mma<T>::pack2(o[db][4 * rq + 2] * inv, o[db][4 * rq + 3] * inv)};
        if (32 * db + 8 * rq + 4 * hi < dr) *reinterpret_cast<u32x2*>(op + 32 * db + 8 * rq) = w;
      }
  } else {
    const float oinv = inv / *p.out_scale;   // acc / l / out_scale, clamped to the e4m3 range (:282-287)
    uint8_t* op = (uint8_t*)p.o + (int64_t)(tok0 + rtok) * p.o_stride_t + (int64_t)rhead * p.o_stride_h + 4 * hi;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int rq = 0; rq < 4; ++rq) {
        float yv[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) yv[r] = fmaxf(-448.0f, fminf(o[db][4 * rq + r] * oinv, 448.0f));
        if (32 * db + 8 * rq + 4 * hi < dr)
          *reinterpret_cast<uint32_t*>(op + 32 * db + 8 * rq) = f32x4_to_fp8x4(yv[0], yv[1], yv[2], yv[3]);
      }
  }
}

template <typename T, bool FP8, bool PREFIX, int D_, int NW_, bool SOFTCAP, bool SPLIT>
__global__ __launch_bounds__(64 * NW_) void fa_fwd_kernel(const FaParams p) {
  __shared__ __attribute__((aligned(1024))) uint8_t lds[fa_lds<D_>()];
  fa_body<T, FP8, PREFIX, D_, NW_, SOFTCAP, SPLIT>(p, lds, blockIdx.x + gridDim.x * blockIdx.y, gridDim.y);
}

}  // namespace fa
}  // namespace va
