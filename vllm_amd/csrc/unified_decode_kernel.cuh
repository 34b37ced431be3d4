// The decode kernel of unified_attention as a device function: its own launch is in unified_decode.hip, the one it shares with
// the tile kernel in prefill_fa.hip.  The bandwidth kernel of paged_attention_mfma.hip re-laid for the FLASH cache layout
// [block][slot][kv head][d] of the V1 engine (vllm/attention/ops/triton_unified_attention.py:52-272 for the maths; caller
// vllm/v1/attention/backends/triton_attn.py:297-317).
//
// One workgroup (four waves, eight in a mixed step's launch) per (sequence, kv head[, key segment]) serves the whole GQA group (16 q
// heads of it at a time), so every K / V byte is read once.  Waves stride over steps of 16 KiB of KV (fp8: 64 tokens,
// 16-bit: 32), each with a private online softmax; one merge through LDS at the end.
//
//   K  a token's row is d-contiguous -- the A-operand order of S^T = K Q^T -- but a lane of the
//      MFMA layout is one token, and 16 lanes reading 16 bytes each of 16 different rows cost
//      the L1 sixteen tag look-ups per 256 bytes (measured 4.5 TB/s).  So K is loaded with
//      whole rows per 8 lanes (fp8, head 128: an instruction = 8 contiguous 128-byte rows),
//      written to a wave-private LDS image (XOR-swizzled on the SOURCE side, so the write is
//      the plain lane order) and read back in MFMA order, conflict-free.  The contraction
//      index is permuted to the chunk order (g4 + 4 i) and Q^T is loaded once in the same order.
//   V  rows are [token][d], the PV product O^T += V^T P^T wants 8 TOKENS of one d per lane.  The
//      contraction slots of lane group g4 are tokens 16 ta + 4 g4 + [0,4) and 16 tb + 4 g4 + [0,4)
//      of a tile pair (ta, tb) -- exactly the tokens whose probabilities the lane holds after the
//      softmax (C layout of S^T), so P goes from the softmax into the B operand WITHOUT leaving
//      the registers (no LDS tile, no shuffle).  For each such token the lane loads d = DT c16 ..
//      + DT (8 bytes fp8 / 16 bytes 16-bit at head 128; per instruction 4 whole token rows of one
//      page) and transposes in registers: v_perm_b32 interleaves the bytes of a token pair, the
//      fp8 -> 16-bit widening (exact) then yields the packed (token, token + 1) operand dwords.
//      MFMA j produces rows d = DT i + j (i = A row): a permutation of d undone in the merge.
//   The loop waits for exactly the loads it consumes (K in front of the LDS image, V in front of P V): every load is
//   unconditional, a wave's last step is peeled, block-table entries are scalar loads.  With loads behind branches and
//   block ids through vector loads a step drained everything in flight: whole engine steps (us, fp8, 32q / 8kv) 61 ragged
//   sequences up to 3000 tokens 49.3 -> 39.6, 64 x 4096 90.6 -> 85.5, 16 ragged up to 16384 77.8 -> 65.2; head 64 37.5 -> 24.5.
//   Addresses are a wave-uniform 64-bit base per (tile, row) plus one 32-bit lane offset per
//   operand that never changes (SGPR base + VGPR offset loads); no workgroup barrier in the loop.
#pragma once
#include "unified_decode.cuh"
#include "mma.cuh"

#include <float.h>

namespace va {
namespace {

typedef __attribute__((ext_vector_type(2))) unsigned int u32x2;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;

template <int N> struct DwVec;
template <> struct DwVec<1> { typedef unsigned int type; };
template <> struct DwVec<2> { typedef u32x2 type; };
template <> struct DwVec<4> { typedef u32x4 type; };
template <> struct DwVec<8> { typedef __attribute__((ext_vector_type(8))) unsigned int type; };   // head 256, 16-bit cache
template <int N>
__device__ __forceinline__ unsigned int dw_get(const typename DwVec<N>::type& v, int i) {
  if constexpr (N == 1) return v;
  else return v[i];
}
template <int N>
__device__ __forceinline__ typename DwVec<N>::type nt_load(const uint8_t* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const typename DwVec<N>::type*>(p));
}

// GEN: soft cap, sliding window or ALiBi; without them the scores need no pass of their own, and only a wave's last step a
// mask.
// wg: number out of nwg of the workgroup's (sequence, kv head) pair, seg: its key segment.  PLAIN: longest-first order without
// the pairing of long and short (pa_lpt_wg).
template <bool FP8, int D, int NW>
constexpr int ua_decode_lds() {
  constexpr int k = NW * ((FP8 && D <= 128) ? 4 : 2) * 16 * D * (FP8 ? 1 : 2), merge = NW * 16 * (D + 4) * 4 + NW * 16 * 8;
  return k > merge ? k : merge;
}
template <typename T, bool FP8, int D, int NW, bool GEN, bool PLAIN>
__device__ __forceinline__ void ua_decode_body(const UniDecodeParams& p, char* lds, int sub_shift, int xcd_group, int order, int wg, int nwg, int seg) {
  constexpr int ES = FP8 ? 1 : 2;             // cache element bytes
  constexpr int TILES = (FP8 && D <= 128) ? 4 : 2;   // 16-token tiles per step (the 256-wide form: 32-token steps -- 223 registers, two workgroups per CU)
  constexpr int STEP_TOK = TILES * 16;
  constexpr int KS = TILES / 2;               // k-steps (tile pairs) of the PV product per step
  constexpr int DT = D / 16;                  // PV MFMAs per k-step = d elements a lane owns per token
  constexpr int KL = D * ES / 64;             // K loads per tile and lane (16 B each)
  constexpr int VDW = DT * ES / 4;            // dwords of one token's V row a lane owns
  constexpr int QF = D / 32;                  // k-steps of the QK product
  static_assert(VDW == 1 || VDW == 2 || VDW == 4 || VDW == 8, "");

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c16 = lane & 15, g4 = lane >> 4;
  // Launches of more than one round of workgroups: consecutive hardware ids go to different XCDs
  // (id % 8); remapped so that the kv heads of a sequence -- adjacent 128-byte pieces of the same
  // token rows -- are fetched through ONE XCD's L2 at about the same time (256 x 4096 fp8:
  // 5.6 -> 5.8 TB/s, 512 x 2048: 5.55 -> 5.94; no gain below two rounds of workgroups).
  if (xcd_group && order <= 0) {
    const int q8 = nwg / 8, r8 = nwg % 8, xcd = wg % 8, idx = wg / 8;
    wg = (xcd < r8 ? xcd * (q8 + 1) : r8 * (q8 + 1) + (xcd - r8) * q8) + idx;
  }
  // GQA groups of more than 16 q heads (MQA models) take ceil(G / 16) workgroups per kv head,
  // chunk fastest: the chunks re-read the same K / V, through L2 when they run together
  // hp > 1 (token-major caches): hp ADJACENT kv heads are taken as one row of hp * head_size elements -- one
  // load instruction then fetches 256 contiguous bytes per token instead of 128 (or 64): pieces below 256 bytes cost
  // 10 (128 B) to 40 % (64 B) of the bandwidth, 256-byte pieces nothing (tools/bench_uni_decode_d.py).  The q heads of
  // the hp groups are the columns of ONE Q^T operand, each zero outside its own head's d range, so S^T, the per-column
  // softmax and O^T come out per head with no other change; a column's output is its head's slice of the d rows.
  const int hp = p.hp;
  const int Gq = p.num_heads / p.num_kv_heads;   // q heads per kv head
  const int nkv = p.num_kv_heads / hp;
  const int Gall = Gq * hp;                      // (hp > 1: at most 16)
  const int chunks = (Gall + 15) >> 4;
  // unsplit launches of 257 .. 1024 workgroups: sequences handed out longest first, the two
  // workgroups of a CU paired long + short (pa_lpt_wg, common.cuh; same output bits)
  int lpt_len = -1;
  if (order > 0) {
    const int groups = chunks * nkv;
    const bool xg = xcd_group != 0;
    wg = p.num_seqs <= 64    ? pa_lpt_wg<1, PLAIN>(p.seq_lens, p.num_seqs, groups, order, lane, wg, lpt_len, xg)
         : p.num_seqs <= 256 ? pa_lpt_wg<4, PLAIN>(p.seq_lens, p.num_seqs, groups, order, lane, wg, lpt_len, xg)
         : p.num_seqs <= 512 ? pa_lpt_wg<8, PLAIN>(p.seq_lens, p.num_seqs, groups, order, lane, wg, lpt_len, xg)
                             : pa_lpt_wg<16, PLAIN>(p.seq_lens, p.num_seqs, groups, order, lane, wg, lpt_len, xg);
  }
  const int chunk = wg % chunks, kvh = (wg / chunks) % nkv, seq = wg / (chunks * nkv);
  const int G = min(16, Gall - 16 * chunk);   // q heads of this workgroup
  const int head0 = kvh * Gall + 16 * chunk;
  // D = head size padded to 64 / 128 / 256: chunks at d >= dr are never loaded (zeros: no contribution to
  // the scores, output columns that are never stored)
  const int dsub = p.head_size, dr = dsub * hp;

  // (all three loads before the first branch: one memory round trip, not two)
  const int seq_len = order > 0 ? lpt_len : p.seq_lens[seq];
  const int qtok = p.cu_seqlens_q[seq], qend = p.cu_seqlens_q[seq + 1];
  if (qend - qtok != 1) return;   // not a decode token: the tile kernel's (or nobody's) business
  const int ctx = seq_len - 1;                       // position of the query
  const bool split = p.num_segments > 1;
  const int kv_lo = GEN && p.window > 0 ? max(0, seq_len - p.window) : 0;   // first visible key
  int start_tok = 0, end_tok = seq_len;
  if (split) {
    const int ntiles = (seq_len + 63) >> 6;
    const int tps = (ntiles + p.num_segments - 1) / p.num_segments;
    if (seg * tps >= ntiles) return;                 // the merge does not read this segment
    start_tok = seg * tps * 64;
    end_tok = min(seq_len, start_tok + tps * 64);
  }
  start_tok = max(start_tok, kv_lo & ~(STEP_TOK - 1));
  const int nsteps = end_tok > start_tok ? (end_tok - start_tok + STEP_TOK - 1) / STEP_TOK : 0;
  const int last_page = seq_len > 0 ? (seq_len - 1) >> (4 + sub_shift) : 0;
  const int sub_mask = (1 << sub_shift) - 1;
  // (constant address space: scalar loads.  Through the struct's plain pointer they were vector loads behind vmcnt(0) -- the
  // whole refill -- at the end of every step, since the kernel also stores)
  typedef const __attribute__((address_space(4))) int cint;
  cint* const bt = (cint*)(uintptr_t)(p.block_table + (int64_t)seq * p.bt_stride);

  float kscale = 1.f, vscale = 1.f;
  if constexpr (FP8) { kscale = *p.k_scale; vscale = *p.v_scale; }
  const float sc2 = p.sm_scale * kscale * kLog2e;
  const bool col_ok = c16 < G;
  const bool alibi = GEN && p.alibi_slopes != nullptr;
  const float slope2 = (alibi && col_ok) ? p.alibi_slopes[head0 + c16] * kLog2e : 0.f;
  const float softcap = GEN ? p.softcap : 0.f;
  const float cap_inv = softcap > 0.f ? 1.0f / (kLog2e * softcap) : 0.f, cap2 = softcap * kLog2e;

  constexpr int K_LDS = TILES * 16 * D * ES;   // one step of K per wave
  char* const k_lds = lds + wave * K_LDS;

  // Q^T fragments (B operand of QK) in the K loads' permutation:
  // fp8 : K load i gives d = 16 (g4 + 4 i) + [0,16) -> two k-steps (lo / hi 8); 16 bit: d = 8 (g4 + 4 i) + [0,8)
  uint4 qf[QF];
  {
    const int dlo = hp > 1 && col_ok ? (c16 / Gq) * dsub : 0;   // the column's head starts at row d = dlo
    const T* qp = (const T*)p.q + (int64_t)qtok * p.q_stride_t + (int64_t)(head0 + (col_ok ? c16 : 0)) * p.q_stride_h - dlo;
#pragma unroll
    for (int s = 0; s < QF; ++s) {
      int d;
      if constexpr (FP8) d = 16 * (g4 + 4 * (s >> 1)) + 8 * (s & 1);
      else d = 8 * (g4 + 4 * s);
      const bool ok = col_ok && d >= dlo && d < dlo + dsub;
      const uint4 v = *reinterpret_cast<const uint4*>(qp + (ok ? d : dlo));
      qf[s] = ok ? v : make_uint4(0, 0, 0, 0);
    }
  }

  float m_run = -FLT_MAX, l_run = 0.f;
  f32x4 o[DT];
#pragma unroll
  for (int j = 0; j < DT; ++j) o[j] = (f32x4){0.f, 0.f, 0.f, 0.f};

  typedef typename DwVec<VDW>::type vrow_t;
  u32x4 kreg[TILES * KL];
  vrow_t vreg[TILES * 4];   // [tile][r]: V row piece of token 16 tile + 4 g4 + r
  int pb[TILES];            // block ids of the step whose loads are issued next

  // lane offsets within a tile (bytes, fixed for the whole kernel)
  // K: instruction i of a tile fetches rows i RPI .. + RPI, CPR lanes per row, each lane one
  // 16-byte chunk; the chunk a lane fetches is XOR-swizzled so that the image it writes to LDS
  // (lane order = [row][position]) is read back conflict-free in the MFMA order
  constexpr int RB = D * ES, CPR = RB / 16, RPI = 64 / CPR;   // row bytes, chunks per row, rows per instruction
  auto kswz = [](int row) { return (row * CPR / 16) & (CPR - 1); };
  // (head sizes below the padded D: a lane whose chunk does not exist fetches the row's first one; K is zeroed in front of the
  // LDS image -- its Q^T rows are zero, but 0 * inf is NaN -- and a V column past the head is never stored.  No load sits
  // behind a branch: the compiler then counts the loads in flight and waits for K alone where K is needed, instead of for
  // everything)
  const bool padded = dr < D;
  bool kval[KL];
  uint32_t koff[KL], krd[KL];
#pragma unroll
  for (int i = 0; i < KL; ++i) {
    const int row = i * RPI + lane / CPR;
    const int chunk = (lane % CPR) ^ kswz(row);
    kval[i] = chunk * 16 < dr * ES;
    koff[i] = (uint32_t)(row * p.kc_slot_bytes + (kval[i] ? chunk << 4 : 0));
    krd[i] = (uint32_t)(c16 * RB + (((g4 + 4 * i) ^ kswz(c16)) << 4));
  }
  uint32_t voff[4];   // row r of the lane's four tokens of a tile
#pragma unroll
  for (int r = 0; r < 4; ++r) voff[r] = (uint32_t)((4 * g4 + r) * p.vc_slot_bytes + (c16 * DT < dr ? c16 * (DT * ES) : 0));
  const uint8_t* const k_head = p.k_cache + (int64_t)kvh * hp * p.kc_head_bytes;
  const uint8_t* const v_head = p.v_cache + (int64_t)kvh * hp * p.vc_head_bytes;

  auto load_pb = [&](int step) {   // (past the last step: entries of the last page, not used)
    const int tile0 = (start_tok >> 4) + step * TILES;
#pragma unroll
    for (int t = 0; t < TILES; ++t)
      pb[t] = bt[min((tile0 + t) >> sub_shift, last_page)];
  };
  // (the empty asm keeps the 32-bit offsets from being widened to 64 bits outside the loop,
  // which would turn every load into a 64-bit VGPR address + add instead of SGPR base + offset)
  auto issue_k = [&](int step) {
    const int tile0 = (start_tok >> 4) + step * TILES;
    uint32_t ko[KL];
#pragma unroll
    for (int i = 0; i < KL; ++i) {
      ko[i] = koff[i];
      asm volatile("" : "+v"(ko[i]));
    }
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
      const uint8_t* base = k_head + (int64_t)pb[t] * p.kc_block_bytes +
                            (int64_t)(((tile0 + t) & sub_mask) * 16) * p.kc_slot_bytes;
#pragma unroll
      for (int i = 0; i < KL; ++i) kreg[t * KL + i] = nt_load<4>(base + ko[i]);
    }
  };
  auto issue_v = [&](int step) {
    const int tile0 = (start_tok >> 4) + step * TILES;
    uint32_t vo[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      vo[r] = voff[r];
      asm volatile("" : "+v"(vo[r]));
    }
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
      const uint8_t* base = v_head + (int64_t)pb[t] * p.vc_block_bytes +
                            (int64_t)(((tile0 + t) & sub_mask) * 16) * p.vc_slot_bytes;
#pragma unroll
      for (int r = 0; r < 4; ++r) vreg[t * 4 + r] = nt_load<VDW>(base + vo[r]);
    }
  };

  // MORE: the wave has another step behind this one -- refills unconditionally, and every token of this one exists
  auto do_step = [&](int step, auto more_c) __attribute__((always_inline)) {
    constexpr bool MORE = decltype(more_c)::value;
    const int tok0 = start_tok + step * STEP_TOK;
    const int pf = step + NW;
    // ---------------- K: registers -> wave-private LDS image -> MFMA order ----------------
    if (padded) {
#pragma unroll
      for (int n = 0; n < TILES * KL; ++n) kreg[n] = kval[n % KL] ? kreg[n] : (u32x4)(0);
    }
#pragma unroll
    for (int n = 0; n < TILES * KL; ++n)
      *reinterpret_cast<u32x4*>(k_lds + n * 1024 + lane * 16) = kreg[n];
    if constexpr (MORE) issue_k(pf);
    // ---------------- S^T = K Q^T ----------------------------------------------------
    f32x4 s[TILES];
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < KL; ++i) {
        const u32x4 kr = *reinterpret_cast<const u32x4*>(k_lds + t * 16 * RB + krd[i]);
        const uint4 raw = make_uint4(kr.x, kr.y, kr.z, kr.w);
        if constexpr (FP8) {
          uint4 lo, hi;
          widen16<T>(raw, lo, hi);
          acc = Mma<T>::mfma(lo, qf[2 * i], acc);
          acc = Mma<T>::mfma(hi, qf[2 * i + 1], acc);
        } else {
          acc = Mma<T>::mfma(raw, qf[i], acc);
        }
      }
      s[t] = acc;
    }

    // ---------------- online softmax: lane holds S^T[token tok0 + 16 t + 4 g4 + r][q head c16] -------
    float mx = -FLT_MAX;
#pragma unroll
    for (int t = 0; t < TILES; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        // triton_unified_attention.py:219-238: softcap, causal / padding mask, window, ALiBi
        const int tok = tok0 + 16 * t + 4 * g4 + r;
        float x = s[t][r] * sc2;
        if (GEN && softcap > 0.f) {   // softcap * tanh(S / softcap) from one exp2 (log2 domain throughout)
          const float y = x * cap_inv;
          const float e2 = fast_exp2(-2.0f * kLog2e * fabsf(y));
          x = copysignf(cap2 * (1.0f - e2) * __builtin_amdgcn_rcpf(1.0f + e2), y);
        }
        if constexpr (GEN) x += slope2 * (float)(tok - ctx);
        if constexpr (GEN || !MORE) x = (tok >= kv_lo && tok < end_tok) ? x : -FLT_MAX;
        s[t][r] = x;
        mx = fmaxf(mx, x);
      }
    mx = max_xor32(max_xor16(mx));
    const float m_new = fmaxf(m_run, mx);
    const float alpha = fast_exp2(m_run - m_new);   // first step: exp2(-huge) = 0
    m_run = m_new;
    float psum = 0.f;
    uint32_t pk[TILES][2];   // P rounded to the query dtype: (r0, r1), (r2, r3) of tile t
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
      float e[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int tok = tok0 + 16 * t + 4 * g4 + r;
        e[r] = fast_exp2(s[t][r] - m_new);
        if constexpr (GEN || !MORE) e[r] = (tok >= kv_lo && tok < end_tok) ? e[r] : 0.f;
        psum += e[r];
      }
      pk[t][0] = Mma<T>::pack2(e[0], e[1]);
      pk[t][1] = Mma<T>::pack2(e[2], e[3]);
    }
    l_run = l_run * alpha + psum;
    if (__any(alpha != 1.0f)) {
#pragma unroll
      for (int j = 0; j < DT; ++j) o[j] *= alpha;
    }

    // ---------------- O^T += V^T P^T ----------------------------------------------------
    if (!MORE && tok0 + STEP_TOK > end_tok) {
      // never-written slots past the sequence may hold NaN patterns: 0 * NaN
#pragma unroll
      for (int t = 0; t < TILES; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          vreg[t * 4 + r] &= (vrow_t)(tok0 + 16 * t + 4 * g4 + r < end_tok ? 0xffffffffu : 0u);
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      // contraction slots 0-3 = tile 2 ks, 4-7 = tile 2 ks + 1 (tokens 4 g4 + [0,4) of each)
      const uint4 pfrag = make_uint4(pk[2 * ks][0], pk[2 * ks][1], pk[2 * ks + 1][0], pk[2 * ks + 1][1]);
#pragma unroll
      for (int j = 0; j < DT; ++j) {
        uint32_t a[4];
#pragma unroll
        for (int pr = 0; pr < 4; ++pr) {
          const vrow_t& ta = vreg[8 * ks + 2 * pr];
          const vrow_t& tb = vreg[8 * ks + 2 * pr + 1];
          if constexpr (FP8) {
            // bytes (ta.b, tb.b, ta.b+1, tb.b+1) of the dword that holds element j
            const uint32_t x = __builtin_amdgcn_perm(dw_get<VDW>(tb, j >> 2), dw_get<VDW>(ta, j >> 2),
                                                     (j & 2) ? 0x07030602u : 0x05010400u);
            a[pr] = Mma<T>::cvt2(x, (j & 1) != 0);
          } else {
            a[pr] = __builtin_amdgcn_perm(dw_get<VDW>(tb, j >> 1), dw_get<VDW>(ta, j >> 1),
                                          (j & 1) ? 0x07060302u : 0x05040100u);
          }
        }
        o[j] = Mma<T>::mfma(make_uint4(a[0], a[1], a[2], a[3]), pfrag, o[j]);
      }
    }
    if constexpr (MORE) {
      issue_v(pf);
      load_pb(pf + NW);
    }
  };

  if (wave < nsteps) {
    load_pb(wave);
    issue_k(wave);
    issue_v(wave);
    load_pb(wave + NW);
  }
  // q, older than K and V, is waited for here (behind the join of both paths): pending at the loop's head it would be
  // waited for -- and with it the refill -- in front of the first MFMA of every step
#pragma unroll
  for (int s = 0; s < QF; ++s) asm volatile("" ::"v"(qf[s].x), "v"(qf[s].y), "v"(qf[s].z), "v"(qf[s].w));
  int step = wave;
  for (; step + NW < nsteps; step += NW) do_step(step, std::true_type{});
  if (step < nsteps) do_step(step, std::false_type{});

  // ---------------- merge the NW waves ----------------------------------------------------
  l_run = sum_xor32(sum_xor16(l_run));
  __syncthreads();   // the K images are dead; LDS becomes the merge buffer
  // [NW][16 q heads][D + 4], in 16-byte accesses, the rows 16 bytes further along the banks than a multiple of them (as
  // [NW][D][16] the threads of a row read the same bank).  Unscaled: the reader has every wave's maximum anyway.
  constexpr int OM = D + 4;
  float* om = reinterpret_cast<float*>(lds);
  float* ml = om + NW * 16 * OM;                // [NW][16][2]
  if (g4 == 0) {
    ml[(wave * 16 + c16) * 2 + 0] = m_run;      // (waves with no step: -FLT_MAX, o = 0)
    ml[(wave * 16 + c16) * 2 + 1] = l_run;
  }
  // lane holds O^T[row 4 g4 + r of MFMA j][q head c16] = d = DT (4 g4 + r) + j
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int j = 0; j < DT; j += 4)
      *reinterpret_cast<f32x4*>(om + (wave * 16 + c16) * OM + DT * (4 * g4 + r) + j) = (f32x4){o[j][r], o[j + 1][r], o[j + 2][r], o[j + 3][r]};
  __syncthreads();

  // thread -> (q head qh, 8 consecutive d); head 256: 32 threads per q head, two passes over the 16 heads
  constexpr int TPH = D / 8, HPP = NW * 64 / TPH;
  const int d0 = (threadIdx.x % TPH) * 8;
  if (d0 >= dr) return;
  for (int qh = threadIdx.x / TPH; qh < G; qh += HPP) {
    const int dlo = hp > 1 ? (qh / Gq) * dsub : 0;   // this column's head: rows [dlo, dlo + dsub)
    if (d0 < dlo || d0 >= dlo + dsub) continue;
    float mt = -FLT_MAX;
#pragma unroll
    for (int w = 0; w < NW; ++w) mt = fmaxf(mt, ml[(w * 16 + qh) * 2]);
    float lt = 0.f;
    f32x4 lo = {0.f, 0.f, 0.f, 0.f}, hi = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float f = fast_exp2(ml[(w * 16 + qh) * 2] - mt), fv = f * vscale;
      lt += ml[(w * 16 + qh) * 2 + 1] * f;
      lo += *reinterpret_cast<const f32x4*>(om + (w * 16 + qh) * OM + d0) * fv;
      hi += *reinterpret_cast<const f32x4*>(om + (w * 16 + qh) * OM + d0 + 4) * fv;
    }
    const float acc[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    const int head = head0 + qh;
    if (split) {
      // unnormalised partial (v_scale applied), running max in the log2 domain, sum
      const int64_t row = ((int64_t)qtok * p.num_heads + head) * p.segm_stride + seg;
      float* so = p.segm_out + row * dsub + (d0 - dlo);
      *reinterpret_cast<f32x4*>(so) = (f32x4){acc[0], acc[1], acc[2], acc[3]};
      *reinterpret_cast<f32x4*>(so + 4) = (f32x4){acc[4], acc[5], acc[6], acc[7]};
      if (d0 == dlo) {
        p.segm_max[row] = lt > 0.f ? mt : -INFINITY;
        p.segm_sum[row] = lt;
      }
      continue;
    }
    const float inv = lt > 0.f ? 1.0f / lt : 0.f;   // acc / L (:276); nothing visible gives 0
    if (p.out_scale) {
      const float oi = inv * (1.0f / *p.out_scale);
      uint8_t* op = (uint8_t*)p.out + (int64_t)qtok * p.o_stride_t + (int64_t)head * p.o_stride_h + (d0 - dlo);
      *reinterpret_cast<uint2*>(op) =
          make_uint2(f32x4_to_fp8x4(acc[0] * oi, acc[1] * oi, acc[2] * oi, acc[3] * oi),
                     f32x4_to_fp8x4(acc[4] * oi, acc[5] * oi, acc[6] * oi, acc[7] * oi));
    } else {
      T* op = (T*)p.out + (int64_t)qtok * p.o_stride_t + (int64_t)head * p.o_stride_h + (d0 - dlo);
      *reinterpret_cast<uint4*>(op) =
          make_uint4(Mma<T>::pack2(acc[0] * inv, acc[1] * inv), Mma<T>::pack2(acc[2] * inv, acc[3] * inv),
                     Mma<T>::pack2(acc[4] * inv, acc[5] * inv), Mma<T>::pack2(acc[6] * inv, acc[7] * inv));
    }
  }
}

}  // namespace
}  // namespace va
