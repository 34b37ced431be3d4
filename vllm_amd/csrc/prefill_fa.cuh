// unified_attention / context_attention_fwd, query chunks of more than one token: the 256-row tile kernel of prefill_fa.hip
// (launched from prefill_attention.hip when fa_plan says so).
#pragma once
#include "common.cuh"

namespace va {

struct FaParams {
  void* o; const void* q;
  const uint8_t* k_cache; const uint8_t* v_cache;        // flash layout [block][slot][kv head][d], any strides (prefix: below)
  const int* block_table; const int* cu_seqlens_q; const int* seq_lens;
  const float* k_scale; const float* v_scale;             // fp8 cache only
  const float* out_scale;                                  // != null: e4m3 output
  int num_heads, num_kv_heads, num_seqs, num_tokens;
  int head_size;       // up to 256 (padded to 128, above 128 to 256, inside the kernel)
  int bs_shift;        // log2(block size)
  int skip_decode;     // sequences of query length 1 were taken by the decode kernel
  int decode_segments = 1;   // > 1: in that many pieces of whole 64-key tiles, which this launch's merge takes along (same stride)
  int tpb = 0;         // tokens per row block (set by launch_unified_fa)
  // (set by launch_unified_fa: what the host knows of the order of the row blocks, so that no workgroup has to find out)
  int halves = 0;      // a half of the workgroup's rows holds whole groups of q heads
  int shares = 0;      // XCDs per head where these may take the row blocks of their head one by one, else 0 (fa_shares)
  int max_k = 0;       // the caller's upper bound of the lengths (read where there is a window)
  int pack;            // q heads per tile-row group: the GQA group (rows = (token, head) pairs) or 1
  int64_t bt_stride, q_stride_t, q_stride_h, o_stride_t, o_stride_h;
  int64_t kc_block_bytes, kc_slot_bytes, kc_head_bytes, vc_block_bytes, vc_slot_bytes, vc_head_bytes;
  float sm_scale;
  float softcap;       // unified_attention: scores softcap * tanh(score / softcap); 0 = none (prefix: 0)
  int window;          // unified_attention: 1 + window_size[0] of the reference call, 0 = none (prefix: 0)
  // context_attention_fwd (prefix = 1): the caches are the paged CONTEXT in the x layout -- K [block][kv head][D / x][BS][x]
  // (x = 16 bytes), V [block][kv head][D][BS]; kc / vc_slot_bytes unused -- and the new tokens' keys / values are dense
  int prefix;
  const void* k_new; const void* v_new;
  int64_t k_stride_t, k_stride_h, v_stride_t, v_stride_h;   // elements
  int blocks_per_seq;  // > 0: num_tokens unknown, grid.x = blocks_per_seq * num_seqs (ceil(max query length / tokens per block))
  int stagger;         // 1 = waves 4-7 stage at the top of the interval (tuning "pf_fa_stagger", default 1)
  // Split over the keys: up to num_segments workgroups per row block, each over its share of the block's tiles; they leave
  // unnormalised fp32 partials [token][q head][segment] that fa_reduce_kernel merges.  1 = no split (buffers unused).
  // seg_slots: workgroups per grid.y to deal out to the row blocks, at least one each.
  int num_segments, seg_slots;
  float* segm_out; float* segm_max; float* segm_sum;
};

// The order in which an unsplit launch takes its row blocks: fa_find (prefill_fa_tile.cuh) carries it out and tells there what each was
// measured to give.  Per grid row (kv head, or head where no group is packed), of which there are gy: `blocks` row blocks of bm rows, of
// `chunks` sequences.
// half blocks from the front and the back of a chunk (decodes: sequences of one token that the same launch takes as decodes)
__host__ __device__ inline bool fa_pairs(int bm, int halves, int gy, int blocks, int decodes, int window) {
  return bm == 256 && halves && window == 0 && (blocks + decodes) * gy <= 256;
}
// every XCD its share of a head's blocks one by one
__host__ __device__ inline bool fa_few(int shares, int gy, int blocks, int chunks, bool pairs, bool over, int window) {
  return shares && !pairs && !over && (blocks * gy > 256 || (chunks == 1 && window == 0));
}
// several chunks, of which not most are short ones over long contexts: the row blocks in the order of their last keys.  The more chunks
// there are, the fewer of an XCD's 32 CUs read the keys of any of them at a time: 32 tpb / chunks query tokens do.  cached: some chunk has a
// context
__host__ __device__ inline bool fa_by_end(int bm, int tpb, int gy, int blocks, int chunks, bool cached) {
  return bm == 128 || (blocks * gy <= 512 ? chunks <= 16 && 4 * chunks <= tpb : blocks * gy <= 2048 && 20 * chunks <= tpb && !cached);
}
// Under a window much shorter than the sequences their row blocks are of one length, and a run of them reads the same keys: in shares
// every XCD would (us, runs / shares, 32 / 4 heads, window 201 of 7000 keys 65 / 77, 16 / 2, 263 of 17800 93 / 104, 91 of 600 39 / 43).  From
// 512 on a block has as much to do as it reads, and in shorter sequences the blocks differ again (16 / 4, window 1257 of 12000 201 / 175,
// 16 / 1, 1362 of 8000 158 / 112, 16 / 2, 425 of 1200 43 / 37; but 16 / 4, 1369 of 6600 105 / 112).
inline int fa_shares(int gy, int window, int max_k) {
  return (gy == 1 || gy == 2 || gy == 4) && (window == 0 || window >= 512 || 5 * (int64_t)window >= max_k) ? 8 / gy : 0;
}

// dtype: VLLM_AMD_F16 / VLLM_AMD_BF16 (queries, output, and the cache unless fp8).  u: the decode tokens beside the chunks, taken
// by the same launch (unified_attention without softcap, window or ALiBi, padded head size 128 for both, u->hp == 1).
int launch_unified_fa(const FaParams& p, int dtype, bool fp8, hipStream_t st, const struct UniDecodeParams* u = nullptr);
// its part for head sizes above 128 (prefill_fa_wide.hip)
void launch_fa_wide(const FaParams& p, int dtype, bool fp8, dim3 grid, hipStream_t st);
// largest num_segments
constexpr int FA_MAX_SEGMENTS = 32;

}  // namespace va
