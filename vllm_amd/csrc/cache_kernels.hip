// KV-cache writes for the paged cache: reshape_and_cache, reshape_and_cache_flash,
// convert_fp8, copy_blocks.  Pure HBM-bound byte movement (+ e4m3 conversion):
// every thread moves 16-byte vectors on the contiguous side of each layout.
//
// Semantics follow the reference operators cited in include/vllm_amd.h
// (csrc/cache_kernels.cu:210-306, 505-576, 71-170); the kernels themselves are
// written for wave64 / 16-byte accesses and share no structure with them.
#include "common.cuh"

namespace va {


// ---------------------------------------------------------------------------
// reshape_and_cache: K -> [blk, h, d/x, off, x]  V -> [blk, h, d, off]
// One workgroup per token; one thread per x-chunk (x elements = one 16-byte
// cache vector of K).  The K store is a single 16-byte (or x*sizeof) vector,
// the V stores are the layout's inherent element scatter (stride block_size).
// ---------------------------------------------------------------------------
template <typename scalar_t, typename cache_t, bool FP8, int X>
__global__ void reshape_and_cache_kernel(
    const scalar_t* __restrict__ key, const scalar_t* __restrict__ value,
    cache_t* __restrict__ key_cache, cache_t* __restrict__ value_cache,
    const int64_t* __restrict__ slot_mapping, int64_t key_stride,
    int64_t value_stride, int num_heads, int head_size, int block_size,
    const float* __restrict__ k_scale_p, const float* __restrict__ v_scale_p) {
  const int64_t token = blockIdx.x;
  const int64_t slot = slot_mapping[token];
  if (slot < 0) return;
  const int64_t blk = slot / block_size;
  const int64_t off = slot % block_size;
  const int chunks_per_head = head_size / X;
  const int nchunks = num_heads * chunks_per_head;
  Divisor ks(1.f), vs(1.f);
  if constexpr (FP8) { ks = Divisor(*k_scale_p); vs = Divisor(*v_scale_p); }

  const scalar_t* krow = key + token * key_stride;
  const scalar_t* vrow = value + token * value_stride;
  const int64_t blk_elems = (int64_t)num_heads * head_size * block_size;

  for (int c = threadIdx.x; c < nchunks; c += blockDim.x) {
    const int h = c / chunks_per_head;
    const int xc = c % chunks_per_head;
    const int src = h * head_size + xc * X;
    Vec<scalar_t, X> kv = *reinterpret_cast<const Vec<scalar_t, X>*>(krow + src);
    Vec<scalar_t, X> vv = *reinterpret_cast<const Vec<scalar_t, X>*>(vrow + src);
    const int64_t kdst = blk * blk_elems + (int64_t)h * head_size * block_size +
                         (int64_t)xc * block_size * X + off * X;
    const int64_t vdst = blk * blk_elems + (int64_t)h * head_size * block_size +
                         (int64_t)(xc * X) * block_size + off;
    if constexpr (FP8) {
      Vec<uint8_t, X> kq;
      kv_quant_vec(kv, ks, kq);
      *reinterpret_cast<Vec<uint8_t, X>*>(key_cache + kdst) = kq;
#pragma unroll
      for (int j = 0; j < X; ++j)
        value_cache[vdst + (int64_t)j * block_size] = f32_to_fp8(kv_quant_prep(vv.v[j], vs));
    } else {
      *reinterpret_cast<Vec<scalar_t, X>*>(key_cache + kdst) = kv;
#pragma unroll
      for (int j = 0; j < X; ++j) value_cache[vdst + (int64_t)j * block_size] = vv.v[j];
    }
  }
}

// ---------------------------------------------------------------------------
// reshape_and_cache for many tokens.  Prefill and chunked prefill hand over runs of consecutive
// slots; the part of a run inside one 16-slot group of the cache ("segment") is one tile: its V
// is transposed through LDS and every V row [d][16 slots] leaves as 16-byte stores instead of
// single elements, and the K vectors of its tokens are contiguous 256-byte pieces.  A workgroup
// (hpw heads) takes the segments that START among its 16 tokens -- so a run that begins anywhere
// in a block (chunk boundaries do) is cut at the cache's groups and not at multiples of 16
// tokens, and only its two ends are partial tiles, written as 4-byte units and single elements.
// The first segment is blockIdx.z = 0's, a second one blockIdx.z = 1's (in one workgroup behind
// each other 1 .. 3 us more); more (decode batches) are scattered token by token.
// Bound by latency: read and write phases of one round of workgroups (4.2 TB/s at 8192 aligned
// tokens).  us, tiles at multiples of 16 tokens -> at the groups, 8 heads of 128: 8192 tokens from
// slot 11 of a block fp8 20.1 -> 14.9, 16-bit 30.7 -> 14.7 (aligned 15.8 -> 13.8, 15.9 -> 14.9), 24 chunks
// of up to 250 16.8 -> 13.4, 24.4 -> 13.1, 60 chunks of up to 33 9.0 -> 8.8, 9.8 -> 8.5.
// Requires block_size % 16 == 0 and head_size <= 256.
// ---------------------------------------------------------------------------
// (five workgroups per CU: 96 registers, two less than hipcc takes for bf16 -> fp8 by itself)
template <typename scalar_t, typename cache_t, bool FP8>
__global__ __launch_bounds__(256, 5) void reshape_and_cache_runs_kernel(
    const scalar_t* __restrict__ key, const scalar_t* __restrict__ value,
    cache_t* __restrict__ key_cache, cache_t* __restrict__ value_cache,
    const int64_t* __restrict__ slot_mapping, int64_t key_stride, int64_t value_stride,
    int num_tokens, int num_heads, int head_size, int block_size, int bs_log2, int hpw,
    const float* __restrict__ k_scale_p, const float* __restrict__ v_scale_p) {
  constexpr int CS = sizeof(cache_t);
  static_assert(sizeof(scalar_t) == 2 && (CS == 1 || CS == 2), "the transposes are of 1- and 2-byte elements");
  constexpr int X = 16 / CS;    // elements of one K cache vector
  constexpr int G = 16;         // tokens per workgroup, slots per tile
  constexpr int U = 4 / CS;     // elements of a 4-byte unit
  constexpr int W = 512;        // head elements (hpw * head_size <= W) per workgroup
  constexpr int KI = W / X * G / 256, VI = W / 8 * G / 256;   // items per thread
  __shared__ int64_t s_slot[2 * G];
  __shared__ __attribute__((aligned(16))) cache_t vt[G][W + X];   // [slot of the group][head, d], padded rows
  typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;
  const int tid = threadIdx.x, lane = tid & 63;
  // slot -> (block, offset): a shift for the usual power-of-two block sizes (a 64-bit
  // division per item otherwise)
  auto split = [&](int64_t slot, int64_t& blk, int64_t& off) {
    if (bs_log2 >= 0) { blk = slot >> bs_log2; off = slot & (block_size - 1); }
    else { blk = slot / block_size; off = slot % block_size; }
  };
  const int t0 = blockIdx.x * G, h0 = blockIdx.y * hpw;
  const int nh = num_heads - h0 < hpw ? num_heads - h0 : hpw;
  const int width = nh * head_size;   // contiguous source elements per token
  const scalar_t* const kbase = key + h0 * head_size;
  const scalar_t* const vbase = value + h0 * head_size;
  const int64_t blk_elems = (int64_t)num_heads * head_size * block_size;
  const int64_t head_off = (int64_t)h0 * head_size * block_size;

  // every wave: slot of token t0 - 1 + lane (32 lanes); cont: it continues the token in front of it in the same group
  const int tok = t0 - 1 + lane;
  const int64_t sl = lane < 32 && tok >= 0 && tok < num_tokens ? slot_mapping[tok] : -1;
  Divisor ks(1.f), vs(1.f);
  if constexpr (FP8) { ks = Divisor(*k_scale_p); vs = Divisor(*v_scale_p); }
  if (tid >= 1 && tid < 32) s_slot[tid - 1] = sl;
  const int64_t before = __shfl_up((long long)sl, 1, 64);
  const uint32_t cont = (uint32_t)__ballot(lane > 0 && sl >= 0 && before >= 0 && sl == before + 1 && (sl & 15) != 0) >> 1;
  const uint32_t valid = (uint32_t)__ballot(sl >= 0) >> 1;   // bit i: token t0 + i
  uint32_t starts = valid & ~cont & 0xffffu;
  __syncthreads();

  const int cpt = width / X;          // K chunks per token
  const int cpv = width / 8;          // V chunks of 8 per token
  const int cpv_log2 = (cpv & (cpv - 1)) == 0 ? 31 - __clz(cpv) : -1;
  auto vitem = [&](int it, int& i, int& c) {   // item -> (token, chunk), chunk fastest
    if (cpv_log2 >= 0) { i = it >> cpv_log2; c = it & (cpv - 1); }
    else { i = it / cpv; c = it % cpv; }
  };
  // tokens t0 + i0 + [0, 16) of the bits in mask (one segment: its first n)
  struct Rows { Vec<scalar_t, X> k[KI]; Vec<scalar_t, 8> v[VI]; };
  auto load = [&](int i0, uint32_t mask, Rows& r) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < KI; ++u) {      // item = (chunk, token), token fastest
      const int it = tid + 256 * u;
      const int i = it % G, c = it / G;
      const bool ok = c < cpt && ((mask >> i) & 1);
      r.k[u] = *reinterpret_cast<const Vec<scalar_t, X>*>(kbase + (ok ? (int64_t)(t0 + i0 + i) * key_stride + c * X : 0));
    }
#pragma unroll
    for (int u = 0; u < VI; ++u) {
      int i, c;
      vitem(tid + 256 * u, i, c);
      const bool ok = i < G && ((mask >> i) & 1);
      r.v[u] = *reinterpret_cast<const Vec<scalar_t, 8>*>(vbase + (ok ? (int64_t)(t0 + i0 + i) * value_stride + c * 8 : 0));
    }
  };
  // run: a segment; single (i0 = 0, no run): V through LDS, too
  auto store = [&](int i0, uint32_t mask, bool run, bool single, const Rows& r) __attribute__((always_inline)) {
    // K: a wave writes 256-byte pieces of a run (16 tokens x one 16-byte vector)
    const int cph = head_size / X;
#pragma unroll
    for (int u = 0; u < KI; ++u) {
      const int it = tid + 256 * u;
      const int i = it % G, c = it / G;
      if (c >= cpt || !((mask >> i) & 1)) continue;
      int64_t blk, off;
      split(s_slot[i0 + i], blk, off);
      Vec<cache_t, X> kq;
      if constexpr (FP8) {
        kv_quant_vec(r.k[u], ks, kq);
      } else {
        kq = r.k[u];
      }
      const int hl = c / cph, xc = c % cph;
      *reinterpret_cast<Vec<cache_t, X>*>(key_cache + blk * blk_elems + head_off +
                                           ((int64_t)hl * head_size * block_size) +
                                           ((int64_t)xc * block_size + off) * X) = kq;
    }

    // V: into the LDS tile (run, single) or scattered
    const bool tile = run || single;
    const int col0 = run ? (int)(s_slot[i0] & 15) : 0;
#pragma unroll
    for (int u = 0; u < VI; ++u) {
      int i, c;
      vitem(tid + 256 * u, i, c);
      if (i >= G || !((mask >> i) & 1)) continue;
      Vec<cache_t, 8> vq;
      if constexpr (FP8) {
        kv_quant_vec(r.v[u], vs, vq);
      } else {
        vq = r.v[u];
      }
      if (tile) {
        *reinterpret_cast<Vec<cache_t, 8>*>(&vt[col0 + i][c * 8]) = vq;
      } else {
        int64_t blk, off;
        split(s_slot[i0 + i], blk, off);
        cache_t* dst = value_cache + blk * blk_elems + head_off + (int64_t)(c * 8) * block_size + off;
#pragma unroll
        for (int j = 0; j < 8; ++j) dst[(int64_t)j * block_size] = vq.v[j];
      }
    }
    if (!tile) return;
    __syncthreads();
    if (!run) {
      // element by element, a wave along d, four stores at a time
      const int per = (width + 63) / 64, n = G * per;
      for (int it = __builtin_amdgcn_readfirstlane(tid >> 6); it < n; it += 16) {
        cache_t x[4];
        cache_t* dst[4];
        bool ok[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int i = (it + 4 * u) / per, d = 64 * (it + 4 * u - i * per) + lane;
          ok[u] = it + 4 * u < n && ((mask >> i) & 1) && d < width;
          const uint32_t slo = __builtin_amdgcn_readlane((int)sl, i + 1), shi = __builtin_amdgcn_readlane((int)(sl >> 32), i + 1);
          int64_t blk, off;
          split((int64_t)((uint64_t)shi << 32 | slo), blk, off);
          dst[u] = value_cache + blk * blk_elems + head_off + (int64_t)d * block_size + off;
          x[u] = vt[i & 15][d < width ? d : 0];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (ok[u]) *dst[u] = x[u];
      }
      return;
    }

    int64_t blk, off;
    split(s_slot[i0] - col0, blk, off);
    cache_t* const vdst = value_cache + blk * blk_elems + head_off + off;
    // whole tiles, rows of 16 / 32 bytes
    if (mask == 0xffffu) {
      if constexpr (CS == 1) {
        // a thread takes four consecutive d: one 4-byte LDS read per slot, a transpose in registers (reads of single elements made
        // this kernel bound by LDS issue)
        for (int w = tid; w < width / 4; w += 256) {
          uint32_t col[16];
#pragma unroll
          for (int p = 0; p < 16; ++p) col[p] = *reinterpret_cast<const uint32_t*>(&vt[p][w * 4]);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const uint32_t sel = 0x0c0c0000u | ((4u + e) << 8) | (uint32_t)e;   // byte e of (S1, S0)
            u32x4 row;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              const uint32_t x = __builtin_amdgcn_perm(col[4 * k + 1], col[4 * k], sel);
              const uint32_t y = __builtin_amdgcn_perm(col[4 * k + 3], col[4 * k + 2], sel);
              row[k] = __builtin_amdgcn_perm(y, x, 0x05040100u);
            }
            *reinterpret_cast<u32x4*>(vdst + (int64_t)(w * 4 + e) * block_size) = row;
          }
        }
      } else {
        // a lane takes two d and eight slots, and lanes 0, 1 of a quad trade their second row for the first one of lanes 2, 3, so that
        // a store instruction covers 1 KiB in one piece (as 16 bytes a lane, 64 bytes apart, 8192 tokens took 16.6 us, now 14.9, 32768
        // 56.9, now 52.6)
        for (int it = tid; it < width; it += 256) {
          const int w = it >> 1, h = it & 1;
          const bool up = (it & 2) != 0;
          uint32_t col[8];
#pragma unroll
          for (int p = 0; p < 8; ++p) col[p] = *reinterpret_cast<const uint32_t*>(&vt[8 * h + p][2 * w]);
          u32x4 first, second;
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const uint32_t x = __builtin_amdgcn_perm(col[2 * k + 1], col[2 * k], 0x05040100u);   // rows 2 w, 2 w + 1
            const uint32_t y = __builtin_amdgcn_perm(col[2 * k + 1], col[2 * k], 0x07060302u);
            const uint32_t z = __builtin_amdgcn_update_dpp(0, up ? x : y, 0x4e, 0xf, 0xf, true);   // of lane ^ 2
            first[k] = up ? z : x;
            second[k] = up ? y : z;
          }
          cache_t* dst = vdst + (int64_t)(2 * (w & ~1) + (up ? 1 : 0)) * block_size + 8 * h;
          *reinterpret_cast<u32x4*>(dst) = first;
          *reinterpret_cast<u32x4*>(dst + 2 * (int64_t)block_size) = second;
        }
      }
      return;
    }
    // what there is of a tile: a row per thread (four rows a thread left most of the workgroup idle behind a chain of small stores:
    // 300 fp8 tokens from slot 11 6.0 us, now 5.2, 60 chunks of up to 33 9.4, now 8.8)
    const int lo = col0, hi = col0 + __popc(mask);
    for (int d = tid; d < width; d += 256) {
      const int e = d % U;
      cache_t* dst = vdst + (int64_t)d * block_size;
      uint32_t col[16], row[4 * CS];
#pragma unroll
      for (int p = 0; p < 16; ++p) col[p] = *reinterpret_cast<const uint32_t*>(&vt[p][d - e]);
      if constexpr (CS == 1) {
        const uint32_t sel = 0x0c0c0000u | ((4u + e) << 8) | (uint32_t)e;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const uint32_t x = __builtin_amdgcn_perm(col[4 * k + 1], col[4 * k], sel);
          const uint32_t y = __builtin_amdgcn_perm(col[4 * k + 3], col[4 * k + 2], sel);
          row[k] = __builtin_amdgcn_perm(y, x, 0x05040100u);
        }
      } else {
        const uint32_t sel = e ? 0x07060302u : 0x05040100u;
#pragma unroll
        for (int k = 0; k < 8; ++k) row[k] = __builtin_amdgcn_perm(col[2 * k + 1], col[2 * k], sel);
      }
#pragma unroll
      for (int h = 0; h < 2; ++h) {   // (uniform branches)
        if (8 * h >= lo && 8 * h + 8 <= hi) {
          if constexpr (CS == 1) *reinterpret_cast<uint2*>(dst + 8 * h) = make_uint2(row[2 * h], row[2 * h + 1]);
          else *reinterpret_cast<u32x4*>(dst + 8 * h) = (u32x4){row[4 * h], row[4 * h + 1], row[4 * h + 2], row[4 * h + 3]};
          continue;
        }
#pragma unroll
        for (int k = 0; k < 8 / U; ++k) {
          const int q = 8 * h + U * k;
          const uint32_t x = row[q / U];
          if (q >= lo && q + U <= hi) {
            *reinterpret_cast<uint32_t*>(dst + q) = x;
          } else {
#pragma unroll
            for (int j = 0; j < U; ++j)
              if (q + j >= lo && q + j < hi) __builtin_memcpy(dst + q + j, (const char*)&x + j * CS, CS);
          }
        }
      }
    }
  };

  Rows r;
  if (__popc(starts) > 2) {
    // token by token: z = 0 those of the first 16 that are not part of a segment that started in front, z = 1 the rest of the
    // last segment behind them
    const uint32_t tail = cont >> 16;   // bit 0: token t0 + 16 continues token t0 + 15
    const uint32_t mask = blockIdx.z ? (1u << __builtin_ctz(~tail)) - 1u : valid & (0xffffu << __builtin_ctz(starts)) & 0xffffu;
    if (mask == 0) return;
    load(blockIdx.z ? G : 0, mask, r);
    // Slots that hardly ever follow each other (a decode batch) go through LDS: a thread that stores its own eight elements touches a
    // line of the cache per lane and store, a wave along d eight (fp8) or sixteen.  us, by threads -> by waves: fp8 1024 tokens 11.4 ->
    // 9.7, 2048 17.4 -> 13.2, 8192 65.3 -> 43.8, 16-bit 1024 12.5 -> 11.8, 8192 171.5 -> 165; below 512 tokens the longer way costs
    // more (256: fp8 6.2 -> 6.5), and tokens in short runs share the lines that their thread touches.
    store(blockIdx.z ? G : 0, mask, false, blockIdx.z == 0 && num_tokens >= 512 && __popc(starts) > 12, r);
    return;
  }
  if (blockIdx.z) starts &= starts - 1;
  if (starts == 0) return;
  const int i0 = __builtin_ctz(starts);
  const uint32_t mask = (2u << __builtin_ctz(~(cont >> (i0 + 1)))) - 1u;   // at most 16: a group's end is never continued
  load(i0, mask, r);
  store(i0, mask, true, false, r);
}

// Scalar fallback for layouts / alignments the vector kernel does not cover
// (odd x, misaligned rows).  Same mapping as the reference element loop.
template <typename scalar_t, typename cache_t, bool FP8>
__global__ void reshape_and_cache_scalar_kernel(
    const scalar_t* __restrict__ key, const scalar_t* __restrict__ value,
    cache_t* __restrict__ key_cache, cache_t* __restrict__ value_cache,
    const int64_t* __restrict__ slot_mapping, int64_t key_stride,
    int64_t value_stride, int num_heads, int head_size, int block_size, int x,
    const float* __restrict__ k_scale_p, const float* __restrict__ v_scale_p) {
  const int64_t token = blockIdx.x;
  const int64_t slot = slot_mapping[token];
  if (slot < 0) return;
  const int64_t blk = slot / block_size;
  const int64_t off = slot % block_size;
  Divisor ks(1.f), vs(1.f);
  if constexpr (FP8) { ks = Divisor(*k_scale_p); vs = Divisor(*v_scale_p); }
  const int n = num_heads * head_size;
  const int64_t blk_elems = (int64_t)n * block_size;
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    const int h = i / head_size, d = i % head_size;
    const int64_t kdst = blk * blk_elems + (int64_t)h * head_size * block_size +
                         (int64_t)(d / x) * block_size * x + off * x + d % x;
    const int64_t vdst = blk * blk_elems + (int64_t)h * head_size * block_size +
                         (int64_t)d * block_size + off;
    scalar_t k = key[token * key_stride + i];
    scalar_t v = value[token * value_stride + i];
    if constexpr (FP8) {
      key_cache[kdst] = f32_to_fp8(kv_quant_prep(k, ks));
      value_cache[vdst] = f32_to_fp8(kv_quant_prep(v, vs));
    } else {
      key_cache[kdst] = k;
      value_cache[vdst] = v;
    }
  }
}

// ---------------------------------------------------------------------------
// reshape_and_cache_flash: K,V -> [blk, off, h, d] through explicit strides.
// One thread per VEC contiguous head elements: both sides are 16-byte vectors.
// ---------------------------------------------------------------------------
template <typename scalar_t, typename cache_t, bool FP8, int VEC>
__global__ void reshape_and_cache_flash_kernel(
    const scalar_t* __restrict__ key, const scalar_t* __restrict__ value,
    cache_t* __restrict__ key_cache, cache_t* __restrict__ value_cache,
    const int64_t* __restrict__ slot_mapping, int64_t block_stride,
    int64_t page_stride, int64_t head_stride, int64_t key_stride,
    int64_t value_stride, int num_heads, int head_size, int block_size,
    const float* __restrict__ k_scale_p, const float* __restrict__ v_scale_p) {
  const int64_t token = blockIdx.x;
  const int64_t slot = slot_mapping[token];
  if (slot < 0) return;
  const int64_t blk = slot / block_size;
  const int64_t off = slot % block_size;
  Divisor ks(1.f), vs(1.f);
  if constexpr (FP8) { ks = Divisor(*k_scale_p); vs = Divisor(*v_scale_p); }
  const int vec_per_head = head_size / VEC;
  const int nvec = num_heads * vec_per_head;
  const scalar_t* krow = key + token * key_stride;
  const scalar_t* vrow = value + token * value_stride;
  for (int c = threadIdx.x; c < nvec; c += blockDim.x) {
    const int h = c / vec_per_head;
    const int d = (c % vec_per_head) * VEC;
    const int src = h * head_size + d;
    const int64_t dst = blk * block_stride + off * page_stride + h * head_stride + d;
    Vec<scalar_t, VEC> kv = *reinterpret_cast<const Vec<scalar_t, VEC>*>(krow + src);
    Vec<scalar_t, VEC> vv = *reinterpret_cast<const Vec<scalar_t, VEC>*>(vrow + src);
    if constexpr (FP8) {
      Vec<uint8_t, VEC> kq, vq;
      kv_quant_vec(kv, ks, kq);
      kv_quant_vec(vv, vs, vq);
      *reinterpret_cast<Vec<uint8_t, VEC>*>(key_cache + dst) = kq;
      *reinterpret_cast<Vec<uint8_t, VEC>*>(value_cache + dst) = vq;
    } else {
      *reinterpret_cast<Vec<scalar_t, VEC>*>(key_cache + dst) = kv;
      *reinterpret_cast<Vec<scalar_t, VEC>*>(value_cache + dst) = vv;
    }
  }
}

// ---------------------------------------------------------------------------
// convert_fp8 (test helper in the reference, also used to build fp8 caches)
// ---------------------------------------------------------------------------
template <typename scalar_t, bool TO_FP8>
__global__ void convert_fp8_kernel(void* __restrict__ dst_, const void* __restrict__ src_,
                                   int64_t n, float scale) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  const Divisor dv(scale);
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    if constexpr (TO_FP8) {
      const scalar_t* src = (const scalar_t*)src_;
      ((uint8_t*)dst_)[i] = f32_to_fp8(kv_quant_prep(src[i], dv));
    } else {
      const uint8_t* src = (const uint8_t*)src_;
      ((scalar_t*)dst_)[i] = from_f32<scalar_t>(fp8_to_f32(src[i]) * scale);
    }
  }
}

// ---------------------------------------------------------------------------
// copy_blocks: grid (pair, 2 {K,V}); 16-byte vectors
// ---------------------------------------------------------------------------
__global__ void copy_blocks_kernel(uint8_t* __restrict__ kc, uint8_t* __restrict__ vc,
                                   const int64_t* __restrict__ mapping, int64_t block_bytes) {
  const int64_t src = mapping[2 * blockIdx.x];
  const int64_t dst = mapping[2 * blockIdx.x + 1];
  uint8_t* base = blockIdx.y == 0 ? kc : vc;
  const uint8_t* s = base + src * block_bytes;
  uint8_t* d = base + dst * block_bytes;
  if ((block_bytes & 15) == 0 && (((uintptr_t)base) & 15) == 0) {
    const int64_t nv = block_bytes >> 4;
    for (int64_t i = threadIdx.x; i < nv; i += blockDim.x)
      reinterpret_cast<uint4*>(d)[i] = reinterpret_cast<const uint4*>(s)[i];
  } else {
    for (int64_t i = threadIdx.x; i < block_bytes; i += blockDim.x) d[i] = s[i];
  }
}

}  // namespace va

using namespace va;

namespace va { int g_cache_runs = 1; int g_cache_hpw = 0; }   // "cache_hpw": heads per workgroup of the runs kernel (0 = heuristic)   // tuning "cache_runs": 0 = always the per-token kernel

static inline bool aligned(const void* p, size_t a) { return (((uintptr_t)p) & (a - 1)) == 0; }

template <typename scalar_t, bool FP8>
static int launch_reshape_and_cache(const void* key, const void* value, void* kc, void* vc,
                                    const int64_t* slot_mapping, int num_tokens, int num_heads,
                                    int head_size, int block_size, int x, int64_t key_stride,
                                    int64_t value_stride, const float* ks, const float* vs,
                                    hipStream_t st) {
  typedef typename std::conditional<FP8, uint8_t, scalar_t>::type cache_t;
  constexpr int XN = FP8 ? 16 : 16 / (int)sizeof(scalar_t);  // natural x
  const bool vec_ok = (x == XN) && (head_size % x == 0) &&
                      (key_stride % x == 0) && (value_stride % x == 0) &&
                      aligned(key, sizeof(scalar_t) * XN) && aligned(value, sizeof(scalar_t) * XN) &&
                      aligned(kc, 16);
  // many tokens: the run-aware kernel
  if constexpr (sizeof(scalar_t) == 2) {
    if (vec_ok && num_tokens >= 256 && block_size % 16 == 0 && head_size % 8 == 0 && head_size <= 256 && aligned(vc, 16) && g_cache_runs) {
      int bs_log2 = -1;
      for (int i = 4; i < 16; ++i) if (block_size == (1 << i)) bs_log2 = i;
      int hpw = 512 / head_size;   // heads per workgroup: hpw * head_size <= 512 elements
      if (hpw > num_heads) hpw = num_heads;
      // fewer heads per workgroup while the launch would not fill the chip a few times over
      // (8192 tokens 19.8 us with 1 head per workgroup, 14.3 with 4; 2048 tokens 6.8 / 6.2
      // with 1 / 2: tools/bench_cache_hpw.py)
      while (hpw > 1 && (int64_t)((num_tokens + 15) / 16) * ((num_heads + hpw - 1) / hpw) < 512) hpw /= 2;
      if (g_cache_hpw > 0 && g_cache_hpw * head_size <= 512 && g_cache_hpw <= num_heads) hpw = g_cache_hpw;
      hipLaunchKernelGGL((reshape_and_cache_runs_kernel<scalar_t, cache_t, FP8>),
                         dim3((num_tokens + 15) / 16, (num_heads + hpw - 1) / hpw, 2), dim3(256), 0, st,
                         (const scalar_t*)key, (const scalar_t*)value, (cache_t*)kc, (cache_t*)vc,
                         slot_mapping, key_stride, value_stride, num_tokens, num_heads, head_size,
                         block_size, bs_log2, hpw, ks, vs);
      VA_LAUNCH_CHECK("reshape_and_cache launch");
      return VLLM_AMD_OK;
    }
  }
  if (vec_ok) {
    const int nchunks = num_heads * head_size / x;
    int threads = nchunks < 256 ? ((nchunks + 63) / 64) * 64 : 256;
    hipLaunchKernelGGL((reshape_and_cache_kernel<scalar_t, cache_t, FP8, XN>), dim3(num_tokens),
                       dim3(threads), 0, st, (const scalar_t*)key, (const scalar_t*)value,
                       (cache_t*)kc, (cache_t*)vc, slot_mapping, key_stride, value_stride,
                       num_heads, head_size, block_size, ks, vs);
  } else {
    int n = num_heads * head_size;
    int threads = n < 512 ? ((n + 63) / 64) * 64 : 512;
    hipLaunchKernelGGL((reshape_and_cache_scalar_kernel<scalar_t, cache_t, FP8>),
                       dim3(num_tokens), dim3(threads), 0, st, (const scalar_t*)key,
                       (const scalar_t*)value, (cache_t*)kc, (cache_t*)vc, slot_mapping,
                       key_stride, value_stride, num_heads, head_size, block_size, x, ks, vs);
  }
  VA_LAUNCH_CHECK("reshape_and_cache launch");
  return VLLM_AMD_OK;
}

extern "C" int vllm_amd_reshape_and_cache(
    const void* key, const void* value, void* key_cache, void* value_cache,
    const int64_t* slot_mapping, int num_tokens, int num_heads, int head_size, int block_size,
    int x, int64_t key_stride, int64_t value_stride, int dtype, int kv_dtype,
    const float* k_scale, const float* v_scale, void* stream) {
  VA_REQUIRE(num_tokens >= 0 && num_heads > 0 && head_size > 0 && block_size > 0 && x > 0,
             VLLM_AMD_EINVAL, "reshape_and_cache: bad shape");
  VA_REQUIRE(head_size % x == 0, VLLM_AMD_EINVAL,
             "reshape_and_cache: head_size %d not divisible by x %d", head_size, x);
  if (num_tokens == 0) return VLLM_AMD_OK;
  VA_REQUIRE(key && value && key_cache && value_cache && slot_mapping, VLLM_AMD_EINVAL,
             "reshape_and_cache: null pointer");
  hipStream_t st = (hipStream_t)stream;
#define RC(T, F) \
  return launch_reshape_and_cache<T, F>(key, value, key_cache, value_cache, slot_mapping, \
      num_tokens, num_heads, head_size, block_size, x, key_stride, value_stride, k_scale, v_scale, st)
  if (kv_dtype == VLLM_AMD_KV_AUTO) {
    if (dtype == VLLM_AMD_F32) RC(float, false);
    if (dtype == VLLM_AMD_F16) RC(f16_t, false);
    if (dtype == VLLM_AMD_BF16) RC(bf16_t, false);
    VA_REQUIRE(false, VLLM_AMD_EUNSUPPORTED, "Unsupported input type of kv cache: %d", dtype);
  } else if (kv_dtype == VLLM_AMD_KV_FP8_E4M3) {
    VA_REQUIRE(k_scale && v_scale, VLLM_AMD_EINVAL, "reshape_and_cache: null scale");
    if (dtype == VLLM_AMD_F32) RC(float, true);
    if (dtype == VLLM_AMD_F16) RC(f16_t, true);
    if (dtype == VLLM_AMD_BF16) RC(bf16_t, true);
    VA_REQUIRE(false, VLLM_AMD_EUNSUPPORTED, "Unsupported input type of kv cache: %d", dtype);
  }
#undef RC
  VA_REQUIRE(false, VLLM_AMD_EUNSUPPORTED, "Unsupported data type of kv cache: %d", kv_dtype);
}

template <typename scalar_t, bool FP8>
static int launch_flash(const void* key, const void* value, void* kc, void* vc,
                        const int64_t* slot_mapping, int num_tokens, int num_heads, int head_size,
                        int block_size, int64_t key_stride, int64_t value_stride,
                        int64_t block_stride, int64_t page_stride, int64_t head_stride,
                        const float* ks, const float* vs, hipStream_t st) {
  typedef typename std::conditional<FP8, uint8_t, scalar_t>::type cache_t;
  constexpr int V = 16 / (int)sizeof(scalar_t);  // 16-byte source vectors (4 or 8 elements)
  const size_t cvb = V * sizeof(cache_t);       // bytes of one cache vector
  const bool vec_ok = head_size % V == 0 && key_stride % V == 0 && value_stride % V == 0 &&
                      block_stride % V == 0 && page_stride % V == 0 && head_stride % V == 0 &&
                      aligned(key, 16) && aligned(value, 16) && aligned(kc, cvb) &&
                      aligned(vc, cvb);
#define FL(VEC)                                                                               \
  do {                                                                                        \
    const int nvec = num_heads * head_size / VEC;                                             \
    int threads = nvec < 256 ? ((nvec + 63) / 64) * 64 : 256;                                 \
    hipLaunchKernelGGL((reshape_and_cache_flash_kernel<scalar_t, cache_t, FP8, VEC>),         \
                       dim3(num_tokens), dim3(threads), 0, st, (const scalar_t*)key,          \
                       (const scalar_t*)value, (cache_t*)kc, (cache_t*)vc, slot_mapping,      \
                       block_stride, page_stride, head_stride, key_stride, value_stride,      \
                       num_heads, head_size, block_size, ks, vs);                             \
  } while (0)
  if (vec_ok) FL(V); else FL(1);
#undef FL
  VA_LAUNCH_CHECK("reshape_and_cache_flash launch");
  return VLLM_AMD_OK;
}

extern "C" int vllm_amd_reshape_and_cache_flash(
    const void* key, const void* value, void* key_cache, void* value_cache,
    const int64_t* slot_mapping, int num_tokens, int num_heads, int head_size, int block_size,
    int64_t key_stride, int64_t value_stride, int64_t block_stride, int64_t page_stride,
    int64_t head_stride, int dtype, int kv_dtype, const float* k_scale, const float* v_scale,
    void* stream) {
  VA_REQUIRE(num_tokens >= 0 && num_heads > 0 && head_size > 0 && block_size > 0,
             VLLM_AMD_EINVAL, "reshape_and_cache_flash: bad shape");
  if (num_tokens == 0) return VLLM_AMD_OK;
  VA_REQUIRE(key && value && key_cache && value_cache && slot_mapping, VLLM_AMD_EINVAL,
             "reshape_and_cache_flash: null pointer");
  hipStream_t st = (hipStream_t)stream;
#define RF(T, F) \
  return launch_flash<T, F>(key, value, key_cache, value_cache, slot_mapping, num_tokens, \
      num_heads, head_size, block_size, key_stride, value_stride, block_stride, page_stride, \
      head_stride, k_scale, v_scale, st)
  if (kv_dtype == VLLM_AMD_KV_AUTO) {
    if (dtype == VLLM_AMD_F32) RF(float, false);
    if (dtype == VLLM_AMD_F16) RF(f16_t, false);
    if (dtype == VLLM_AMD_BF16) RF(bf16_t, false);
    VA_REQUIRE(false, VLLM_AMD_EUNSUPPORTED, "Unsupported input type of kv cache: %d", dtype);
  } else if (kv_dtype == VLLM_AMD_KV_FP8_E4M3) {
    VA_REQUIRE(k_scale && v_scale, VLLM_AMD_EINVAL, "reshape_and_cache_flash: null scale");
    if (dtype == VLLM_AMD_F32) RF(float, true);
    if (dtype == VLLM_AMD_F16) RF(f16_t, true);
    if (dtype == VLLM_AMD_BF16) RF(bf16_t, true);
    VA_REQUIRE(false, VLLM_AMD_EUNSUPPORTED, "Unsupported input type of kv cache: %d", dtype);
  }
#undef RF
  VA_REQUIRE(false, VLLM_AMD_EUNSUPPORTED, "Unsupported data type of kv cache: %d", kv_dtype);
}

extern "C" int vllm_amd_convert_fp8(void* dst, const void* src, int64_t n, float scale, int dtype,
                                    int to_fp8, void* stream) {
  VA_REQUIRE(n >= 0, VLLM_AMD_EINVAL, "convert_fp8: negative size");
  if (n == 0) return VLLM_AMD_OK;
  VA_REQUIRE(dst && src, VLLM_AMD_EINVAL, "convert_fp8: null pointer");
  hipStream_t st = (hipStream_t)stream;
  int64_t blocks = (n + 255) / 256;
  if (blocks > 256 * 16) blocks = 256 * 16;
#define CV(T)                                                                                 \
  do {                                                                                        \
    if (to_fp8)                                                                               \
      hipLaunchKernelGGL((convert_fp8_kernel<T, true>), dim3((unsigned)blocks), dim3(256), 0, \
                         st, dst, src, n, scale);                                             \
    else                                                                                      \
      hipLaunchKernelGGL((convert_fp8_kernel<T, false>), dim3((unsigned)blocks), dim3(256), 0, \
                         st, dst, src, n, scale);                                             \
  } while (0)
  if (dtype == VLLM_AMD_F32) CV(float);
  else if (dtype == VLLM_AMD_F16) CV(f16_t);
  else if (dtype == VLLM_AMD_BF16) CV(bf16_t);
  else VA_REQUIRE(false, VLLM_AMD_EUNSUPPORTED, "Unsupported data type: %d", dtype);
#undef CV
  VA_LAUNCH_CHECK("convert_fp8 launch");
  return VLLM_AMD_OK;
}

extern "C" int vllm_amd_copy_blocks(void* key_cache, void* value_cache,
                                    const int64_t* block_mapping, int num_pairs,
                                    int64_t block_bytes, void* stream) {
  VA_REQUIRE(num_pairs >= 0 && block_bytes > 0, VLLM_AMD_EINVAL, "copy_blocks: bad shape");
  if (num_pairs == 0) return VLLM_AMD_OK;
  VA_REQUIRE(key_cache && value_cache && block_mapping, VLLM_AMD_EINVAL,
             "copy_blocks: null pointer");
  hipLaunchKernelGGL(copy_blocks_kernel, dim3(num_pairs, 2), dim3(256), 0, (hipStream_t)stream,
                     (uint8_t*)key_cache, (uint8_t*)value_cache, block_mapping, block_bytes);
  VA_LAUNCH_CHECK("copy_blocks launch");
  return VLLM_AMD_OK;
}
