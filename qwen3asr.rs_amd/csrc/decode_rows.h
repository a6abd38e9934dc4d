// The paged-attention decode's rows kernel (gfx950), shared by its two
// launch forms: over a work list (decode_kernels.hip) and, for small grids,
// straight over the batch (decode_small_kernels.hip). decode_kernels.hip
// describes the path.
#pragma once

#include <math.h>

#include <type_traits>

#include "vpa_device.h"
#include "vpa_internal.h"

namespace vpa {
namespace {

#ifndef VPA_DECODE_STREAM_LOADS
#define VPA_DECODE_STREAM_LOADS 1
#endif
// K/V tile loads of the decode: every byte is read once per call, so they
// stream (non-temporal) unless VPA_DECODE_STREAM_LOADS is 0.
__device__ __forceinline__ uint4 tile_load(const uint4* p) {
  if constexpr (VPA_DECODE_STREAM_LOADS) return load_stream(p);
  else return *p;
}
// Workgroup barrier for data exchanged through LDS: waits for this wave's LDS
// operations only (outstanding global loads and stores stay in flight).
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}
// v with its 16-bit element e (0..7; uniform) replaced by val, without a
// runtime-indexed array
__device__ __forceinline__ uint4 put_u16(uint4 v, int e, uint32_t val) {
  const uint32_t sh = (uint32_t)(e & 1) * 16u;
  const uint32_t keep = ~(0xffffu << sh), ins = (val & 0xffffu) << sh;
  const int w = e >> 1;
  v.x = w == 0 ? (v.x & keep) | ins : v.x;
  v.y = w == 1 ? (v.y & keep) | ins : v.y;
  v.z = w == 2 ? (v.z & keep) | ins : v.z;
  v.w = w == 3 ? (v.w & keep) | ins : v.w;
  return v;
}
// 16-byte non-temporal store (the fused append's whole sectors)
__device__ __forceinline__ void tile_store(uint4* p, const uint4& v) {
  typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
  __builtin_nontemporal_store(u32x4{v.x, v.y, v.z, v.w}, reinterpret_cast<u32x4*>(p));
}

// Floats per split-K partial row of the rows path: D outputs + a 32-float
// line holding {max, sum}.
template <int D>
constexpr int kPartRow = D + 32;

__device__ __forceinline__ int clamp_context(uint32_t ctx, int max_ctx, int cap) {
  return min((int)min(ctx, (uint32_t)max_ctx), cap);
}

// Grids of at most 64 sequences need no work list: every wave works its
// workgroup's item out from the context lengths, one sequence per lane.
//
// Chunk length: the smallest of 256, 512 and 1024 tokens that leaves at most
// `target` workgroups (one per compute unit), 1024 if none does. One CU pulls
// about 60 KB/us whatever the waves on it, so with few (sequence, kv head)
// pairs a call ends sooner the more CUs share a context; with more workgroups
// than CUs the extra partial rows and uneven CUs cost more than the shorter
// chunks give (16 x 100-1500 tokens: 13.4 us with targets of 256, 13.7 with
// 512; 4 x 3000-4000 14.2 and 15.4). 128-token chunks gain nothing over 256
// (1 x 450 7.7 us, 7.4 whole; 1 x 1500 8.6 and 8.4).
__device__ __forceinline__ int small_chunk_blocks(int nblk_lane, int num_seqs, int num_kv_heads,
                                                  int target, int block_size) {
  const int lane = threadIdx.x & 63;
  int shift = 8 - __builtin_ctz((unsigned)block_size);  // 256 / block_size blocks
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int n = lane < num_seqs ? max(1, (nblk_lane + (1 << shift) - 1) >> shift) : 0;
    if (wave_sum_i32(n) * num_kv_heads <= target) break;
    ++shift;
  }
  return 1 << shift;
}

// Item `want` of the grid: whole chunks of every sequence first, then each
// sequence's last, shorter one by length class (the order of the plan
// kernel's list: longest first). seq < 0 past the last item. An empty context
// is one item.
struct SmallItem {
  int seq, chunk, chunk_blocks;
  uint32_t ctx;
};
template <int BS>
__device__ __forceinline__ SmallItem small_item(const uint32_t* __restrict__ context_lens,
                                                int num_seqs, int max_ctx, int cap_tokens,
                                                int num_kv_heads, int target, uint32_t want) {
  const int lane = threadIdx.x & 63;
  const bool have = lane < num_seqs;
  const uint32_t ctx = have ? context_lens[lane] : 0u;
  const int nblk = (max(clamp_context(ctx, max_ctx, cap_tokens), 0) + BS - 1) / BS;
  SmallItem it;
  it.chunk_blocks = small_chunk_blocks(nblk, num_seqs, num_kv_heads, target, BS);
  const int shift = __builtin_ctz(it.chunk_blocks);
  const int full = nblk >> shift, rest = nblk - (full << shift);
  const int upto = wave_scan_i32(full);  // inclusive
  const int nfull = __builtin_amdgcn_readlane(upto, 63);
  it.seq = -1;
  it.chunk = 0;
  it.ctx = 0;
  int r = (int)want;
  if (r < nfull) {
    it.seq = __builtin_ctzll(__ballot(upto > r));
    it.chunk = r - (__builtin_amdgcn_readlane(upto, it.seq) -
                    __builtin_amdgcn_readlane(full, it.seq));
  } else {
    r -= nfull;
    const bool last = have && (rest > 0 || nblk == 0);
    const int cls = ((it.chunk_blocks - rest) * 8) >> shift;  // 0 (longest) .. 8 (empty)
#pragma unroll
    for (int c = 0; c <= 8; ++c) {
      const uint64_t mask = __ballot(last && cls == c);
      const int n = __builtin_popcountll(mask);
      if (r < n) {
        const int rank = __builtin_amdgcn_mbcnt_hi(
            (uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
        it.seq = __builtin_ctzll(__ballot(last && cls == c && rank == r));
        it.chunk = __builtin_amdgcn_readlane(full, it.seq);
        break;
      }
      r -= n;
    }
    if (it.seq < 0) return it;
  }
  it.ctx = (uint32_t)__builtin_amdgcn_readlane((int)ctx, it.seq);
  return it;
}

#ifndef VPA_DECODE_NV
#define VPA_DECODE_NV 8
#endif
#ifndef VPA_DECODE_FP8_NV
#define VPA_DECODE_FP8_NV 4
#endif
#ifndef VPA_DECODE_ROWS_WAVES_PER_EU
#define VPA_DECODE_ROWS_WAVES_PER_EU 3
#endif

// Workgroup of NW waves = one (sequence, kv head, chunk of NW * PT tokens)
// work unit. Wave w attends over partition w of the chunk (PT tokens); the NW
// partial results are merged in LDS, so HBM partial rows are only written for
// sequences longer than one chunk.
//
// C is the cache element type: T itself, or fp8_t (E4M3FN bytes, 16 per
// vector). With fp8 each 16-byte K or V vector is converted once to two
// vectors of T (exact, v_cvt_scalef32_pk_*_fp8 with scale 1) and the same
// v_dot2 products follow; a lane's q chunk is then 16 dims (two vectors),
// *k_scale is folded into the softmax scale and *v_scale into the output.
// Waves per SIMD the rows kernel is compiled for: instances with many q
// vectors per lane (16-byte vectors: G x chunks per lane, two per chunk for
// fp8) would spill at 3 (with 512-token waves: 16 and more).
#ifndef VPA_DECODE_FP8_WAVES_PER_EU
#define VPA_DECODE_FP8_WAVES_PER_EU VPA_DECODE_ROWS_WAVES_PER_EU
#endif
template <typename C, int D, int BS, int G>
constexpr int rows_waves_per_eu() {
  constexpr bool f8 = sizeof(C) == 1;
  constexpr int qvec = G * (D * BS / ((f8 ? 16 : 8) * 64)) * (f8 ? 2 : 1);
  return qvec >= 16 ? 2 : f8 ? VPA_DECODE_FP8_WAVES_PER_EU : VPA_DECODE_ROWS_WAVES_PER_EU;
}

// Waves per SIMD of a small-grid instance: its workgroups are 8 waves and at
// most one or two of them share a CU, so registers beyond 128 (four waves per
// SIMD) are taken only where the q vectors, or the append over tiles of 6 or
// 8 loads, need them.
template <typename C, int D, int BS, int G, bool kAppend>
constexpr int small_waves_per_eu() {
  constexpr bool f8 = sizeof(C) == 1;
  constexpr int kpl = D * BS / ((f8 ? 16 : 8) * 64);  // loads per tile
  constexpr int qvec = G * kpl * (f8 ? 2 : 1);
  return qvec >= 16 || (kAppend && kpl >= 6) ? 2 : 4;
}

// kAppend (16-bit caches): the launch also appends each sequence's new K/V
// row (new_key / new_value, one token per sequence) at position L - 1 of its
// context, the slot vASR's decode metadata gives the step's token
// (paged_kv_cache.rs:985-1017), in place of a reshape_and_cache launch before
// it. The wave whose partition ends at the context's last block holds that
// block's K and V tiles in registers anyway: it stages the two new rows in
// LDS at its start, puts the token's values into the tiles before using
// them, and writes back whole 32-byte sectors with non-temporal stores: the
// 16 key units of the token with their neighbours (tokens 2i, 2i + 1 share a
// sector), and the whole value tile (every 32-byte value row holds the
// token). No partially written sector reaches HBM.
//
// kSmall: no work list (at most 64 sequences). With small_target 0 every
// context fits one chunk of chunk_blocks blocks and workgroup w serves
// sequence w / kv heads, whose block ids and query are loaded together with
// its context length; otherwise the workgroup works its item out
// (small_item). Wave i of a chunk takes its blocks i, i + NW, ... (not a run
// of them), so the block ids do not depend on the length.
template <typename T, typename C, int D, int BS, int G, int PT, int NW, bool kAppend = false,
          bool kSmall = false>
__global__ __launch_bounds__(64 * NW)
__attribute__((amdgpu_waves_per_eu(kSmall ? small_waves_per_eu<C, D, BS, G, kAppend>()
                                           : rows_waves_per_eu<C, D, BS, G>())))
void paged_decode_rows_kernel(
    T* __restrict__ out, const T* __restrict__ query, const C* __restrict__ key_cache,
    const C* __restrict__ value_cache, const uint32_t* __restrict__ block_tables,
    int32_t block_table_stride, float scale, int32_t num_heads, int32_t num_kv_heads,
    int64_t num_blocks, int64_t block_stride, int64_t head_stride, float* __restrict__ part_out,
    int32_t max_parts, const uint2* __restrict__ items, const uint32_t* __restrict__ queue,
    int32_t num_seqs, int32_t max_ctx, int32_t cap_tokens, const float* __restrict__ k_scale,
    const float* __restrict__ v_scale, const T* __restrict__ new_key,
    const T* __restrict__ new_value, int64_t new_key_stride, int64_t new_value_stride,
    int32_t kv_rep, const uint32_t* __restrict__ context_lens, int32_t chunk_blocks,
    int32_t small_target) {
  constexpr bool kF8 = std::is_same_v<C, fp8_t>;
  static_assert(kF8 || std::is_same_v<C, T>, "cache type is the query type or fp8");
  static_assert(!(kAppend && kF8), "the fused append writes 16-bit caches");
  constexpr int X = pack_x<C>();
  static_assert(X == (kF8 ? 16 : 8), "16-bit or fp8 cache elements only");
  constexpr int PB = PT / BS;        // blocks per wave partition
  // fp8 at 8-token blocks: a 16-byte value vector holds two rows (dims 2r
  // and 2r + 1) of the block's 8 tokens; otherwise VPR vectors make a row.
  constexpr bool kPairRows = kF8 && BS == 8;
  constexpr int VPR = kPairRows ? 1 : BS / X;  // 16-byte vectors per value row
  constexpr int NVV = D * BS / X / 64;          // value vectors per lane per block
  constexpr int NACC = kPairRows ? 2 * NVV : NVV;  // value rows per lane
  constexpr int DSTEP = 64 / VPR;    // row stride between a lane's value vectors
  constexpr int NPL = PT / 64;       // partition tokens per lane in the softmax
  // Stages of NV loads per lane: 8 (8 KiB per wave) for 16-bit caches, 4
  // for fp8, whose stages of 8 hold twice the tokens and twice the
  // conversion and dot-product work between loads (measured: 4 loads per
  // stage 3-5 % faster on fp8 c3 than 8). A K stage reads BKS
  // key tiles: load k of a tile gives lane l vector l + 64k, i.e. token
  // l % BS and 16-byte chunk l / BS + k * (64 / BS), so each instruction
  // reads 1 KiB contiguous and the lane needs only those chunks of q
  // (held in registers); the partial dot products of a token are summed
  // over its 64 / BS lanes with DPP / permlane swaps. A V stage reads BKS
  // value tiles the same way (lane l: row l / (BS/8) + k * 64 / (BS/8),
  // tokens (l % (BS/8)) * 8 .. +7).
  constexpr int KPL = D * BS / (X * 64);  // loads per lane per tile (K or V)
  // 16-byte loads per lane per stage: the whole tiles that fit NV0 loads,
  // at least one tile (head dims 96 and 192 give 3 or 6 loads per tile)
  constexpr int NV0 = kSmall ? 4 : kF8 ? VPA_DECODE_FP8_NV : VPA_DECODE_NV;
  constexpr int NV = KPL >= NV0 ? KPL : (NV0 / KPL) * KPL;
  constexpr int LPT = 64 / BS;            // lanes per token in a key tile
  constexpr int BKS = NV / KPL;           // tiles per stage
  static_assert(KPL == NVV && KPL >= 1 && KPL <= NV && NV % KPL == 0, "stage shape");
  static_assert(VPR >= 1 && VPR <= 4 && PB <= 64 && PT % 64 == 0 && PT >= D, "shape");

  __shared__ float s_logit[NW][G][PT];
  __shared__ __align__(16) uint16_t s_p[NW][G][PT];
  __shared__ float s_m[NW][G], s_l[NW][G];
  constexpr int NR = D / 8;  // 16-byte vectors of a new 16-bit K (or V) row
  __shared__ __align__(16) uint4 s_new[kAppend ? 2 * NR : 1];

  const int lane = threadIdx.x & 63;
  // Uniform where a stage holds at most two tiles: the partition bounds,
  // block ids and tile addresses derived from the wave index then stay in
  // scalar registers (with more tiles per stage their addresses would not
  // fit them and spill).
  const int wave = BKS <= 2 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)
                            : (int)(threadIdx.x >> 6);
  const uint32_t w = blockIdx.x;
  const int j = (int)(w % (uint32_t)num_kv_heads);
  const uint32_t want = w / (uint32_t)num_kv_heads;  // index of this workgroup's item
  constexpr int QV = kF8 ? 2 : 1;  // 16-byte vectors of q per chunk
  uint4 qv[G][KPL][QV];            // this lane's q chunks
  auto load_q = [&](int s) {
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const T* qrow = query + ((int64_t)s * num_heads + j * G + g) * D;
#pragma unroll
      for (int k = 0; k < KPL; ++k)
#pragma unroll
        for (int h2 = 0; h2 < QV; ++h2)
          qv[g][k][h2] =
              *reinterpret_cast<const uint4*>(qrow + (lane / BS + k * LPT) * X + 8 * h2);
    }
  };
  int s, chunk;
  int cshift;          // log2 of the blocks of a chunk, at most PB * NW
  uint32_t ctx;        // the sequence's context length, unclamped
  uint32_t my_bt = 0;  // block ids of the partition (lane b holds its block b)
  if constexpr (kSmall) {
    auto load_bt = [&] {
      const int col = chunk * chunk_blocks + wave + NW * lane;
      if (lane < PB && col < min((chunk + 1) * chunk_blocks, block_table_stride))
        my_bt = block_tables[(int64_t)s * block_table_stride + col];
    };
    if (small_target == 0) {  // every context in one chunk (uniform)
      s = (int)want;
      chunk = 0;
      ctx = context_lens[s];
      load_bt();
      load_q(s);
      // (keeps the compiler from sinking the loads below the exits that follow)
      asm volatile("" ::"s"(ctx), "v"(my_bt));
    } else {
      const SmallItem it = small_item<BS>(context_lens, num_seqs, max_ctx, cap_tokens,
                                          num_kv_heads, small_target, want);
      if (it.seq < 0) return;  // surplus workgroup of the grid
      s = it.seq;
      chunk = it.chunk;
      ctx = it.ctx;
      chunk_blocks = it.chunk_blocks;
      load_bt();
      load_q(s);
    }
  } else {
    // the list holds num_seqs * ceil(max_ctx / 128) >= gridDim.x / num_kv_heads
    // entries, so the item is read together with the header (one round trip;
    // the chunk length comes from there too: as a kernel argument it sat in a
    // cache line of its own and cost 0.2 us per launch)
    const uint32_t chunk_log2 = queue[0], nitems = queue[1];
    const uint2 item = items[want];
    // (the empty asm keeps the compiler from sinking the item load below the
    // count test)
    asm volatile("" ::"s"(nitems), "s"(item.x), "s"(item.y));
    if (want >= nitems) return;  // surplus workgroup of the grid
    s = (int)(item.x >> 16);
    chunk = (int)(item.x & 0xffffu);
    ctx = item.y;
    // a work list built by an earlier call is only trusted within this call's
    // bounds (sequence index, context cap, chunk length), so every access
    // stays in range
    if (s >= num_seqs) return;
    cshift = max((int)min(chunk_log2, (uint32_t)__builtin_ctz(PT * NW)) - __builtin_ctz(BS), 0);
  }
  const int L = clamp_context(ctx, max_ctx, cap_tokens);
  if (L <= 0) {
    if (chunk == 0)
      for (int i = threadIdx.x; i < G * D; i += 64 * NW)
        store_from_f32<T>(out + ((int64_t)s * num_heads + j * G) * D + i, 0.f);
    return;
  }
  if constexpr (kSmall) cshift = __builtin_ctz((unsigned)chunk_blocks);
  const int cblk = 1 << cshift;
  const int nblk = (L + BS - 1) / BS;
  const int nchunks = (nblk + cblk - 1) >> cshift;
  // an item past the sequence's chunks (the grid's surplus; a list built for
  // other lengths or another max_context_len) would write a partial row
  // outside (s, h) or race with chunk 0 on the output: skip it
  if (chunk >= nchunks || (!kSmall && chunk >= max_parts)) return;
  // the chunk's blocks are split evenly over the NW waves (at most PB each),
  // so short sequences keep every wave busy
  const int c_begin = chunk * cblk;
  const int c_nb = min(cblk, nblk - c_begin);
  const int b_begin = kSmall ? c_begin + wave : c_begin + (c_nb * wave) / NW;
  const int nb = kSmall ? (c_nb - wave + NW - 1) / NW  // 0 (or 0.x rounded to it): idle wave
                         : c_begin + (c_nb * (wave + 1)) / NW - b_begin;
  // The partition's tiles in the order they are read: as they lie, or
  // (kSmall) last block first, so that a fused append's stores are under way
  // while the rest is read instead of holding up the kernel's end (28 layers of
  // one 450-token sequence with appends: 251 us against 257). Index in the
  // partition, and block of the sequence, of tile i.
  auto part_block = [&](int i) { return kSmall ? nb - 1 - i : i; };
  auto seq_block = [&](int i) { return b_begin + (kSmall ? NW * (nb - 1 - i) : i); };
  const int app_tile = kSmall ? 0 : nb - 1;  // of the context's last block, where it is here
  // fused append: this wave's partition ends at the context's last block,
  // which holds the new token at offset app_off (a context clamped by
  // max_context_len or the table appends nothing)
  const bool app =
      kAppend && nb > 0 && seq_block(app_tile) == nblk - 1 && ctx == (uint32_t)L;
  const int app_off = (L - 1) % BS;

  float acc[G][NACC];
  float m[G], lsum[G];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    m[g] = -INFINITY;
    lsum[g] = 0.f;
#pragma unroll
    for (int k = 0; k < NACC; ++k) acc[g][k] = 0.f;
  }

  float vs = 1.f;  // value scale of an fp8 cache
  if constexpr (kF8) {
    scale *= *k_scale;
    vs = *v_scale;
  }
  // logits are kept in log2 units (scale * log2 e folded in), so every
  // exponential below is one v_exp_f32; the partial rows' maxima are in the
  // same units for decode_merge_kernel
  scale *= 1.4426950408889634f;

  if (nb > 0) {
    // block ids of the partition and this lane's q chunks
    if constexpr (!kSmall) {
      my_bt = lane < nb ? block_tables[(int64_t)s * block_table_stride + b_begin + lane] : 0u;
      load_q(s);
    }

    // the new K and V rows of head j (the appending wave's lanes 0 .. 2 NR - 1),
    // loaded before the first tiles so that the wait for those covers them
    uint4 nrow = make_uint4(0u, 0u, 0u, 0u);
    if (kAppend && app && lane < 2 * NR)
      nrow = *reinterpret_cast<const uint4*>(
          lane < NR ? new_key + (int64_t)s * new_key_stride + (int64_t)j * D + lane * 8
                    : new_value + (int64_t)s * new_value_stride + (int64_t)j * D +
                          (lane - NR) * 8);

    // j counts kv_rep replicas of every kv head (more query heads per kv
    // head than G): its cache head is j / kv_rep
    const int64_t head_off = (int64_t)(j / kv_rep) * head_stride;
    const uint4* kbase = reinterpret_cast<const uint4*>(key_cache + head_off);
    const uint4* vbase = reinterpret_cast<const uint4*>(value_cache + head_off);
    const int64_t bstride_v = block_stride / X;
    const int t = lane % BS;     // K: token of this lane within a tile
    const int seg = lane % VPR;  // V: 8-token segment of this lane
    const int nks = (((nb + BKS - 1) / BKS) + 1) & ~1;  // stages per pass, rounded up to even
    float* const my_logit = &s_logit[wave][0][0];
    uint16_t* const my_p = &s_p[wave][0][0];

    // Block id of tile u of stage st (uniform); blocks past the partition
    // or out of the pool read block 0 (in bounds) and are masked when
    // consumed, so loads never branch.
    // (the pool check compares 32 bits, in scalar registers, unless the
    // pool holds more than 2^32 blocks)
    const bool huge_pool = num_blocks > (int64_t)0xffffffffu;
    auto tile_block = [&](int st, int u, bool& ok) -> uint32_t {
      const int bi = st * BKS + u;
      const uint32_t phys = (uint32_t)__builtin_amdgcn_readlane((int)my_bt, bi < nb ? part_block(bi) : 0);
      ok = bi < nb && (huge_pool || phys < (uint32_t)num_blocks);
      return ok ? phys : 0u;
    };
    auto load_stage = [&](const uint4* base, int st, uint4(&buf)[NV]) {
#pragma unroll
      for (int u = 0; u < BKS; ++u) {
        // (few tiles per wave: a tile past the partition is not worth a load
        // of block 0)
        if (kSmall && st * BKS + u >= nb) continue;
        bool ok;
        const uint4* tp = base + (int64_t)tile_block(st, u, ok) * bstride_v + lane;
#pragma unroll
        for (int k = 0; k < KPL; ++k) buf[u * KPL + k] = tile_load(tp + 64 * k);
      }
    };
    // logits of BKS tiles
    auto compute_k = [&](int st, const uint4(&buf)[NV]) {
#pragma unroll
      for (int u = 0; u < BKS; ++u) {
        bool ok;
        const uint32_t phys = tile_block(st, u, ok);
        const int bi = st * BKS + u;
        const bool valid = ok && seq_block(bi) * BS + t < L;
        uint4 kt[KPL];
#pragma unroll
        for (int k = 0; k < KPL; ++k) kt[k] = buf[u * KPL + k];
        if constexpr (kAppend) {
          if (app && ok && bi == app_tile) {  // (uniform) the new token's block
            // lane l holds chunk l / BS + k LPT of token t: the token's
            // lanes take the new row's chunks, then the lanes of its 32-byte
            // sectors write them back whole
            if (t == app_off)
#pragma unroll
              for (int k = 0; k < KPL; ++k) kt[k] = s_new[lane / BS + k * LPT];
            if ((t >> 1) == (app_off >> 1)) {
              uint4* dst = const_cast<uint4*>(kbase) + (int64_t)phys * bstride_v + lane;
#pragma unroll
              for (int k = 0; k < KPL; ++k) tile_store(dst + 64 * k, kt[k]);
            }
          }
        }
        float qk[G];
#pragma unroll
        for (int g = 0; g < G; ++g) qk[g] = 0.f;
#pragma unroll
        for (int k = 0; k < KPL; ++k) {
          if constexpr (kF8) {
            uint4 klo, khi;
            fp8x16_to_pk<T>(kt[k], klo, khi);
#pragma unroll
            for (int g = 0; g < G; ++g)
              qk[g] = dot16<T>(qv[g][k][1], khi, dot16<T>(qv[g][k][0], klo, qk[g]));
          } else {
#pragma unroll
            for (int g = 0; g < G; ++g) qk[g] = dot16<T>(qv[g][k][0], kt[k], qk[g]);
          }
        }
#pragma unroll
        for (int g = 0; g < G; ++g) {
          const float r = sum_lanes_mod<BS>(qk[g]);
          if (lane < BS && bi < PB) my_logit[g * PT + bi * BS + lane] = valid ? r * scale : -INFINITY;
        }
      }
    };
    // P.V over BKS tiles
    auto compute_v = [&](int st, const uint4(&buf)[NV]) {
#pragma unroll
      for (int u = 0; u < BKS; ++u) {
        bool ok;
        const uint32_t phys = tile_block(st, u, ok);
        if (!ok) continue;
        const int bi = st * BKS + u;
        uint4 vv[NVV];
#pragma unroll
        for (int k = 0; k < NVV; ++k) vv[k] = buf[u * KPL + k];
        if constexpr (kAppend) {
          if (app && bi == app_tile) {  // (uniform) the new token's block
            // lane l holds rows l / VPR + k DSTEP, tokens seg X .. seg X + X - 1:
            // the lanes of the token's segment put in its values, then the
            // whole tile is written back
            if (seg == app_off / X) {
              const uint16_t* nv = reinterpret_cast<const uint16_t*>(&s_new[NR]);
#pragma unroll
              for (int k = 0; k < NVV; ++k)
                vv[k] = put_u16(vv[k], app_off % X, nv[lane / VPR + k * DSTEP]);
            }
            uint4* dst = const_cast<uint4*>(vbase) + (int64_t)phys * bstride_v + lane;
#pragma unroll
            for (int k = 0; k < NVV; ++k) tile_store(dst + 64 * k, vv[k]);
          }
        }
        if constexpr (kPairRows) {
          // vector k of lane l: rows 2 (l + 64 k) and 2 (l + 64 k) + 1, the
          // block's 8 tokens each, against the block's 8 probabilities
          const int tok0 = seq_block(bi) * BS;
#pragma unroll
          for (int k = 0; k < NVV; ++k) {
            uint4 vh[2];
            fp8x16_to_pk<T>(vv[k], vh[0], vh[1]);
            if (tok0 + BS > L) {  // past the context in the last block: stale values
#pragma unroll
              for (int h2 = 0; h2 < 2; ++h2) {
                union {
                  uint4 v;
                  uint16_t e[8];
                } wv;
                wv.v = vh[h2];
#pragma unroll
                for (int e = 0; e < 8; ++e)
                  if (tok0 + e >= L) wv.e[e] = 0;
                vh[h2] = wv.v;
              }
            }
#pragma unroll
            for (int g = 0; g < G; ++g) {
              const uint4 pk = *reinterpret_cast<const uint4*>(&my_p[g * PT + bi * BS]);
              acc[g][2 * k] = dot16<T>(pk, vh[0], acc[g][2 * k]);
              acc[g][2 * k + 1] = dot16<T>(pk, vh[1], acc[g][2 * k + 1]);
            }
          }
          continue;
        }
        const int tok0 = seq_block(bi) * BS + seg * X;
        if constexpr (kF8) {
#pragma unroll
          for (int k = 0; k < NVV; ++k) {
            uint4 vh[2];
            fp8x16_to_pk<T>(vv[k], vh[0], vh[1]);
            if (tok0 + X > L) {  // past the context in the last block: stale values
#pragma unroll
              for (int h2 = 0; h2 < 2; ++h2) {
                union {
                  uint4 v;
                  uint16_t e[8];
                } wv;
                wv.v = vh[h2];
#pragma unroll
                for (int e = 0; e < 8; ++e)
                  if (tok0 + 8 * h2 + e >= L) wv.e[e] = 0;
                vh[h2] = wv.v;
              }
            }
#pragma unroll
            for (int g = 0; g < G; ++g) {
              const uint4* pp = reinterpret_cast<const uint4*>(&my_p[g * PT + bi * BS + seg * X]);
              acc[g][k] = dot16<T>(pp[1], vh[1], dot16<T>(pp[0], vh[0], acc[g][k]));
            }
          }
          continue;
        }
        if (tok0 + X > L) {
          // past the context in the last block: zero the values (stale contents)
#pragma unroll
          for (int k = 0; k < NVV; ++k) {
            union {
              uint4 v;
              uint16_t e[8];
            } wv;
            wv.v = vv[k];
#pragma unroll
            for (int e = 0; e < X; ++e)
              if (tok0 + e >= L) wv.e[e] = 0;
            vv[k] = wv.v;
          }
        }
#pragma unroll
        for (int g = 0; g < G; ++g) {
          const uint4 pk = *reinterpret_cast<const uint4*>(&my_p[g * PT + bi * BS + seg * X]);
#pragma unroll
          for (int k = 0; k < NVV; ++k) acc[g][k] = dot16<T>(pk, vv[k], acc[g][k]);
        }
      }
    };

    // ---- software pipeline (nks even): the next stage's loads are in
    // flight while the current stage is computed; the first two V stages are
    // issued during the last two K stages, before the softmax ----
    uint4 bufA[NV], bufB[NV];
    load_stage(kbase, 0, bufA);
    load_stage(kbase, 1, bufB);
    if (kAppend && app) {
      if (lane < 2 * NR) s_new[lane] = nrow;
      lds_wave_sync();
    }
    for (int st = 0; st + 2 < nks; st += 2) {
      compute_k(st, bufA);
      load_stage(kbase, st + 2, bufA);
      compute_k(st + 1, bufB);
      load_stage(kbase, st + 3, bufB);
    }
    compute_k(nks - 2, bufA);
    load_stage(vbase, 0, bufA);
    // (the last stage of the even count may have no tile; its logits are not
    // read. Where a wave has few blocks it is a good part of all, and over an
    // fp8 cache, whose tiles are converted first, not worth computing: us per
    // layer, 8 x 154-256 tokens 7.2 -> 6.5, head dim 64 7.6 -> 6.6; the list
    // form 6.7 and 7.5. 16-bit tiles cost no more than the branch does.)
    if (!(kSmall && kF8) || (nks - 1) * BKS < nb) compute_k(nks - 1, bufB);
    load_stage(vbase, 1, bufB);

    // ---- softmax over the partition ----
    lds_wave_sync();
    {
      const int ntok = nb * BS;
#pragma unroll
      for (int g = 0; g < G; ++g) {
        float v[NPL];
        float mx = -INFINITY;
#pragma unroll
        for (int i = 0; i < NPL; ++i) {
          const int idx = i * 64 + lane;
          v[i] = idx < ntok ? my_logit[g * PT + idx] : -INFINITY;
          mx = fmaxf(mx, v[i]);
        }
        mx = wave_max_dpp(mx);
        float sm = 0.f;
#pragma unroll
        for (int i = 0; i < NPL; ++i) {
          if (i * 64 >= ntok) break;  // (uniform) the P.V pass reads only the first ntok
          const float p = v[i] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(v[i] - mx);
          sm += p;
          T pt;
          store_from_f32<T>(&pt, p);
          my_p[g * PT + i * 64 + lane] = pt.x;
        }
        m[g] = mx;
        lsum[g] = wave_sum_dpp(sm);
      }
    }
    lds_wave_sync();

    for (int st = 0; st + 2 < nks; st += 2) {
      compute_v(st, bufA);
      load_stage(vbase, st + 2, bufA);
      compute_v(st + 1, bufB);
      load_stage(vbase, st + 3, bufB);
    }
    compute_v(nks - 2, bufA);
    compute_v(nks - 1, bufB);

    // sum the VPR lanes that hold the same value row
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int k = 0; k < NACC; ++k) {
        if constexpr (VPR >= 2) acc[g][k] += dpp<kDppQuadXor1>(acc[g][k]);
        if constexpr (VPR >= 4) acc[g][k] += dpp<kDppQuadXor2>(acc[g][k]);
        if constexpr (kF8) acc[g][k] *= vs;
      }
  }

  // ---- merge the NW partitions of the chunk in LDS ----
  // Each wave leaves its unnormalised output (in its own s_logit slot, free
  // after the softmax) and its max / sum; then the workgroup combines them.
  // The barriers wait for LDS only: __syncthreads() would also wait for this
  // wave's outstanding global stores (the fused append's sector writes),
  // which nothing here reads.
  lds_barrier();
  {
    float* my_row = &s_logit[wave][0][0];
    if constexpr (kPairRows) {
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int k = 0; k < NACC; ++k) my_row[g * D + 2 * (lane + 64 * (k / 2)) + k % 2] = acc[g][k];
    } else {
      const int row0 = lane / VPR;
      if (lane % VPR == 0) {
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
          for (int k = 0; k < NVV; ++k) my_row[g * D + row0 + k * DSTEP] = acc[g][k];
      }
    }
    if (lane == 0) {
#pragma unroll
      for (int g = 0; g < G; ++g) {
        s_m[wave][g] = m[g];
        s_l[wave][g] = lsum[g];
      }
    }
  }
  lds_barrier();
  // thread e of the workgroup combines output elements e, e + 64*NW, ...
  // (contiguous per head row, so stores write whole lines)
  const bool single = nchunks == 1;
  for (int e = threadIdx.x; e < G * D; e += 64 * NW) {
    const int g = e / D, d = e - (e / D) * D;
    float mx = -INFINITY;
#pragma unroll
    for (int q = 0; q < NW; ++q) mx = fmaxf(mx, s_m[q][g]);
    float num = 0.f, den = 0.f;
#pragma unroll
    for (int q = 0; q < NW; ++q) {
      const float wq = s_m[q][g] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(s_m[q][g] - mx);
      num = fmaf(wq, s_logit[q][0][g * D + d], num);
      den = fmaf(wq, s_l[q][g], den);
    }
    const int h = j * G + g;
    if (single) {
      store_from_f32<T>(out + ((int64_t)s * num_heads + h) * D + d, num / (den + 1e-6f));
    } else {
      // split-K partial row: D floats of unnormalised output, then one
      // 128-byte line {max, sum, 0...} (whole lines: partial-line stores
      // cost a read-modify-write in HBM)
      float* prow = part_out + (((int64_t)s * num_heads + h) * max_parts + chunk) * kPartRow<D>;
      prow[d] = num;
      if (d < 32) prow[D + d] = d == 0 ? mx : (d == 1 ? den : 0.f);
    }
  }
}

// Shapes whose rows kernel takes the fused append: at least 2 KiB of 16-bit
// (block, head) tile, i.e. at most two tiles per 8-load stage (more tiles per
// stage spill scalar registers with the append's extra state).
constexpr bool fused_append_shape(int d, int bs) { return d * bs >= 2048; }

}  // namespace
}  // namespace vpa
