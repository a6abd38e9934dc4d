// Chunked prefill of few rows on the 16-bit MFMA kernel (prefill_paged.h,
// kSplit): the four waves of a workgroup split one 32-row tile's keys. One
// long request's chunk (512 tokens, 64 tiles of 128 rows) left three quarters
// of the CUs idle and each of the others a serial run over every key. What
// bounds it then is a step of four tiles on one workgroup per CU (128 KiB of
// LDS): its DMAs from L2 and one wave per SIMD's chain of MFMAs and softmax.
#include "prefill_paged.h"
#include "vpa_device.h"
#include "vpa_internal.h"

namespace vpa {
namespace {

template <typename T, typename C, int BS>
hipError_t split_group(int group, const PrefillArgs& a, const CacheGeom& g, hipStream_t stream) {
  switch (group) {
    case 1:
      return launch_prefill_s<T, C, 128, BS, 1, true>(a, g, stream);
    case 2:
      return launch_prefill_s<T, C, 128, BS, 2, true>(a, g, stream);
    case 4:
      return launch_prefill_s<T, C, 128, BS, 4, true>(a, g, stream);
    default:
      return launch_prefill_s<T, C, 128, BS, 0, true>(a, g, stream);
  }
}

template <typename T, typename C>
hipError_t split_block(const PrefillArgs& a, const CacheGeom& g, hipStream_t stream) {
  const int group = a.num_heads / g.num_kv_heads;
  if (g.block_size == 16) return split_group<T, C, 16>(group, a, g, stream);
  if (g.block_size == 32) return split_group<T, C, 32>(group, a, g, stream);
  return hipErrorInvalidValue;
}

}  // namespace

// Where the 32-row tiles get a CU each (a workgroup fills one: 128 KiB of
// LDS) and there are enough keys that a wave's share pays for the merge.
// Measured (us, 128-row tiles -> split keys; bf16, 16 heads over 8, sequences
// x new over prior tokens): 1 x 100 over 400 14.8 -> 10.9, 1 x 512 over 0 14.7
// -> 12.0, over 1500 37.4 -> 22.7, over 6000 116 -> 62 (26 GFLOP: 424 TFLOP/s),
// 4 x 100 over 500 18.7 -> 13.4. Up to 64 rows, whose 128-row form runs half
// its waves, need more than 192 keys (4 x 16 over 96 7.2 -> 7.6, 8 x 16 over
// 176 7.8 -> 9.1, over 208 9.2 -> 9.1), and 384 from a tile per two CUs on (16
// x 16 over 304 10.4 -> 11.2). fp8 caches and the groups at run time gain from
// 64 keys on (fp8 4 x 8 over 88 6.2 -> 5.7).
// With up to two 32-row tiles per CU some CUs serve two, and the 128-row
// tiles, which read each K / V operand from L2 a quarter as often, win (4 x
// 200 over 500 21.0 -> 25.2, 8 x 100 over 2000 47.7 -> 68.9, 2 x 512 over 0
// 16.4 -> 17.0), but for one long causal chunk, whose last rows see far more
// keys than its first (1 x 700 over 500 30.8 -> 26.1, 1 x 1024 over 500 37.2
// -> 33.5; over 6000 143.9 -> 150), and the groups at run time (32 heads over
// 4: 1 x 400 over 2000 77.1 -> 64.0, 4 x 100 over 500 25.7 -> 27.5).
// Those batches were of equal queries and contexts. Where they differ, one
// sequence's rows are what is left at the end, and the split form gains far
// more than it costs an equal batch: over 6000 / 800 tokens 256 + 3 x 16 rows of
// an fp8 cache 119 -> 49.5, 512 + 32 over 6000 / 400 133 -> 78, 79-90 rows of 6
// over 11-1469 40.1 -> 23.8. The host has the largest of each only, so several
// sequences split up to a 128-row tile per four CUs, and per two over 512 keys
// (396 ragged batches: 4 more than 5 % slower than unsplit, by 25 % at most).
// Head dim 128, the decoder's, at 16- and 32-token blocks, is what is built: a
// 16-bit cache's two stages of four tiles do not fit the LDS at head dims 192
// and 256 (192 and 256 KiB); 64 and 96, 8-token blocks and the larger head
// dims over fp8 caches have not been tried.
bool prefill_split_keys(const PrefillArgs& a, const CacheGeom& g) {
  if (g.head_dim != 128 || g.block_size < 16) return false;
  const int group = a.num_heads / g.num_kv_heads;
  const bool any_group = group != 1 && group != 2 && group != 4;
  const int64_t pairs = (int64_t)a.num_seqs * g.num_kv_heads;
  const int64_t tiles = prefill_row_tiles(a.max_query_len, group, 32) * pairs;
  const int64_t cus = device_cu_count();
  if (tiles <= cus) {
    const bool few_rows = (int64_t)a.max_query_len * group <= 64 && !any_group &&
                          a.k_scale == nullptr;
    return a.max_kv_len > (!few_rows ? 2 : 4 * tiles <= cus ? 6 : 12) * kPrefillKeys;
  }
  const int64_t big_tiles = prefill_row_tiles(a.max_query_len, group, kPrefillWaves * 32) * pairs;
  if (a.num_seqs > 1 && 4 * big_tiles <= cus) return a.max_kv_len > 2 * kPrefillKeys;
  if (a.num_seqs > 1 || any_group)
    return 2 * big_tiles <= cus && a.max_kv_len >= 16 * kPrefillKeys;
  return tiles <= 2 * cus && a.causal && a.max_query_len > 512 &&
         a.max_kv_len < 4 * (int64_t)a.max_query_len;
}

hipError_t launch_prefill_split(int dtype, int cache_dtype, const PrefillArgs& a,
                                const CacheGeom& g, hipStream_t stream) {
  const bool f8 = cache_dtype == VPA_DTYPE_FP8_E4M3;
  if (dtype == VPA_DTYPE_BF16)
    return f8 ? split_block<bf16_t, fp8_t>(a, g, stream) : split_block<bf16_t, bf16_t>(a, g, stream);
  if (dtype == VPA_DTYPE_F16)
    return f8 ? split_block<f16_t, fp8_t>(a, g, stream) : split_block<f16_t, f16_t>(a, g, stream);
  return hipErrorInvalidValue;
}

}  // namespace vpa
