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

// Up to one 128-row tile per four CUs, whose 32-row tiles then have a CU each,
// unless a wave would get no more than half a tile of keys; up to one per two
// CUs where the keys are many. Above, the tiles of 128 rows, which read each
// K / V operand from L2 a quarter as often, fill the chip. Measured (us, 128-row
// tiles -> split keys; bf16, 16 heads over 8, sequences x new over prior
// tokens): 1 x 100 over 400 14.8 -> 10.9, 1 x 512 over 0 14.7 -> 12.0, over
// 1500 37.4 -> 22.7, over 6000 116 -> 62 (26 GFLOP: 424 TFLOP/s), 1 x 1024
// over 1024 35.7 -> 30.7, 2 x 512 over 512 21.3 -> 19.7; the other way round,
// 1 x 16 over 0 5.9 -> 7.8, 4 x 200 over 0 10.1 -> 11.9, 4 x 400 over 400 20.2
// -> 31.0; 32 heads over 4: 1 x 512 over 1500 45.9 -> 43.4, 1 x 1024 over 1024
// 44.3 -> 52.5. Head dim 128, the decoder's, at 16- and 32-token blocks only.
bool prefill_split_keys(const PrefillArgs& a, const CacheGeom& g) {
  if (g.head_dim != 128 || g.block_size < 16) return false;
  const int64_t tiles = prefill_row_tiles(a.max_query_len, a.num_heads / g.num_kv_heads,
                                          kPrefillWaves * 32) *
                        a.num_seqs * g.num_kv_heads;
  const int64_t cus = device_cu_count();
  return (tiles * 4 <= cus && a.max_kv_len > 2 * kPrefillKeys) ||
         (tiles * 2 <= cus && a.max_kv_len >= 16 * kPrefillKeys);
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
