// Chunked-prefill launches of the 16-bit MFMA kernel (prefill_paged.h): the
// instances whose waves each take 32 rows. prefill_split_kernels.hip has the
// ones whose waves split a row tile's keys.
#include "prefill_paged.h"
#include "vpa_device.h"
#include "vpa_internal.h"

namespace vpa {
namespace {

template <typename T, typename C, int D, int BS>
hipError_t dispatch_group(int group, const PrefillArgs& a, const CacheGeom& g,
                          hipStream_t stream) {
  switch (group) {
    case 1:
      return launch_prefill_s<T, C, D, BS, 1, false>(a, g, stream);
    case 2:
      return launch_prefill_s<T, C, D, BS, 2, false>(a, g, stream);
    case 4:
      return launch_prefill_s<T, C, D, BS, 4, false>(a, g, stream);
    default:
      return launch_prefill_s<T, C, D, BS, 0, false>(a, g, stream);
  }
}

// Shapes: head_dim 64, 96, 128, 192 or 256, block sizes 8, 16, 32, with a
// (block, head) tile of a whole number of 1 KiB DMAs (D * BS / x a multiple
// of 64 units): head_dim 96 at 16-bit needs 16- or 32-token blocks, at fp8
// 32-token ones; fp8 at 8-token blocks takes head_dim 128 and 256. At fp8
// head_dim 64 a 32-key tile is 128 units, moved by two of the four waves.
constexpr bool prefill_shape(bool fp8, int d, int bs) {
  const int x = fp8 ? 16 : 8;
  const bool dim = d == 64 || d == 96 || d == 128 || d == 192 || d == 256;
  const bool blk = bs == 8 || bs == 16 || bs == 32;
  return dim && blk && (d * bs / x) % 64 == 0;
}

template <typename T, typename C, int D, int BS>
hipError_t dispatch_if(int group, const PrefillArgs& a, const CacheGeom& g, hipStream_t stream,
                       bool& done) {
  constexpr bool kF8 = std::is_same_v<C, fp8_t>;
  if constexpr (prefill_shape(kF8, D, BS)) {
    if (g.head_dim == D && g.block_size == BS) {
      done = true;
      return dispatch_group<T, C, D, BS>(group, a, g, stream);
    }
  }
  return hipSuccess;
}

template <typename T, typename C, int D>
hipError_t dispatch_dim(int group, const PrefillArgs& a, const CacheGeom& g, hipStream_t stream,
                        bool& done) {
  hipError_t e = dispatch_if<T, C, D, 8>(group, a, g, stream, done);
  if (!done) e = dispatch_if<T, C, D, 16>(group, a, g, stream, done);
  if (!done) e = dispatch_if<T, C, D, 32>(group, a, g, stream, done);
  return e;
}

template <typename T, typename C>
hipError_t dispatch_shape(int group, const PrefillArgs& a, const CacheGeom& g,
                          hipStream_t stream) {
  bool done = false;
  hipError_t e = dispatch_dim<T, C, 128>(group, a, g, stream, done);
  if (!done) e = dispatch_dim<T, C, 64>(group, a, g, stream, done);
  if (!done) e = dispatch_dim<T, C, 96>(group, a, g, stream, done);
  if (!done) e = dispatch_dim<T, C, 192>(group, a, g, stream, done);
  if (!done) e = dispatch_dim<T, C, 256>(group, a, g, stream, done);
  return done ? e : hipErrorInvalidValue;
}

}  // namespace

bool prefill_supported(int dtype, int cache_dtype, int head_dim, int block_size, int group) {
  if (!(dtype == VPA_DTYPE_BF16 || dtype == VPA_DTYPE_F16) || group < 1) return false;
  const bool fp8 = cache_dtype == VPA_DTYPE_FP8_E4M3;
  if (!fp8 && cache_dtype != dtype) return false;
  return prefill_shape(fp8, head_dim, block_size);
}


hipError_t launch_prefill_paged(int dtype, int cache_dtype, void* out, const void* query,
                                const void* key_cache, const void* value_cache,
                                const uint32_t* block_tables, int32_t block_table_stride,
                                const uint32_t* cu_seqlens_q, const uint32_t* context_lens,
                                int32_t num_seqs, int32_t max_query_len, int32_t max_kv_len,
                                int64_t total_query_rows, float scale, float denom_eps,
                                int32_t causal, int32_t num_heads, const CacheGeom& g,
                                const float* k_scale, const float* v_scale,
                                hipStream_t stream) {
  const int group = num_heads / g.num_kv_heads;
  const PrefillArgs a{out,       query,        key_cache,      value_cache,  block_tables,
                      block_table_stride,      cu_seqlens_q,   context_lens, num_seqs,
                      max_query_len,           max_kv_len,     total_query_rows,
                      scale,     denom_eps,    causal,         num_heads,    k_scale,
                      v_scale};
  const bool f8 = cache_dtype == VPA_DTYPE_FP8_E4M3;
  if (prefill_split_keys(a, g)) return launch_prefill_split(dtype, cache_dtype, a, g, stream);
  if (dtype == VPA_DTYPE_BF16)
    return f8 ? dispatch_shape<bf16_t, fp8_t>(group, a, g, stream)
              : dispatch_shape<bf16_t, bf16_t>(group, a, g, stream);
  if (dtype == VPA_DTYPE_F16)
    return f8 ? dispatch_shape<f16_t, fp8_t>(group, a, g, stream)
              : dispatch_shape<f16_t, f16_t>(group, a, g, stream);
  return hipErrorInvalidValue;
}

}  // namespace vpa
