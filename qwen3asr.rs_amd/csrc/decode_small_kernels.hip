// Paged-attention decode of small grids (gfx950): the rows kernel without a
// work list (decode_rows.h, kSmall), for at most 64 sequences.
//
// A decode of a few sequences is bound by latency and by what single CUs
// pull, not by HBM: a workgroup moves about 60 KB/us however many waves it
// has, and every dependent load in front of its tiles and every launch
// counts. So a context is shared by more workgroups (chunks of 256 to 1024
// tokens, chosen from the lengths on the device), workgroups have eight
// waves with stages of 4 loads (tiles past a wave's own are not loaded), and
// no plan launch comes before the call.
//
// Measured (us per layer of a graph, bf16, 16 heads over 8, head dim 128, 16-token
// blocks; list form of 2048-token chunks -> this form; sequences x tokens):
// 1 x 64 5.0 -> 3.9, 1 x 300-450 7.4 -> 6.9, 1 x 1500 14.6 -> 8.4, 1 x 4000
// 24.0 -> 9.8, 1 x 8000 24.7 -> 12.9, 8 x 100-1500 16.6 -> 9.8, 16 x 100-1500
// 17.7 -> 13.4, 4 x 6000-8000 30.5 -> 22.3. At 1 x 450 (7.4 us), sixteen
// waves took 7.8 and stages of 8 loads 7.2 (but 8.8 at 1 x 800 for 8.2).
#include <algorithm>

#include "decode_rows.h"
#include "vpa_device.h"
#include "vpa_internal.h"

namespace vpa {
namespace {

constexpr int kSmallMaxChunk = 1024;  // tokens, small_chunk_blocks' largest

// Waves per workgroup: eight; four over 32-token blocks of eight 16-byte loads
// per lane (16-bit head dim 128), which take more than 128 registers, so that
// a CU could not hold two workgroups of eight, and of which a context of 512
// tokens has only 16 (us per layer, eight -> four; sequences x tokens: 64 x
// 13-38 10.1 -> 7.7, 64 x 77-128 11.8 -> 9.5, 8 x 154-256 7.6 -> 6.9, 8 x
// 256-512 9.9 either way; the list form 7.2, 10.8, 7.1 and 9.4).
template <typename C, int D, int BS>
constexpr int kSmallWaves = BS == 32 && D * BS * (int)sizeof(C) / 1024 == 8 ? 4 : 8;

// Tokens per wave: the largest chunk's share, and at least head_dim (the
// merge reuses a wave's logits for its output).
template <int D, int NW>
constexpr int kSmallPT = D <= kSmallMaxChunk / NW ? kSmallMaxChunk / NW : D;

template <typename T, typename C, int D, int BS, int G>
hipError_t launch_small_t(const DecodeArgs& a, const CacheGeom& g, const DecodeWorkspace& ws,
                          int target, hipStream_t stream) {
  constexpr int NW = kSmallWaves<C, D, BS>, PT = kSmallPT<D, NW>;
  static_assert(PT % 64 == 0 && PT * NW >= kSmallMaxChunk, "chunk");
  // target > 0: at most `target` workgroups where the chunks are shorter than
  // the largest, else the largest chunks of every sequence
  const int64_t largest = std::max(1, (a.max_ctx + kSmallMaxChunk - 1) / kSmallMaxChunk);
  const int64_t items = target == 0 ? a.num_seqs
                                    : std::max<int64_t>(target / g.num_kv_heads,
                                                        a.num_seqs * largest);
  const int64_t units = items * g.num_kv_heads;
  auto go = [&](auto kernel) {
    const DecodeAppend none{nullptr, nullptr, 0, 0};
    const DecodeAppend& app = a.append != nullptr ? *a.append : none;
    hipLaunchKernelGGL(kernel, dim3((unsigned)units), dim3(64 * NW), 0, stream,
                       static_cast<T*>(a.out), static_cast<const T*>(a.query),
                       static_cast<const C*>(a.key_cache), static_cast<const C*>(a.value_cache),
                       a.block_tables, a.block_table_stride, a.scale, a.num_heads,
                       g.num_kv_heads, g.num_blocks, g.block_stride, g.head_stride, ws.part_out,
                       ws.max_parts, static_cast<const uint2*>(nullptr),
                       static_cast<const uint32_t*>(nullptr), a.num_seqs, a.max_ctx,
                       a.block_table_stride * g.block_size, a.k_scale, a.v_scale,
                       static_cast<const T*>(app.key), static_cast<const T*>(app.value),
                       app.key_token_stride, app.value_token_stride, g.kv_rep, a.context_lens,
                       kSmallMaxChunk / BS, target);
    return hipGetLastError();
  };
  if constexpr (!std::is_same_v<C, fp8_t> && fused_append_shape(D, BS)) {
    if (a.append != nullptr)
      return go(paged_decode_rows_kernel<T, C, D, BS, G, PT, NW, true, true>);
  }
  return go(paged_decode_rows_kernel<T, C, D, BS, G, PT, NW, false, true>);
}

template <typename T, typename C, int D, int BS>
hipError_t launch_small_g(int group, const DecodeArgs& a, const CacheGeom& g,
                          const DecodeWorkspace& ws, int target, hipStream_t stream) {
  // the rows kernel's shapes: 16-bit tiles of 1 to 8 whole KiB, and the fp8
  // tiles of those that are whole KiB too (at 8-token blocks, two rows per
  // value unit: head dims 128 and 256)
  constexpr bool kF8 = std::is_same_v<C, fp8_t>;
  constexpr int kUnits = D * BS / 8;
  constexpr bool kRows = kUnits % 64 == 0 && kUnits / 64 <= 8;
  constexpr bool kShape =
      kRows && (!kF8 || (BS == 8 ? D % 128 == 0 : (D * BS / 16) % 64 == 0));
  if constexpr (kShape) {
    if (group == 1) return launch_small_t<T, C, D, BS, 1>(a, g, ws, target, stream);
    if (group == 2) return launch_small_t<T, C, D, BS, 2>(a, g, ws, target, stream);
    if (group == 4) return launch_small_t<T, C, D, BS, 4>(a, g, ws, target, stream);
  }
  return hipErrorInvalidValue;
}

template <typename T, typename C, int D>
hipError_t launch_small_d(int group, const DecodeArgs& a, const CacheGeom& g,
                          const DecodeWorkspace& ws, int target, hipStream_t stream) {
  switch (g.block_size) {
    case 8:
      return launch_small_g<T, C, D, 8>(group, a, g, ws, target, stream);
    case 16:
      return launch_small_g<T, C, D, 16>(group, a, g, ws, target, stream);
    case 32:
      return launch_small_g<T, C, D, 32>(group, a, g, ws, target, stream);
    default:
      return hipErrorInvalidValue;
  }
}

template <typename T, typename C>
hipError_t launch_small(int group, const DecodeArgs& a, const CacheGeom& g,
                        const DecodeWorkspace& ws, int target, hipStream_t stream) {
  switch (g.head_dim) {
    case 64:
      return launch_small_d<T, C, 64>(group, a, g, ws, target, stream);
    case 96:
      return launch_small_d<T, C, 96>(group, a, g, ws, target, stream);
    case 128:
      return launch_small_d<T, C, 128>(group, a, g, ws, target, stream);
    case 192:
      return launch_small_d<T, C, 192>(group, a, g, ws, target, stream);
    case 256:
      return launch_small_d<T, C, 256>(group, a, g, ws, target, stream);
    default:
      return hipErrorInvalidValue;
  }
}

}  // namespace

// One chunk per context up to 512 tokens: a merge launch costs about as much
// as the second half of such a context takes (1 x 450: 7.4 us whole; in four
// chunks 7.7). Above, up to 128 (sequence, kv head) pairs: at 192 and more
// the list form, whose four-wave workgroups the dispatcher packs better, is
// as fast or faster (24 x 700-1000 tokens 15.9 us there with 1024-token
// chunks, 19.0 here; 16 x 13.9 and 14.7; 16 x 100-1500 15.9 and 13.4).
//
// Up to a maximum of 2048 tokens the list form is one launch once the step's
// list is there, and this one always two. Per layer of a planned step (us,
// list -> here; 16 heads over 8, head dim 128; maximum and the share of it
// that the contexts fill): 1 sequence, 2048, 5-15 % 6.2 -> 8.0, 30-50 % 12.0
// -> 9.1, half to all 18.0 -> 9.5; 1, 1024, 5.9 -> 7.6, 8.3 -> 9.0 and 10.7 ->
// 9.2; 8, 1024, 6.5 -> 8.2, 9.2 -> 9.8 and 14.0 -> 10.7; 16, 1024, 6.7 -> 8.3,
// 9.5 -> 10.9 and 14.9 -> 14.6. So a maximum frozen at more than about three
// times the longest context costs up to 2 us, and one that a context fills to
// the half or more, as the table widths of captured graphs do, gains as much
// or more. Without a list (a call that would build its own first) this form
// is the faster one throughout (1 sequence, 2048: 10.9, 16.7 and 22.8 -> 7.3,
// 8.6 and 9.0). Longer contexts of 8 and more sequences are the other place
// where a planned step can lose, worst with one or two workgroups per CU (8 x
// 3072-6144 31.1 -> 37.5, 16 x 4096-8192 72.3 -> 73.6; but 8 x 300-900 14.8 ->
// 10.3).
int decode_small_target(int num_seqs, int num_kv_heads, int max_ctx, int max_parts) {
  if (num_seqs > kSmallMaxSeqs) return -1;
  if (max_ctx <= 512) return 0;
  if (num_seqs * num_kv_heads > 128 || max_parts < (max_ctx + 255) / 256) return -1;
  return 256;
}

hipError_t launch_decode_small(int dtype, int cache_dtype, int group, const DecodeArgs& a,
                               const CacheGeom& g, const DecodeWorkspace& ws, int target,
                               hipStream_t stream) {
  const bool f8 = cache_dtype == VPA_DTYPE_FP8_E4M3;
  if (dtype == VPA_DTYPE_BF16)
    return f8 ? launch_small<bf16_t, fp8_t>(group, a, g, ws, target, stream)
              : launch_small<bf16_t, bf16_t>(group, a, g, ws, target, stream);
  if (dtype == VPA_DTYPE_F16)
    return f8 ? launch_small<f16_t, fp8_t>(group, a, g, ws, target, stream)
              : launch_small<f16_t, f16_t>(group, a, g, ws, target, stream);
  return hipErrorInvalidValue;
}

}  // namespace vpa
