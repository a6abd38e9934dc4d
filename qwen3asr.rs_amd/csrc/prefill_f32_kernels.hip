// Chunked-prefill attention of f32 queries over the paged cache (f32, or fp8
// with scales) on gfx950's f32 matrix instructions (the Metal prefill's
// `float` and `float, uint8_t` instances, vasr-paged-attn/src/metal/kernels/
// prefill_paged_attn.metal:1606, 1610).
//
// Semantics are the 16-bit MFMA kernel's (prefill_kernels.hip): query i of a
// sequence with n queries and L keys sees keys t <= i + L - n when causal,
// every key otherwise; keys in blocks outside the pool are skipped; out =
// sum p v / (sum p + denom_eps) with p = exp(s - max), 0 for a row that sees
// no key. Any number of query heads per kv head: a kv head's (position,
// head) rows are enumerated heads-fastest.
//
// Work unit: one wave, 32 rows, 32 keys per tile. v_mfma_f32_32x32x2_f32
// multiplies and adds in f32, so nothing is held or computed in fewer bits
// than on the vector ALUs. It takes 64 cycles for 256 bytes of each operand,
// eight times the cycles per byte of the 16-bit instruction (sixteen per
// operation), which decides the rest: the matrix pipes are what bounds this
// kernel (busy 63 % of the time a SIMD has a wave, and for 18 % of the call it
// has none; 8 sequences of 64-512 new over 0-1024 tokens), the operands can come
// straight from the caches, and no LDS tile, transpose or barrier is needed. Both operands fall on the cache layouts: MFMA sums over k in any
// order that A and B share, so
//   S^T = K . Q^T   lane l holds key l % 32; its half h = l / 32 takes the
//     16-byte units 2 i + h of the key row [D/4][BS][4], four MFMAs per unit
//     (fp8: bytes 8 h .. 8 h + 7 of every 16-dim unit, eight MFMAs);
//   O^T += V^T . P^T  the accumulator's element r = 4 i + e of half h is key
//     8 i + 4 h + e, so P^T is the B operand as it stands and A is the
//     16-byte unit at key 8 i + 4 h of value row [D][BS] (fp8: 4 bytes).
// Loads run one group (16 MFMAs, 1024 cycles) ahead of their use, across
// tiles.
//
// The waves of a workgroup take four consecutive 32-row tiles (kSplit
// false), or one tile whose keys they split, tile t to wave t % 4, merged
// through LDS at the end (kSplit true): four times the workgroups, each a
// quarter as long.
//
// Measured with the append before it (16 heads over 8, head dim 128, 8
// sequences of 64-512 new over 0-1024 prior tokens, 15.1 GFLOP): 199 us,
// against 821 us on the vector kernel; a chunk of 512 over 6000 alone runs
// at 99 TFLOP/s (a large f32 matrix product reaches 154 on this card). Error
// against 64 bits 2.1e-7, the vector kernel's 2.3e-7.
//
// Rounding: a score is summed over 16 dims at a time, the P.V sums over one
// tile at a time (then added to the rescaled running output), so no rounding
// chain runs over more than 16 and 32 products. (Two chains of half the head
// dim put an element of the f32-query fp8-cache parity cases 1.3 times past
// the 1e-5 bound.)
#include <type_traits>

#include "vpa_device.h"
#include "vpa_internal.h"

namespace vpa {
namespace {

typedef float f32x16_t __attribute__((ext_vector_type(16)));

constexpr int kFThreads = 256;
constexpr int kFRows = 32;  // rows per wave
constexpr int kFKeys = 32;  // keys per tile

// max over lanes l and l ^ 32
__device__ __forceinline__ float max_halves(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false,
                                                  false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// Two fp8 bytes (pair `hi` of a word) as f32 (exact, through bf16)
__device__ __forceinline__ void fp8_pair(uint32_t w, bool hi, float& a, float& b) {
  const uint32_t p = hi ? fp8x2_to_pk<bf16_t>(w, true) : fp8x2_to_pk<bf16_t>(w, false);
  a = low_half_f32<bf16_t>(p);
  b = high_half_f32<bf16_t>(p);
}

// One group of A operands as loaded: sixteen elements per lane.
template <typename C>
struct Group {
  static constexpr int kWords = std::is_same_v<C, fp8_t> ? 4 : 16;
  uint32_t w[kWords];
  __device__ __forceinline__ float4 quad(int i) const {
    if constexpr (kWords == 16)
      return make_float4(__uint_as_float(w[4 * i]), __uint_as_float(w[4 * i + 1]),
                         __uint_as_float(w[4 * i + 2]), __uint_as_float(w[4 * i + 3]));
    float4 f;
    fp8_pair(w[i % kWords], false, f.x, f.y);
    fp8_pair(w[i % kWords], true, f.z, f.w);
    return f;
  }
};

template <typename C, int D, int BS, bool kSplit>
__global__ __launch_bounds__(kFThreads)
__attribute__((amdgpu_waves_per_eu(D > 128 ? 1 : 2))) void prefill_paged_f32_kernel(
    float* __restrict__ out, const float* __restrict__ query, const C* __restrict__ key_cache,
    const C* __restrict__ value_cache, const uint32_t* __restrict__ block_tables,
    int32_t block_table_stride, const uint32_t* __restrict__ cu_seqlens_q,
    const uint32_t* __restrict__ context_lens, int32_t max_query_len, int32_t max_kv_len,
    int64_t total_query_rows, float scale_log2, float denom_eps, int32_t causal,
    int32_t num_heads, int32_t num_kv_heads, int32_t group, int64_t num_blocks,
    int64_t block_stride, int64_t head_stride, int32_t row_tiles,
    const float* __restrict__ k_scale, const float* __restrict__ v_scale) {
  constexpr bool kF8 = std::is_same_v<C, fp8_t>;
  static_assert(kF8 || std::is_same_v<C, float>, "f32 or fp8 cache");
  static_assert(D % 32 == 0 && kFKeys % BS == 0 && BS >= 8, "shape");
  constexpr int NG = D / 32;  // groups of 32 dims: of a key row, of the output
  constexpr int kRowsPerWg = kSplit ? kFRows : 4 * kFRows;
  constexpr int kPitch = 36;  // floats per row of a merge buffer (16-byte rows, spread banks)
  __shared__ __align__(16) float s_o[kSplit ? 2 : 1][kSplit ? 4 : 1][kSplit ? kFRows * kPitch : 1];
  __shared__ float s_m[4][kFRows], s_l[4][kFRows];
  // query operands [quad][lane] of each wave's rows (of the one tile, kSplit):
  // in registers they would take D / 2 of a lane's 256
  __shared__ __align__(16) float4 s_q[kSplit ? 1 : 4][NG * 4][64];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 31, half = lane >> 5;
  // consecutive workgroups: kv heads, then the row tiles of one sequence
  // (heaviest first)
  const int j = (int)(blockIdx.x % (uint32_t)num_kv_heads);
  const int rest = (int)(blockIdx.x / (uint32_t)num_kv_heads);
  const int s = rest / row_tiles;
  const int rt = row_tiles - 1 - rest % row_tiles;

  const uint32_t qa = cu_seqlens_q[s], qb = cu_seqlens_q[s + 1];
  int q_len = qb > qa ? (int)min(qb - qa, (uint32_t)max_query_len) : 0;
  if ((int64_t)qa >= total_query_rows) q_len = 0;
  else q_len = (int)min((int64_t)q_len, total_query_rows - (int64_t)qa);
  const int k_len = (int)min(context_lens[s], (uint32_t)max_kv_len);
  // (32 bits past this: more rows than 2^32 do not fit the card)
  if ((int64_t)rt * kRowsPerWg >= (int64_t)q_len * group) return;
  const uint32_t ugroup = (uint32_t)group;
  const uint32_t row0 = (uint32_t)rt * kRowsPerWg;
  const uint32_t wrow0 = kSplit ? row0 : row0 + (uint32_t)wave * kFRows;
  const int shift = k_len - q_len;  // bottom-right causal alignment
  const int wpos0 = (int)min(wrow0 / ugroup, (uint32_t)q_len);
  if (!kSplit && wpos0 >= q_len) return;  // (no barrier follows)
  const int wpos_end = (int)min((wrow0 + kFRows - 1) / ugroup + 1, (uint32_t)q_len);
  const int wave_keys = max(0, causal ? min(k_len, wpos_end + shift) : k_len);
  const int n_tiles = (wave_keys + kFKeys - 1) / kFKeys;
  const int wave_min_limit = causal ? wpos0 + shift : k_len - 1;

  // this lane's row (column of S^T and O^T)
  const int pos = (int)min((wrow0 + col) / ugroup, (uint32_t)q_len);
  const int head = j * group + (int)((wrow0 + col) % ugroup);
  const bool row_ok = pos < q_len;
  const int limit = causal ? pos + shift : k_len - 1;  // last key the row sees

  float vs = 1.f;
  if constexpr (kF8) {
    scale_log2 *= *k_scale;
    vs = *v_scale;
  }

  // this lane's query operands, in the key groups' order (a row past the
  // sequence's queries reads its first row, in bounds, and is not stored)
  float4(&sq)[NG * 4][64] = s_q[kSplit ? 0 : wave];
  {
    const float* qrow =
        query + (((int64_t)qa + (row_ok ? pos : 0)) * num_heads + head) * D;
#pragma unroll
    for (int i = 0; i < 4 * NG; ++i) {
      if (kSplit && i % 4 != wave) continue;  // (the waves share the writing)
      const int d = kF8 ? 32 * (i / 4) + 16 * (i / 2 % 2) + 8 * half + 4 * (i % 2)
                        : 8 * i + 4 * half;
      sq[i][lane] = *reinterpret_cast<const float4*>(qrow + d);
    }
  }
  if constexpr (kSplit) __syncthreads();
  auto load_q = [&](float4(&b)[4], int g) {
#pragma unroll
    for (int i = 0; i < 4; ++i) b[i] = sq[4 * g + i][lane];
  };

  const C* kbase = key_cache + (int64_t)j * head_stride;
  const C* vbase = value_cache + (int64_t)j * head_stride;
  const uint32_t* bt = block_tables + (int64_t)s * block_table_stride;
  const int last_blk = max(k_len - 1, 0) / BS;

  // block id of key `col` of tile t (the index clamped to the sequence's
  // last block; keys past the context are masked)
  auto tile_id = [&](int t) -> uint32_t { return bt[min((t * kFKeys + col) / BS, last_blk)]; };
  // (this lane's key row of a tile, and its value rows by block)
  auto key_row = [&](uint32_t id) -> const C* {
    const int64_t phys = (int64_t)id < num_blocks ? (int64_t)id : 0;
    return kbase + phys * block_stride +
           (kF8 ? (col % BS) * 16 + 8 * half : (half * BS + col % BS) * 4);
  };
  auto load_k = [&](Group<C>& b, const C* row, int g) {
    if constexpr (kF8) {
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const uint2 u = *reinterpret_cast<const uint2*>(row + (2 * g + c) * BS * 16);
        b.w[2 * c] = u.x;
        b.w[2 * c + 1] = u.y;
      }
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint4 u = *reinterpret_cast<const uint4*>(row + (8 * g + 2 * i) * BS * 4);
        b.w[4 * i] = u.x;
        b.w[4 * i + 1] = u.y;
        b.w[4 * i + 2] = u.z;
        b.w[4 * i + 3] = u.w;
      }
    }
  };
  const int voff = col * BS + 4 * half;
  auto load_v = [&](Group<C>& b, uint32_t id, int dt) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {  // keys 8 i + 4 half .. + 3, in block 8 i / BS of the tile
      const uint32_t bid = (uint32_t)__builtin_amdgcn_readlane((int)id, 8 * i);
      const int64_t phys = (int64_t)bid < num_blocks ? (int64_t)bid : 0;
      const C* p = vbase + phys * block_stride + voff + 32 * dt * BS + (8 * i) % BS;
      if constexpr (kF8) {
        b.w[i] = *reinterpret_cast<const uint32_t*>(p);
      } else {
        const uint4 u = *reinterpret_cast<const uint4*>(p);
        b.w[4 * i] = u.x;
        b.w[4 * i + 1] = u.y;
        b.w[4 * i + 2] = u.z;
        b.w[4 * i + 3] = u.w;
      }
    }
  };

  f32x16_t o[NG];
#pragma unroll
  for (int dt = 0; dt < NG; ++dt)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[dt][e] = 0.f;
  float m = -INFINITY;  // the row's running max (log2 units)
  float lsum = 0.f;     // this lane's share of the row's sum against m

  constexpr int kStep = kSplit ? 4 : 1;
  int t = kSplit ? wave : 0;
  if (t < n_tiles) {
    uint32_t id = tile_id(t);
    uint32_t id_next = tile_id(t + kStep);
    Group<C> buf[2];
    float4 qb[2][4];
    load_k(buf[0], key_row(id), 0);
    for (; t < n_tiles; t += kStep) {
      const int k0 = t * kFKeys;
      // keys of the tile that exist: in the context and in a block of the pool
      const uint32_t vmask =
          (uint32_t)__ballot(k0 + col < k_len && (int64_t)id < num_blocks);
      const bool full = vmask == 0xffffffffu && k0 + kFKeys - 1 <= wave_min_limit;

      // S^T = K . Q^T, every 16 dims summed on their own
      f32x16_t sum;
      const C* krow = key_row(id);
      load_q(qb[0], 0);
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        if (g + 1 < NG) load_k(buf[(g + 1) & 1], krow, g + 1);
        else load_v(buf[(g + 1) & 1], id, 0);
        if (g + 1 < NG) load_q(qb[(g + 1) & 1], g + 1);
        __builtin_amdgcn_sched_barrier(0);  // the next group's loads ahead of this one's MFMAs
#pragma unroll
        for (int i2 = 0; i2 < 2; ++i2) {
          f32x16_t acc;
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[e] = 0.f;
#pragma unroll
          for (int i = 2 * i2; i < 2 * i2 + 2; ++i) {
            const float4 a = buf[g & 1].quad(i);
            const float4 b = qb[g & 1][i];
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.x, b.x, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.y, b.y, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.z, b.z, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.w, b.w, acc, 0, 0, 0);
          }
#pragma unroll
          for (int e = 0; e < 16; ++e) sum[e] = g + i2 == 0 ? acc[e] : sum[e] + acc[e];
          // (added here and now: the compiler would otherwise keep every
          // 16-dim sum of the row in registers of its own and spill)
          asm volatile("" : "+v"(sum));
        }
      }

      float p[16];
      float mx = -INFINITY;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key = 8 * (r / 4) + 4 * half + r % 4;
        const bool ok = full || (((vmask >> key) & 1u) && k0 + key <= limit);
        p[r] = ok ? sum[r] * scale_log2 : -INFINITY;
        mx = fmaxf(mx, p[r]);
      }
      const float m_new = fmaxf(m, max_halves(mx));
      float alpha = 1.f;
      if (m_new != -INFINITY) alpha = m == -INFINITY ? 0.f : exp2f(m - m_new);
#pragma unroll
      for (int r = 0; r < 16; ++r)
        p[r] = p[r] == -INFINITY ? 0.f : exp2f(p[r] - m_new);
      m = m_new;
      float ps[8];
#pragma unroll
      for (int r = 0; r < 8; ++r) ps[r] = p[r] + p[r + 8];
      lsum = fmaf(lsum, alpha, ((ps[0] + ps[4]) + (ps[1] + ps[5])) +
                                   ((ps[2] + ps[6]) + (ps[3] + ps[7])));

      // O^T = O^T alpha + V^T . P^T, one 32-dim tile after the other
      const uint32_t id_after = tile_id(t + 2 * kStep);
#pragma unroll
      for (int dt = 0; dt < NG; ++dt) {
        Group<C>& cur = buf[(NG + dt) & 1];
        Group<C>& nxt = buf[(NG + dt + 1) & 1];
        if (dt + 1 < NG) load_v(nxt, id, dt + 1);
        else load_k(nxt, key_row(id_next), 0);  // (past the last tile: loaded, not used)
        __builtin_amdgcn_sched_barrier(0);
        f32x16_t ta;
#pragma unroll
        for (int e = 0; e < 16; ++e) ta[e] = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float4 a = cur.quad(i);
          if (vmask != 0xffffffffu) {  // (uniform) stale values: zero the absent keys
            const uint32_t bits = vmask >> (8 * i + 4 * half);
            a.x = (bits & 1u) ? a.x : 0.f;
            a.y = (bits & 2u) ? a.y : 0.f;
            a.z = (bits & 4u) ? a.z : 0.f;
            a.w = (bits & 8u) ? a.w : 0.f;
          }
          ta = __builtin_amdgcn_mfma_f32_32x32x2f32(a.x, p[4 * i], ta, 0, 0, 0);
          ta = __builtin_amdgcn_mfma_f32_32x32x2f32(a.y, p[4 * i + 1], ta, 0, 0, 0);
          ta = __builtin_amdgcn_mfma_f32_32x32x2f32(a.z, p[4 * i + 2], ta, 0, 0, 0);
          ta = __builtin_amdgcn_mfma_f32_32x32x2f32(a.w, p[4 * i + 3], ta, 0, 0, 0);
        }
#pragma unroll
        for (int e = 0; e < 16; ++e) o[dt][e] = fmaf(o[dt][e], alpha, ta[e]);
        __builtin_amdgcn_sched_barrier(0);
      }
      id = id_next;
      id_next = id_after;
    }
  }

  // (m is the row's true max, so the epsilon is added as it stands; a row
  // that sees no key gives 0)
  const float total = sum_xor32(lsum);
  if constexpr (!kSplit) {
    if (row_ok) {
      const float inv = total > 0.f ? vs / (total + denom_eps) : 0.f;
      float* orow = out + (((int64_t)qa + pos) * num_heads + head) * D;
#pragma unroll
      for (int dt = 0; dt < NG; ++dt)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          *reinterpret_cast<float4*>(orow + 32 * dt + 8 * i + 4 * half) =
              make_float4(o[dt][4 * i] * inv, o[dt][4 * i + 1] * inv, o[dt][4 * i + 2] * inv,
                          o[dt][4 * i + 3] * inv);
    }
  } else {
    if (half == 0) {
      s_m[wave][col] = m;
      s_l[wave][col] = total;
    }
    __syncthreads();
    auto weight = [&](int w, int r, float mx) {
      return s_m[w][r] == -INFINITY ? 0.f : exp2f(s_m[w][r] - mx);
    };
    auto row_max = [&](int r) {
      return fmaxf(fmaxf(s_m[0][r], s_m[1][r]), fmaxf(s_m[2][r], s_m[3][r]));
    };
    const float wgt = weight(wave, col, row_max(col));
    // thread e of the workgroup combines 4 dims of row e / 8
    const int r = threadIdx.x >> 3, d4 = (threadIdx.x & 7) * 4;
    const uint32_t orow_i = row0 + (uint32_t)r;
    const int opos = (int)min(orow_i / ugroup, (uint32_t)q_len);
    const float rmx = row_max(r);
    float den = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) den = fmaf(weight(w, r, rmx), s_l[w][r], den);
    const float inv = den > 0.f ? vs / (den + denom_eps) : 0.f;
    float* orow = out + (((int64_t)qa + opos) * num_heads + j * group +
                         (int)(orow_i % ugroup)) * D + d4;
#pragma unroll
    for (int dt = 0; dt < NG; ++dt) {
      float* mine = &s_o[dt & 1][wave][col * kPitch];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<float4*>(mine + 8 * i + 4 * half) =
            make_float4(o[dt][4 * i] * wgt, o[dt][4 * i + 1] * wgt, o[dt][4 * i + 2] * wgt,
                        o[dt][4 * i + 3] * wgt);
      __syncthreads();  // (two buffers: the next round's writes need no barrier of their own)
      float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const float4 x = *reinterpret_cast<const float4*>(&s_o[dt & 1][w][r * kPitch + d4]);
        a.x += x.x;
        a.y += x.y;
        a.z += x.z;
        a.w += x.w;
      }
      if (opos < q_len)
        *reinterpret_cast<float4*>(orow + 32 * dt) =
            make_float4(a.x * inv, a.y * inv, a.z * inv, a.w * inv);
    }
  }
}

struct F32Args {
  float* out;
  const float* query;
  const void* key_cache;
  const void* value_cache;
  const uint32_t* block_tables;
  int32_t block_table_stride;
  const uint32_t* cu_seqlens_q;
  const uint32_t* context_lens;
  int32_t num_seqs, max_query_len, max_kv_len;
  int64_t total_query_rows;
  float scale, denom_eps;
  int32_t causal, num_heads;
  const float* k_scale;
  const float* v_scale;
};

template <typename C, int D, int BS, bool kSplit>
hipError_t launch_f32_t(const F32Args& a, const CacheGeom& g, hipStream_t stream) {
  constexpr int kRows = kSplit ? kFRows : 4 * kFRows;
  const int group = a.num_heads / g.num_kv_heads;
  const int64_t row_tiles = ((int64_t)a.max_query_len * group + kRows - 1) / kRows;
  const int64_t grid = (int64_t)a.num_seqs * row_tiles * g.num_kv_heads;
  if (grid == 0) return hipSuccess;
  hipLaunchKernelGGL((prefill_paged_f32_kernel<C, D, BS, kSplit>), dim3((uint32_t)grid),
                     dim3(kFThreads), 0, stream, a.out, a.query,
                     static_cast<const C*>(a.key_cache), static_cast<const C*>(a.value_cache),
                     a.block_tables, a.block_table_stride, a.cu_seqlens_q, a.context_lens,
                     a.max_query_len, a.max_kv_len, a.total_query_rows,
                     a.scale * 1.4426950408889634f, a.denom_eps, a.causal, a.num_heads,
                     g.num_kv_heads, group, g.num_blocks, g.block_stride, g.head_stride,
                     (int32_t)row_tiles, a.k_scale, a.v_scale);
  return hipGetLastError();
}

// Whether a workgroup's waves split one row tile's keys. It fills the chip
// with few rows and balances ragged ones; it costs a merge per 32 rows, which
// only pays off where a wave still gets more than two or three tiles of keys.
// Measured (us, split / not; sequences x new over prior tokens, 16 heads over
// 8): 1 x 100 over 0 11 / 23, 1 x 512 over 6000 264 / 1035, 8 x 512 over 1000
// 241 / 380, 64 x 512 over 512 1344 / 1473, 32 x 300 over 0 143 / 152; 32
// heads over 4 with many short rows: 32 x 300 over 0 259 / 225, 64 x 64 over
// 200 172 / 153. One tile of keys has nothing to split (64 x 1 over 31, head
// dim 192 over fp8 30.0 / 25.0). Where a sequence has no more than 32 rows,
// three of the four waves of the other form have none, and its LDS (all four
// waves' queries) keeps workgroups off the CU: above head dim 64 that costs
// more than the merge from two tiles of keys on (head dim 128, 128 x 1 over
// 199 56 / 91; 192 over fp8, 128 x 1 over 63 58 / 84; but head dim 64, 128 x 1
// over 95 20.9 / 16.3).
bool split_keys(const F32Args& a, const CacheGeom& g) {
  if (a.max_kv_len <= kFKeys) return false;
  const int64_t rows = (int64_t)a.max_query_len * (a.num_heads / g.num_kv_heads);
  const int64_t tiles = (rows + 4 * kFRows - 1) / (4 * kFRows) * a.num_seqs * g.num_kv_heads;
  if (rows <= kFRows && g.head_dim > 64 && (a.max_kv_len > 2 * kFKeys || g.head_dim > 128))
    return true;
  return a.max_kv_len > 10 * kFKeys || tiles < 4 * (int64_t)device_cu_count();
}

template <typename C, int D, int BS>
hipError_t launch_f32_shape(const F32Args& a, const CacheGeom& g, hipStream_t stream) {
  return split_keys(a, g) ? launch_f32_t<C, D, BS, true>(a, g, stream)
                          : launch_f32_t<C, D, BS, false>(a, g, stream);
}

template <typename C, int D>
hipError_t launch_f32_dim(const F32Args& a, const CacheGeom& g, hipStream_t stream) {
  switch (g.block_size) {
    case 8:
      return launch_f32_shape<C, D, 8>(a, g, stream);
    case 16:
      return launch_f32_shape<C, D, 16>(a, g, stream);
    case 32:
      return launch_f32_shape<C, D, 32>(a, g, stream);
    default:
      return hipErrorInvalidValue;
  }
}

template <typename C>
hipError_t launch_f32(const F32Args& a, const CacheGeom& g, hipStream_t stream) {
  switch (g.head_dim) {
    case 64:
      return launch_f32_dim<C, 64>(a, g, stream);
    case 96:
      return launch_f32_dim<C, 96>(a, g, stream);
    case 128:
      return launch_f32_dim<C, 128>(a, g, stream);
    case 192:
      return launch_f32_dim<C, 192>(a, g, stream);
    case 256:
      return launch_f32_dim<C, 256>(a, g, stream);
    default:
      return hipErrorInvalidValue;
  }
}

}  // namespace

hipError_t launch_prefill_f32(int dtype, int cache_dtype, void* out, const void* query,
                              const void* key_cache, const void* value_cache,
                              const uint32_t* block_tables, int32_t block_table_stride,
                              const uint32_t* cu_seqlens_q, const uint32_t* context_lens,
                              int32_t num_seqs, int32_t max_query_len, int32_t max_kv_len,
                              int64_t total_query_rows, float scale, float denom_eps,
                              int32_t causal, int32_t num_heads, const CacheGeom& g,
                              const float* k_scale, const float* v_scale, hipStream_t stream) {
  if (dtype != VPA_DTYPE_F32) return hipErrorInvalidValue;
  // Over one tile of keys a wave here is a chain of D matrix instructions of
  // 64 cycles, and where the vector kernel's workgroups have a CU each that is
  // quicker (us, vector / here; 16 heads over 8, sequences x new over prior
  // tokens: 1 x 1 over 0 8.8 / 9.7, 1 x 32 over 0 9.8 / 10.3; head dim 64, 1 x
  // 16 over 0 5.9 / 7.0, 32 x 1 over 31 6.6 / 5.9; with more workgroups than
  // CUs, head dim 128, 64 x 16 over 16 27.1 / 13.9)
  if (max_kv_len <= kFKeys &&
      prefill_vector_workgroups(num_seqs, max_query_len, num_heads / g.num_kv_heads,
                                g.num_kv_heads) <= device_cu_count())
    return launch_prefill_vector(dtype, cache_dtype, out, query, key_cache, value_cache,
                                 block_tables, block_table_stride, cu_seqlens_q, context_lens,
                                 num_seqs, max_query_len, max_kv_len, total_query_rows, scale,
                                 denom_eps, causal, num_heads, g, k_scale, v_scale, stream);
  const F32Args a{static_cast<float*>(out), static_cast<const float*>(query), key_cache,
                  value_cache, block_tables, block_table_stride, cu_seqlens_q, context_lens,
                  num_seqs, max_query_len, max_kv_len, total_query_rows, scale, denom_eps,
                  causal, num_heads, k_scale, v_scale};
  return cache_dtype == VPA_DTYPE_FP8_E4M3 ? launch_f32<fp8_t>(a, g, stream)
                                           : launch_f32<float>(a, g, stream);
}

}  // namespace vpa
