// Pooled extraction: the lookup of a multi-hot feature and its per-sample combination in one kernel
// (ugk_extract_pool_*).  The kernels of 4-byte ids are in ugk_pool.hip, those of 8-byte ids in ugk_pool_i64.hip, which the build
// compiles side by side (together they take the compiler longer than the rest of the library).
#pragma once

#include <hip/hip_fp16.h>

#include <cstdlib>
#include <type_traits>

#include "ugk_internal.h"
#include "ugk_mix.cuh"
#include "ugk_table.cuh"

namespace ugk {
namespace {

// ---- pooled extraction -------------------------------------------------------------------------------------
// out[r, :] = combine_j( w_j * row(ids[j]) ) over the ids j of segment r = [seg_off[r], seg_off[r + 1]): the lookup of
// a multi-hot feature and the per-sample combination that follows it (embedding_lookup_sparse behind
// python_tf2/collcache_tf2/collcache_tf2/core/sparse_lookup_layer.py:196-265) in one pass, so that the nnz x row_bytes
// intermediate of a lookup followed by a segment sum is never written or read back.  A group of LPR lanes owns an
// output row: its lanes resolve LPR of the row's ids at a time (the table lookup is the fused extraction's), then
// every id's row is read once, 16 bytes per lane and chunk, and added in fp32 in the order of the ids.
// the elements of a 16-byte chunk as floats and back.  `bf16` picks between the two two-byte formats at run time (a
// wavefront-uniform branch), so that bfloat16 rows cost no kernels of their own.
template <typename E>
struct PoolElem;
template <>
struct PoolElem<float> {
  static constexpr int kPerChunk = 4;
  static __device__ __forceinline__ void unpack(const u32x4 &v, float *x, bool) {
    x[0] = __uint_as_float(v.x), x[1] = __uint_as_float(v.y), x[2] = __uint_as_float(v.z), x[3] = __uint_as_float(v.w);
  }
  static __device__ __forceinline__ u32x4 pack(const float *x, bool) {
    return u32x4{__float_as_uint(x[0]), __float_as_uint(x[1]), __float_as_uint(x[2]), __float_as_uint(x[3])};
  }
};
// round to nearest even; NaN stays NaN
__device__ __forceinline__ uint32_t float_to_bf16_bits(float f) {
  const uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (u >> 16) | 0x40u;
  return (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
}
template <>
struct PoolElem<__half> {
  static constexpr int kPerChunk = 8;
  static __device__ __forceinline__ void unpack(const u32x4 &v, float *x, bool bf16) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
    if (bf16) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        x[2 * k] = __uint_as_float(w[k] << 16);
        x[2 * k + 1] = __uint_as_float(w[k] & 0xffff0000u);
      }
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        x[2 * k] = __half2float(__ushort_as_half((unsigned short)(w[k] & 0xffffu)));
        x[2 * k + 1] = __half2float(__ushort_as_half((unsigned short)(w[k] >> 16)));
      }
    }
  }
  static __device__ __forceinline__ u32x4 pack(const float *x, bool bf16) {
    uint32_t w[4];
    if (bf16) {
#pragma unroll
      for (int k = 0; k < 4; ++k) w[k] = float_to_bf16_bits(x[2 * k]) | (float_to_bf16_bits(x[2 * k + 1]) << 16);
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k)
        w[k] = (uint32_t)__half_as_ushort(__float2half(x[2 * k])) |
               ((uint32_t)__half_as_ushort(__float2half(x[2 * k + 1])) << 16);
    }
    return u32x4{w[0], w[1], w[2], w[3]};
  }
};

constexpr int kPoolChunks = 4;  // 16-byte chunks of a row a lane may own at most: rows of up to LPR x 64 bytes

// Bound by the host link where rows are missing from the cache (65,536 samples of 16 ids over rows of 512 bytes, 2.6 %
// of them over the link: 280 us, 51 GB/s of link; 398 us before), else by the lines of the rows.  What decides is how
// many rows are on their way at once and that no load waits for another: a lane reads its CH chunks of U ids before it
// adds the first of them (a row of the host table whose chunks were read one after the other cost its wavefront CH
// round trips over the link), and CH and U are template parameters so that short rows do not pay for the registers of
// long ones.
// KEEP: the loads are ordinary ones: ids repeat in real batches, and the hot rows stay in L2.  Uniform ids, which reuse
// nothing, are up to a tenth faster with non-temporal ones where rows are whole lines, and which law its ids follow a launch
// does not know.  Where that matters (MIXED) keep_waves of a workgroup's four wavefronts load ordinarily: a row that many
// wavefronts read comes by one of those soon and stays in L2 for all of them, and rows read once mostly pass through.  Two
// bodies and not a branch around the loads: of two loads that differ in the hint only the compiler makes one.  800,000 ids
// over rows of 512 bytes, all in HBM, 4 ids per sample, none / one / two / three / all four ordinary: uniform 90 / 88 / 92 / 97 /
// 100 us, Zipf 1.05 76 / 62 / 60 / 58 / 56.
// CLIP: every looked-up row is clipped to the l2 norm max_norm before it is weighted (clip_by_norm over the row:
// x * max_norm / max(||x||, max_norm)).  The whole row has to be seen before any of it can be added, so the chunks of
// the U rows in flight are held in registers (up to 64 more than without), the squares summed per row over the lanes
// of the group, and the row's weight scaled; a kernel of its own, so that the plain combination keeps its registers.
// STORE: a launch whose end the host polls for writes its rows through and copies ids for the host, any other does neither and
// is another kernel.  With the choice at run time the others took longer, us per stream-ordered launch, rows in HBM: 60,000
// ids of 1 KB, one per sample 29.8 against 25.8, two 20.1 / 18.8, four 17.1 / 15.1; 262,144 of 64 bytes, one 13.3 / 12.7, two
// 10.8 / 10.1; 8,192 of 4 KB, sixteen 11.2 / 10.5.
template <typename K, int KIND, int LPR, int CH, int U, typename E, bool CLIP, bool KEEP, Store STORE>
__device__ __forceinline__ void pool_samples(const ugk_table_t &t, const K *__restrict__ ids,
                                             const long long *__restrict__ seg_off, const float *__restrict__ weights,
                                             size_t n_rows, long long nnz, const u32x4 *__restrict__ cache,
                                             uint64_t cache_rows, const u32x4 *__restrict__ host, uint64_t host_rows,
                                             u32x4 *__restrict__ out, uint32_t vpr, int combiner, bool bf16,
                                             float max_norm, uint32_t *status, uint32_t *host_mirror,
                                             const Ending<STORE> &done, uint32_t &wave_local,
                                             uint32_t &wave_host) {
  constexpr int RPW = kWave / LPR;  // output rows per wavefront and pass
  constexpr int EPC = PoolElem<E>::kPerChunk;
  static_assert(LPR % U == 0, "ids are taken in rounds of U");
  constexpr int kParts = LPR * CH <= 32 ? 8 : LPR * CH <= 128 ? 32 : 64;  // sums of weights per sample (see below)
  static_assert(LPR * 2 >= kParts && LPR <= kParts * 2, "a lane has one sum of weights, two, or half of one");
  const int lane = (int)lane_id();
  const int sub = lane % LPR, rg = lane / LPR;
  const size_t wave_global = (size_t)blockIdx.x * kWavesPerBlock + threadIdx.x / kWave;
  const size_t n_waves = (size_t)gridDim.x * kWavesPerBlock;
  for (size_t row0 = wave_global * RPW; row0 < n_rows; row0 += n_waves * RPW) {  // wavefront-uniform
    const size_t r = row0 + rg;
    const bool row_ok = r < n_rows;
    long long beg = row_ok ? seg_off[r] : 0, end = row_ok ? seg_off[r + 1] : 0;
    if (beg < 0 || end > nnz || end < beg) {  // a segment outside the ids: nothing is read for it, its row is zeros
      if (sub == 0) {
        atomicOr(status, UGK_ST_BAD_SEGMENT);
        if (host_mirror) tell_host<uint32_t>(host_mirror, UGK_ST_BAD_SEGMENT);
      }
      beg = end = 0;
    } else if (row_ok && sub == 0 && ((r == 0 && beg != 0) || (r + 1 == n_rows && end != nnz))) {
      // the offsets do not cover the ids from the first to the last (neighbouring segments share their boundary word,
      // so the two ends are all that can be wrong): the per-source id counts would not add up to nnz
      atomicOr(status, UGK_ST_BAD_SEGMENT);
      if (host_mirror) tell_host<uint32_t>(host_mirror, UGK_ST_BAD_SEGMENT);
    }
    float acc[CH][EPC];
#pragma unroll
    for (int c = 0; c < CH; ++c)
#pragma unroll
      for (int e = 0; e < EPC; ++e) acc[c][e] = 0.f;
    // This lane's share of the row's sum of weights (or of their squares), added in an order that the row's length fixes and
    // the shape does not: kParts sums, sum k over the ids k, k + kParts, ... of the sample.  Fewer lanes than sums take two
    // in turn; twice as many lanes keep each sum twice and add two ids a round to it.  (The shape depends on the whole
    // batch: without this a sample's last bits would depend on the samples beside it.)
    float wsum = 0.f, wsum_odd = 0.f;
    bool odd = false;
    for (long long j0 = beg; __ballot(j0 < end) != 0ull; j0 += LPR) {  // until every group of the wavefront is through
      const long long j = j0 + sub;
      const bool active = j < end;
      const uint64_t key = active ? key_to_u64<K>(ids[j]) : 0;
      const Found f = table_lookup<KIND>(t, key, active);
      const MixRow row = mix_resolve(t, key, active, f, cache, cache_rows, host, host_rows, out, vpr, status, host_mirror);
      if (done.words) {
        wave_local += __popcll(__ballot(row.from_cache));
        wave_host += __popcll(__ballot(active && !row.from_cache));
      }
      const bool use = active && row.has_row;  // a key without a row adds nothing (the launch is flagged)
      const float w = use ? (weights ? weights[j] : 1.f) : 0.f;
      for (int s0 = 0; s0 < LPR; s0 += U) {
        if (__ballot(active && sub >= s0) == 0ull) break;  // no group has an id left in this round
        grow_t p[U];
        float wv[U];
        bool ok[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int src = rg * LPR + s0 + u;
          p[u] = reinterpret_cast<grow_t>(shfl64(row.bits, src));
          wv[u] = __shfl(w, src);
          ok[u] = __shfl((int)use, src) != 0;
        }
        if constexpr (CLIP) {
          u32x4 v[CH][U];
          float ss[U];
#pragma unroll
          for (int u = 0; u < U; ++u) ss[u] = 0.f;
#pragma unroll
          for (int c = 0; c < CH; ++c) {
            const uint32_t col = (uint32_t)c * LPR + sub;
#pragma unroll
            for (int u = 0; u < U; ++u) v[c][u] = col < vpr ? __builtin_nontemporal_load(p[u] + col) : u32x4{0, 0, 0, 0};
          }
#pragma unroll
          for (int c = 0; c < CH; ++c) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
              float x[EPC];
              PoolElem<E>::unpack(v[c][u], x, bf16);  // a chunk past the row's end is zeros in either two-byte format
#pragma unroll
              for (int e = 0; e < EPC; ++e) ss[u] = fmaf(x[e], x[e], ss[u]);
            }
          }
#pragma unroll
          for (int u = 0; u < U; ++u) {
#pragma unroll
            for (int d = LPR / 2; d > 0; d >>= 1) ss[u] += __shfl_xor(ss[u], d);
            wv[u] *= max_norm / fmaxf(sqrtf(ss[u]), max_norm);
          }
#pragma unroll
          for (int c = 0; c < CH; ++c) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
              float x[EPC];
              PoolElem<E>::unpack(v[c][u], x, bf16);
              if (ok[u]) {
#pragma unroll
                for (int e = 0; e < EPC; ++e) acc[c][e] = fmaf(wv[u], x[e], acc[c][e]);
              }
            }
          }
        } else {
          // No branch around the loads (behind one they would wait for each other): a lane past the end of the row
          // reads the row's last chunk again, and what it adds up is never written.
          u32x4 v[CH][U];
#pragma unroll
          for (int c = 0; c < CH; ++c) {
            const uint32_t col = min((uint32_t)c * LPR + sub, vpr - 1);
#pragma unroll
            for (int u = 0; u < U; ++u) v[c][u] = KEEP ? p[u][col] : __builtin_nontemporal_load(p[u] + col);
          }
#pragma unroll
          for (int c = 0; c < CH; ++c) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
              float x[EPC];
              PoolElem<E>::unpack(v[c][u], x, bf16);
              if (ok[u]) {
#pragma unroll
                for (int e = 0; e < EPC; ++e) acc[c][e] = fmaf(wv[u], x[e], acc[c][e]);
              }
            }
          }
        }
      }
      if constexpr (STORE == kThrough) {
        if (active) copy_key_along<K>(done, (uint64_t)j, (K)key);
      }
      // (behind the rows: in front of them their loads would wait for the weights)
      const float wterm = combiner == 2 ? w * w : w;
      if constexpr (LPR < kParts) {
        if (odd) wsum_odd += wterm;
        else wsum += wterm;
        odd = !odd;
      } else if constexpr (LPR > kParts) {
        static_assert(LPR == 16 && kParts == 8, "lane l and lane l xor 8 of 16");
        constexpr int kRowRor8 = 0x128;  // DPP control: the 16 lanes of a row rotated by 8, no trip through LDS
        const float other = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(wterm), kRowRor8, 0xf, 0xf, true));
        const bool second = (sub & kParts) != 0;
        wsum += second ? other : wterm;
        wsum += second ? wterm : other;
      } else {
        wsum += wterm;
      }
    }
    // the row's denominator: every lane of the group holds a share
    if constexpr (LPR < kParts) wsum += wsum_odd;
#pragma unroll
    for (int d = (LPR < kParts ? LPR : kParts) / 2; d > 0; d >>= 1) wsum += __shfl_xor(wsum, d);
    const float denom = combiner == 1 ? wsum : combiner == 2 ? sqrtf(wsum) : 1.f;
    if (row_ok) {
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        const uint32_t col = (uint32_t)c * LPR + sub;
        if (col < vpr) {
          float y[EPC];
#pragma unroll
          for (int e = 0; e < EPC; ++e) y[e] = denom != 0.f ? acc[c][e] / denom : 0.f;  // div_no_nan
          const u32x4 packed = PoolElem<E>::pack(y, bf16);
          if constexpr (STORE == kThrough) store_through(reinterpret_cast<uint64_t>(out + r * vpr + col), packed);
          else out[r * vpr + col] = packed;
        }
      }
    }
  }
}


// A sample per workgroup, for batches of few samples with many ids each.  What such a launch takes is not bandwidth but the
// chain of a sample: a lane group that resolves LPR ids at a time and keeps U rows on their way goes through the ids of a
// sample of 40 in ten rounds trips to memory and three lookups, on a chip that is mostly idle.  Here 256 lanes resolve up to
// 256 ids at once and have kFewTileBytes of rows on their way at once, whichever ids and chunks those are; the rows meet in
// LDS, where a lane per 4-byte word adds them in the order of the ids, as pool_samples does: the same sums, bit for bit.
constexpr uint32_t kFewTileBytes = 32768;
template <typename E>
__device__ __forceinline__ void pool_unpack_word(uint32_t w, float *x, bool bf16) {
  if constexpr (sizeof(E) == 4) {
    x[0] = __uint_as_float(w);
  } else if (bf16) {
    x[0] = __uint_as_float(w << 16), x[1] = __uint_as_float(w & 0xffff0000u);
  } else {
    x[0] = __half2float(__ushort_as_half((unsigned short)(w & 0xffffu)));
    x[1] = __half2float(__ushort_as_half((unsigned short)(w >> 16)));
  }
}
template <typename E>
__device__ __forceinline__ uint32_t pool_pack_word(const float *x, bool bf16) {
  if constexpr (sizeof(E) == 4) return __float_as_uint(x[0]);
  else if (bf16) return float_to_bf16_bits(x[0]) | (float_to_bf16_bits(x[1]) << 16);
  else return (uint32_t)__half_as_ushort(__float2half(x[0])) | ((uint32_t)__half_as_ushort(__float2half(x[1])) << 16);
}

template <typename K, int KIND, int G, typename E, Store STORE>
__device__ __forceinline__ void pool_few_samples(const ugk_table_t &t, const K *__restrict__ ids,
                                                 const long long *__restrict__ seg_off, const float *__restrict__ weights,
                                                 size_t n_rows, long long nnz, const u32x4 *__restrict__ cache,
                                                 uint64_t cache_rows, const u32x4 *__restrict__ host, uint64_t host_rows,
                                                 u32x4 *__restrict__ out, uint32_t vpr, int combiner, bool bf16,
                                                 uint32_t *status, uint32_t *host_mirror, const Ending<STORE> &done,
                                                 uint32_t &wave_local, uint32_t &wave_host) {
  constexpr int kGroups = kBlock / G;
  constexpr uint32_t kTileChunks = kFewTileBytes / 16 / kGroups;
  constexpr int U = kTileChunks / G;           // chunks on their way per lane
  constexpr int EPW = sizeof(E) == 4 ? 1 : 2;  // elements per word
  constexpr int kMaxWords = 4;                 // words of a row a lane may own: rows of up to G chunks
  __shared__ u32x4 tiles[kGroups][kTileChunks];
  __shared__ uint64_t rows_at[kGroups][G];  // where the id's row is read, kNoRowBit: it has none
  __shared__ float weights_of[kGroups][G];
  __shared__ float denominators[kGroups];
  const uint32_t tid = threadIdx.x % G, group = threadIdx.x / G, words = vpr * 4;
  u32x4 *tile = tiles[group];
  uint64_t *row_at = rows_at[group];
  float *weight = weights_of[group];
  auto sync = [] {  // between the lanes of the group
    if constexpr (G == kBlock) {
      __syncthreads();
    } else {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
  };
  const uint32_t tile_rows = min(kTileChunks / vpr, (uint32_t)G);  // (8 at least)
  const uint32_t magic = vpr > 1 ? (uint32_t)(0x100000000ull / vpr) + 1u : 0u;  // i / vpr = mulhi(i, magic) for i < kTileChunks
  // sums of weights per sample, the order that pool_samples' shapes for rows of this length keep
  const uint32_t parts = vpr <= 32 ? 8 : vpr <= 128 ? 32 : 64;
  for (size_t r = (size_t)blockIdx.x * kGroups + group; r < n_rows; r += (size_t)gridDim.x * kGroups) {
    long long beg = seg_off[r], end = seg_off[r + 1];
    const bool bad = beg < 0 || end > nnz || end < beg;  // outside the ids: nothing is read for it, its row is zeros
    if (tid == 0 && (bad || (r == 0 && beg != 0) || (r + 1 == n_rows && end != nnz))) {
      atomicOr(status, UGK_ST_BAD_SEGMENT);
      if (host_mirror) tell_host<uint32_t>(host_mirror, UGK_ST_BAD_SEGMENT);
    }
    if (bad) beg = end = 0;
    float acc[kMaxWords][EPW] = {};
    float wsum = 0.f;
    for (long long j0 = beg; j0 < end; j0 += G) {  // the same for all lanes of the group
      const long long j = j0 + tid;
      const bool active = j < end;
      const uint64_t key = active ? key_to_u64<K>(ids[j]) : 0;
      const float w_of_id = active && weights ? weights[j] : 1.f;
      const Found f = table_lookup<KIND>(t, key, active);
      const MixRow row = mix_resolve(t, key, active, f, cache, cache_rows, host, host_rows, out, vpr, status, host_mirror);
      if (done.words) {
        wave_local += __popcll(__ballot(row.from_cache));
        wave_host += __popcll(__ballot(active && !row.from_cache));
      }
      const bool use = active && row.has_row;  // a key without a row adds nothing (the launch is flagged)
      row_at[tid] = use ? row.bits : row.bits | kNoRowBit;
      weight[tid] = use ? w_of_id : 0.f;
      sync();
      const uint32_t here = (uint32_t)min((long long)G, end - j0);
      if (combiner != 0 && tid < parts)
        for (uint32_t i = tid; i < here; i += parts) {
          const float w = weight[i];
          const float wterm = combiner == 2 ? w * w : w;
          wsum += wterm;
        }
      for (uint32_t i0 = 0; i0 < here; i0 += tile_rows) {
        const uint32_t rows = min(tile_rows, here - i0), chunks = rows * vpr;
        // (a lane past the end reads the last chunk again instead of branching around its load)
        auto fetch = [&](auto n) {
          u32x4 v[n()];
          bool none[n()];
#pragma unroll
          for (int u = 0; u < n(); ++u) {
            const uint32_t i = min((uint32_t)u * G + tid, chunks - 1);
            const uint32_t q = vpr > 1 ? __umulhi(i, magic) : i;
            const uint64_t at = row_at[i0 + q];
            none[u] = (at & kNoRowBit) != 0;
            v[u] = reinterpret_cast<grow_t>(at & ~(uint64_t)kNoRowBit)[i - q * vpr];
          }
#pragma unroll
          for (int u = 0; u < n(); ++u) {
            const uint32_t i = (uint32_t)u * G + tid;
            if (i < chunks) tile[i] = none[u] ? u32x4{0, 0, 0, 0} : v[u];
          }
        };
        if (chunks <= 2 * G) fetch(std::integral_constant<int, 2>{});
        else fetch(std::integral_constant<int, U>{});
        sync();
#pragma unroll
        for (int c = 0; c < kMaxWords; ++c) {
          const uint32_t word = (uint32_t)c * G + tid;
          if (word >= words) break;
          const uint32_t *column = reinterpret_cast<const uint32_t *>(tile) + word;
#pragma unroll 8
          for (uint32_t i = 0; i < rows; ++i) {
            float x[EPW];
            pool_unpack_word<E>(column[i * words], x, bf16);
#pragma unroll
            for (int e = 0; e < EPW; ++e) acc[c][e] = fmaf(weight[i0 + i], x[e], acc[c][e]);
          }
        }
        sync();  // the next rows, the next ids' rows and weights
      }
      if constexpr (STORE == kThrough) {
        if (active) copy_key_along<K>(done, (uint64_t)j, (K)key);
      }
    }
    float denom = 1.f;
    if (combiner != 0) {
      if (tid < (uint32_t)kWave) {
        for (uint32_t d = parts / 2; d > 0; d >>= 1) wsum += __shfl_xor(wsum, d);
        if (tid == 0) denominators[group] = combiner == 1 ? wsum : sqrtf(wsum);
      }
      sync();
      denom = denominators[group];
    }
    uint32_t *to = reinterpret_cast<uint32_t *>(out + r * vpr);
#pragma unroll
    for (int c = 0; c < kMaxWords; ++c) {
      const uint32_t word = (uint32_t)c * G + tid;
      if (word < words) {
        float y[EPW];
#pragma unroll
        for (int e = 0; e < EPW; ++e) y[e] = denom != 0.f ? acc[c][e] / denom : 0.f;  // div_no_nan
        const uint32_t packed = pool_pack_word<E>(y, bf16);
        if constexpr (STORE == kThrough) store_through(reinterpret_cast<uint64_t>(to + word), packed);
        else to[word] = packed;
      }
    }
    sync();  // the next sample's denominator
  }
}

// CH 0: a sample per LPR lanes, a wavefront or the workgroup (pool_few_samples)
template <typename K, int KIND, int LPR, int CH, int U, typename E, bool CLIP, bool MIXED, Store STORE>
__global__ __launch_bounds__(kBlock) void extract_pool_kernel(ugk_table_t t, const K *__restrict__ ids,
                                                              const long long *__restrict__ seg_off,
                                                              const float *__restrict__ weights, size_t n_rows,
                                                              long long nnz, const u32x4 *__restrict__ cache,
                                                              uint64_t cache_rows,
                                                              const u32x4 *__restrict__ host, uint64_t host_rows,
                                                              u32x4 *__restrict__ out, uint32_t vpr, int combiner, bool bf16,
                                                              float max_norm, uint32_t *status, uint32_t *host_mirror,
                                                              Ending<STORE> done, uint32_t keep_waves) {
  __shared__ uint32_t block_tot[2];
  if (threadIdx.x < 2) block_tot[threadIdx.x] = 0;
  __syncthreads();
  uint32_t wave_local = 0, wave_host = 0;
  if constexpr (CH == 0)
    pool_few_samples<K, KIND, LPR, E, STORE>(t, ids, seg_off, weights, n_rows, nnz, cache, cache_rows, host, host_rows, out, vpr,
                                        combiner, bf16, status, host_mirror, done, wave_local, wave_host);
  else if (!MIXED || wave_in_block() < keep_waves)
    pool_samples<K, KIND, LPR, CH, U, E, CLIP, true, STORE>(t, ids, seg_off, weights, n_rows, nnz, cache, cache_rows, host,
                                                            host_rows, out, vpr, combiner, bf16, max_norm, status,
                                                            host_mirror, done, wave_local, wave_host);
  else if constexpr (MIXED)
    pool_samples<K, KIND, LPR, CH, U, E, CLIP, false, STORE>(t, ids, seg_off, weights, n_rows, nnz, cache, cache_rows, host,
                                                             host_rows, out, vpr, combiner, bf16, max_norm, status,
                                                             host_mirror, done, wave_local, wave_host);
  if (done.words) mix_leave_counts(block_tot, wave_local, wave_host, done);
}

constexpr int kPoolMaxRows = 8;  // output rows a lane group may own per pass

// The same for short segments.  A lane group owns `rows_per_group` consecutive output rows per pass and walks their
// ids as one list: position f of the list is id seg_beg[k] + (f - seg_start[k]) of the group's row k, the last k whose
// seg_start is <= f.  The lanes resolve LPR positions at a time; the rows behind them are then read U at a time
// whatever segments they belong to and added in the order of the list, an output row being written when the list
// moves on to a later one.  What keeps memory busy is then the number of ids, not the shape of the segments: with one
// row per group a sample of one id leaves most of the group's lookups and loads unused.  The bookkeeping costs
// registers (three wavefronts per SIMD instead of four) and a lane's chunks are read one after the other, so it is not
// for flat tables, behind which rows come over the host link: 60 % of the table uncached behind a flat table, 262,144 samples
// of one id over rows of 512 bytes, 123 against 98 us with one row per group; behind a hash table, whose lookup works on all
// lanes of a wavefront at once and wants them to hold ids, 195,312 of them 107 against 128 us.  (Without any table the rule
// in extract_pool_lpr says which rows it is for.)
template <typename K, int KIND, int LPR, typename E, bool KEEP>
__device__ __forceinline__ void pool_short_samples(const ugk_table_t &t, const K *__restrict__ ids,
                                                   const long long *__restrict__ seg_off,
                                                   const float *__restrict__ weights, size_t n_rows, long long nnz,
                                                   int rows_per_group, const u32x4 *__restrict__ cache,
                                                   uint64_t cache_rows, const u32x4 *__restrict__ host,
                                                   uint64_t host_rows, u32x4 *__restrict__ out, uint32_t vpr,
                                                   int combiner, bool bf16, uint32_t *status, uint32_t *host_mirror,
                                                   const unsigned long long *counts, uint32_t &wave_local,
                                                   uint32_t &wave_host,
                                                   long long (&seg_beg)[kWavesPerBlock][kWave / LPR][kPoolMaxRows],
                                                   uint32_t (&seg_start)[kWavesPerBlock][kWave / LPR][kPoolMaxRows]) {
  constexpr int RPW = kWave / LPR;  // lane groups per wavefront
  constexpr int EPC = PoolElem<E>::kPerChunk;
  constexpr int U = 4;  // rows in flight per lane group
  static_assert(LPR % U == 0 && LPR >= kPoolMaxRows, "ids are taken in rounds of U; a lane per owned row");
  const int lane = (int)lane_id();
  const int sub = lane % LPR, rg = lane / LPR, wv_in_block = (int)(threadIdx.x / kWave);
  const size_t wave_global = (size_t)blockIdx.x * kWavesPerBlock + wv_in_block;
  const size_t n_waves = (size_t)gridDim.x * kWavesPerBlock;
  const size_t rows_per_wave = (size_t)RPW * rows_per_group;
  long long *my_beg = seg_beg[wv_in_block][rg];
  uint32_t *my_start = seg_start[wv_in_block][rg];
  for (size_t row0 = wave_global * rows_per_wave; row0 < n_rows; row0 += n_waves * rows_per_wave) {  // wavefront-uniform
    const size_t g0 = row0 + (size_t)rg * rows_per_group;  // the group's first row
    const int n_own = g0 < n_rows ? (int)min((size_t)rows_per_group, n_rows - g0) : 0;
    long long beg = 0;
    uint32_t len = 0;
    if (sub < n_own) {
      const long long b = seg_off[g0 + sub], e = seg_off[g0 + sub + 1];
      // a segment outside the ids: nothing is read for it, its row is zeros.  (The list of a group is counted in 32
      // bits; the launcher keeps batches of 2^28 ids and more away from this kernel, so the last test never fires.)
      if (b < 0 || e > nnz || e < b || e - b >= (1ll << 28)) {
        atomicOr(status, UGK_ST_BAD_SEGMENT);
        if (host_mirror) tell_host<uint32_t>(host_mirror, UGK_ST_BAD_SEGMENT);
      } else {
        beg = b, len = (uint32_t)(e - b);
        if ((g0 + sub == 0 && b != 0) || (g0 + sub + 1 == n_rows && e != nnz)) {  // the ids are not covered end to end
          atomicOr(status, UGK_ST_BAD_SEGMENT);
          if (host_mirror) tell_host<uint32_t>(host_mirror, UGK_ST_BAD_SEGMENT);
        }
      }
    }
    uint32_t incl = len;  // inclusive prefix over the group's rows (lanes past the owned rows add nothing)
#pragma unroll
    for (int d = 1; d < kPoolMaxRows; d <<= 1) {
      const uint32_t up = (uint32_t)__shfl_up((int)incl, d, LPR);
      if (sub >= d) incl += up;
    }
    const uint32_t total = (uint32_t)__shfl((int)incl, rg * LPR + kPoolMaxRows - 1);  // ids of the group this pass
    if (sub < kPoolMaxRows) my_beg[sub] = beg, my_start[sub] = incl - len;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    float acc[kPoolChunks][EPC];
#pragma unroll
    for (int c = 0; c < kPoolChunks; ++c)
#pragma unroll
      for (int e = 0; e < EPC; ++e) acc[c][e] = 0.f;
    int cur = 0;       // the owned row the accumulators belong to
    float wsum = 0.f;  // its sum of weights (or of their squares) so far
    // one chunk of an owned row is complete: divide (div_no_nan), write, start the next row
    auto flush = [&](int c, uint32_t col, int k, float ws) {
      const float denom = combiner == 1 ? ws : combiner == 2 ? sqrtf(ws) : 1.f;
      float y[EPC];
#pragma unroll
      for (int e = 0; e < EPC; ++e) y[e] = denom != 0.f ? acc[c][e] / denom : 0.f, acc[c][e] = 0.f;
      out[(g0 + k) * vpr + col] = PoolElem<E>::pack(y, bf16);
    };
    for (uint32_t f0 = 0; __ballot(f0 < total) != 0ull; f0 += LPR) {  // until every group of the wavefront is through
      const uint32_t f = f0 + sub;
      const bool active = f < total;
      int k = 0;
      if (rows_per_group > 1) {
#pragma unroll
        for (int q = 1; q < kPoolMaxRows; ++q) k += my_start[q] <= f ? 1 : 0;  // rows past the owned ones start at total
      }
      const long long j = active ? my_beg[k] + (long long)(f - my_start[k]) : 0;
      const uint64_t key = active ? key_to_u64<K>(ids[j]) : 0;
      const Found fd = table_lookup<KIND>(t, key, active);
      const MixRow row = mix_resolve(t, key, active, fd, cache, cache_rows, host, host_rows, out, vpr, status, host_mirror);
      if (counts) {
        wave_local += __popcll(__ballot(row.from_cache));
        wave_host += __popcll(__ballot(active && !row.from_cache));
      }
      const bool use = active && row.has_row;  // a key without a row adds nothing (the launch is flagged)
      const float w = use ? (weights ? weights[j] : 1.f) : 0.f;
      const int meta = active ? (k | (use ? 0x100 : 0) | 0x200) : 0;  // owned row, "adds something", "is an id"
      for (int s0 = 0; s0 < LPR; s0 += U) {
        if (__ballot(active && sub >= s0) == 0ull) break;  // no group has an id left in this round
        grow_t p[U];
        float wv[U];
        int m[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int src = rg * LPR + s0 + u;
          p[u] = reinterpret_cast<grow_t>(shfl64(row.bits, src));
          wv[u] = __shfl(w, src);
          m[u] = __shfl(meta, src);
        }
#pragma unroll
        for (int c = 0; c < kPoolChunks; ++c) {
          const uint32_t col = (uint32_t)c * LPR + sub;
          if (col < vpr) {
            u32x4 v[U];
#pragma unroll
            for (int u = 0; u < U; ++u) v[u] = KEEP ? p[u][col] : __builtin_nontemporal_load(p[u] + col);
            int cc = cur;  // every chunk walks the same ids from the same state
            float ws = wsum;
#pragma unroll
            for (int u = 0; u < U; ++u) {
              float x[EPC];
              PoolElem<E>::unpack(v[u], x, bf16);
              if (m[u] & 0x200) {
                for (const int ku = m[u] & 0xff; cc < ku; ++cc, ws = 0.f) flush(c, col, cc, ws);
                if (m[u] & 0x100) {
#pragma unroll
                  for (int e = 0; e < EPC; ++e) acc[c][e] = fmaf(wv[u], x[e], acc[c][e]);
                  ws += combiner == 2 ? wv[u] * wv[u] : wv[u];
                }
              }
            }
          }
        }
        // the state after these ids, for the lanes of every chunk alike (a lane may own no chunk at all)
#pragma unroll
        for (int u = 0; u < U; ++u) {
          if (m[u] & 0x200) {
            if (cur < (m[u] & 0xff)) cur = m[u] & 0xff, wsum = 0.f;
            if (m[u] & 0x100) wsum += combiner == 2 ? wv[u] * wv[u] : wv[u];
          }
        }
      }
    }
    // the row the list ended in, and the empty ones behind it
#pragma unroll
    for (int c = 0; c < kPoolChunks; ++c) {
      const uint32_t col = (uint32_t)c * LPR + sub;
      if (col < vpr) {
        float ws = wsum;
        for (int cc = cur; cc < n_own; ++cc, ws = 0.f) flush(c, col, cc, ws);
      }
    }
    __builtin_amdgcn_wave_barrier();  // the next pass rewrites the group's list
  }
}

template <typename K, int KIND, int LPR, typename E, bool MIXED>
__global__ __launch_bounds__(kBlock) void extract_pool_rows_kernel(ugk_table_t t, const K *__restrict__ ids,
                                                              const long long *__restrict__ seg_off,
                                                              const float *__restrict__ weights, size_t n_rows,
                                                              long long nnz, int rows_per_group,
                                                              const u32x4 *__restrict__ cache, uint64_t cache_rows,
                                                              const u32x4 *__restrict__ host, uint64_t host_rows,
                                                              u32x4 *__restrict__ out, uint32_t vpr, int combiner, bool bf16,
                                                              uint32_t *status, uint32_t *host_mirror,
                                                              unsigned long long *counts, uint32_t keep_waves) {
  __shared__ uint32_t block_tot[2];
  __shared__ long long seg_beg[kWavesPerBlock][kWave / LPR][kPoolMaxRows];    // first id of the group's row k
  __shared__ uint32_t seg_start[kWavesPerBlock][kWave / LPR][kPoolMaxRows];   // its first position in the group's list
  if (threadIdx.x < 2) block_tot[threadIdx.x] = 0;
  __syncthreads();
  uint32_t wave_local = 0, wave_host = 0;
  if (!MIXED || wave_in_block() < keep_waves)
    pool_short_samples<K, KIND, LPR, E, true>(t, ids, seg_off, weights, n_rows, nnz, rows_per_group, cache, cache_rows,
                                              host, host_rows, out, vpr, combiner, bf16, status, host_mirror, counts,
                                              wave_local, wave_host, seg_beg, seg_start);
  else if constexpr (MIXED)
    pool_short_samples<K, KIND, LPR, E, false>(t, ids, seg_off, weights, n_rows, nnz, rows_per_group, cache, cache_rows,
                                               host, host_rows, out, vpr, combiner, bf16, status, host_mirror, counts,
                                               wave_local, wave_host, seg_beg, seg_start);
  if (counts) mix_leave_counts(block_tot, wave_local, wave_host, Ending<kOrdinary>(counts));
}

template <typename K, int KIND, typename E>
int extract_pool_lpr(ugk_table_t t, const K *ids, const long long *seg_off, const float *weights, size_t n_rows,
                     const void *cache, uint64_t cache_rows, const void *host, uint64_t host_rows, void *out,
                     uint32_t vpr, uint64_t nnz, int combiner, bool bf16, float max_norm, uint32_t *status,
                     uint32_t *host_mirror, uint64_t *counts, uint32_t *num_groups, DoneRequest &request, hipStream_t st) {
  // Lanes per output row, chunks per lane and ids in flight (LPR, CH, U).  The fewest lanes that hold a row with the
  // fewest registers are best for few ids per sample (a lane group resolves LPR ids at a time and keeps U rows on
  // their way, and both are wasted on a sample that has fewer), more lanes and more rows in flight for many.  us per
  // call, rows in HBM, Zipf 1.05, about 400,000 ids (200,000 of 1 KB, 100,000 of 2 KB), by ids per sample:
  //   64 B    (8,4,4) / (4,1,2) / (4,1,4):              2 ids 76 / 34 / 38,  4: 65 / 33 / 35,  8: 41 / 29 / 29,
  //                                                     40: 37 / 41 / 37;  1 id 43 with (4,1,2), 51 with (4,1,4)
  //   128 B   (8,4,4) / (8,1,2) / (8,1,4):              2 ids 68 / 41 / 42,  4: 58 / 40 / 38,  40: 34 / 41 / 33
  //   256 B   (8,4,4) / (8,2,2) / (16,2,4):             2 ids 73 / 45 / 82,  8: 42 / 36 / 43,  40: 39 / 42 / 34
  //           many ids, 800,000 of them, Zipf / uniform, no branch around the loads: (16,2,4), whose second chunk is past the
  //           end of these rows (their last chunk again, for nothing), then (16,1,4), then (16,1,2): 16 ids 29 / 45, 24 / 42,
  //           26 / 46; 40 ids 31 / 45, 20 / 40, 22 / 40; of two-byte elements 16 ids 35 / 48, 26 / 45, 24 / 43; 40 ids
  //           32 / 44, 27 / 44, 24 / 40.  Where rows come over the host link (16,1,4) keeps more of them on their way
  //   512 B   (8,4,4) / (8,4,2) / (16,2,2) / (16,2,4):  2 ids 93 / 74 / 82 / 100,  4: 80 / 75 / 77 / 84,
  //                                                     8: 49 / 46 / 47 / 49,  40: 48 / 57 / 44 / 40
  //   512 B of two-byte elements, the same:             2 ids 68 / 61 / 54 / 67,  8: 43 / 45 / 38 / 39,
  //                                                     40: 53 / 63 / 45 / 41
  //   1 KB    (32,4,4) / (16,4,2) / (32,2,4):           2 ids 130 / 72 / 97,  8: 57 / 47 / 49,  40: 49 / 56 / 39
  //   2 KB    (32,4,4) / (32,4,2):                      2 ids 91 / 68,  8: 49 / 44,  40: 46 / 41
  // and with 512-byte rows over the host link among them, (8,4,4) / (8,4,2) / (16,2,4): 4 ids 115 / 110 / 89, 16 ids
  // 394 / 387 / 279.
  // (These were taken with a branch around the loads of each chunk; without it the chosen shapes gained another 5 to 25 %,
  // and (8,4,4) with its chunks one after the other stayed behind them: 64-byte rows aside, it ran at 0.81 to 1.31 of the speed
  // of the kernel this replaces, the chosen shapes at 0.79 to 1.60, the low ends for uniform ids.)
  const uint64_t rows64 = n_rows;
  const bool upto2 = nnz <= rows64 * 5 / 2, upto6 = nnz <= rows64 * 6, upto12 = nnz <= rows64 * 12;
  const bool clip = max_norm > 0.f;
  int shape;
  uint32_t keep_waves = kWavesPerBlock;
  if (clip) shape = vpr <= 32 ? 844 : vpr <= 128 ? 3244 : 6444;
  else if (vpr <= 4) shape = upto6 ? 412 : nnz <= rows64 * 24 ? 414 : 814;
  else if (vpr <= 8) shape = 814;
  else if (vpr <= 16) shape = upto12 ? 822 : KIND == 0 && sizeof(E) == 2 ? 1612 : 1614;
  else if (vpr <= 32) shape = upto2 && sizeof(E) == 4 ? 842 : upto12 ? 1622 : 1624;
  else if (vpr <= 64) shape = upto12 ? 1642 : 3224;
  else if (vpr <= 128) shape = 3242;
  else shape = 6442;
  // Rows all in HBM whose ordinary loads cost uniform ids something: some wavefronts load them non-temporally (see
  // pool_samples), in a shape that makes up for what that costs skewed ones.  800,000 ids out of 2 GiB, fp32, without the
  // hint / this, uniform and Zipf 1.05 (all loads non-temporal and one chunk at a time, before either): 384 bytes 4 ids
  // 76.9 / 68.5 and 56.2 / 52.1 (71.4 and 62.4), 8 ids 68.6 / 62.7 and 39.2 / 38.9 (66.1 and 51.0), 40 ids 60.3 / 53.4 and
  // 35.1 / 29.3 (55.8 and 44.7); 512 bytes 2 ids 119.7 / 111.2 and 88.7 / 87.0 (116.1 and 121.6), 4 ids 99.6 / 86.8 and 61.3 /
  // 60.7 (92.0 and 81.5), 6 ids 92.9 / 83.8 and 50.5 / 50.6 (91.3 and 75.6), 40 ids 78.6 / 70.9 and 40.2 / 36.9 (73.0 and
  // 55.4); out of 6 GiB 4 ids 105 / 89 and 64 / 62 (92 and 80).  Left alone, for it takes from skewed ids what it gives uniform
  // ones: 512 bytes 8 ids (89.6 and 45.1; 85.5 and 66.1 before; 94 and 47, 86 and 68 out of 6 GiB) and 16 ids (81 and 38; 80
  // and 62; 88 and 40, 80 and 63 out of 6 GiB), 400,000 ids of 1 KB 4 ids (98.8 / 91.5 and 55.6 / 58.3; 92.1 and 85.6 before)
  // and 8 ids (89.3 and 43.4; 85.1 and 66.8), of 2 KB 4 ids (192 and 116; 176 and 151).  Rows of other lengths, which begin
  // and end inside a line, are faster for uniform ids as well with ordinary loads (400 bytes 4 ids 95 against 128).
  if (KIND == 0 && !clip && vpr > 16 && vpr <= 32 && vpr % 8 == 0) {
    if (upto2) keep_waves = vpr == 32 && sizeof(E) == 4 ? 1 : keep_waves;
    else if (upto6) shape = 842, keep_waves = vpr == 32 && nnz <= rows64 * 9 / 2 ? 1 : 2;
    else if (upto12 && vpr < 32) shape = 842, keep_waves = 3;
    else if (nnz > rows64 * 24 && sizeof(E) == 4) shape = 1622, keep_waves = 3;
  }
  // Launches of few samples are a sample's own time, on a chip that has wavefronts to spare: more lanes per sample, and a
  // sample per wavefront or workgroup from 12 ids on (pool_few_samples).  us per launch, rows in HBM, uniform ids, mean:
  //   lanes, as above / as here: 64 B 8 ids x 4,096 5.0 / 4.4, 16 ids x 8,192 7.6 / 6.4, x 16,384 10.4 / 9.6; 256 B 8 ids x 1,024
  //     4.3 / 3.7, x 4,096 5.6 / 4.8 (x 16,384 9.1 / 8.9, 2 ids x 8,192 4.1 / 4.5); 512 B 4 ids x 1,024 5.8 / 3.8, x 4,096 6.4 / 5.0,
  //     x 8,192 7.6 / 6.4 (x 32,768 16.8 / 17.9); 512 B 40 ids x 4,096 22.5 / 19.4, x 8,192 30.2 / 31.2; 1 KB 8 ids x 1,024 6.9 /
  //     5.5, x 4,096 9.7 / 9.0 (x 8,192 15.3 / 15.5)
  //   a workgroup per sample, lanes as here / this: 512 B 16 ids x 256 5.3 / 4.1, x 1,024 6.7 / 5.8, 40 ids x 64 11.4 / 5.0, x 1,024
  //     12.2 / 8.0, 100 ids x 64 39.3 / 7.2; 1 KB 16 ids x 256 6.2 / 4.8, x 1,024 7.2 / 7.1, 40 ids x 1,024 14.4 / 11.3 (8 ids 5.5 /
  //     5.8); 2 KB 8 ids x 256 6.5 / 5.1, x 1,024 7.7 / 7.8, 40 ids x 256 18.5 / 9.1; 4 KB 16 ids x 512 11.3 / 10.7 (x 1,024 15.4 /
  //     16.6; of two-byte elements, whose words are two sums each, 16 ids x 64 10.2 / 9.9, 8.9 / 9.6 for 16 samples)
  //   a wavefront per sample: 64 B 16 ids x 1,024 4.7 / 4.2, x 2,048 5.7 / 4.8, 40 ids x 4,096 11.7 / 8.7; 256 B 16 ids x 2,048 5.4 /
  //     5.8 (two-byte 7.7 / 6.5), 40 ids x 2,048 9.8 / 8.0, x 4,096 13.0 / 11.3; 512 B 40 ids x 2,048 15.1 / 11.8
  const uint64_t cus = (uint64_t)cu_count();
  if (!clip) {
    if (vpr <= 4 && !upto6 && rows64 <= cus * 64) shape = 814;
    else if (vpr > 8 && vpr <= 16 && rows64 <= cus * 16) shape = KIND == 0 && sizeof(E) == 2 ? 1612 : 1614;
    else if (vpr > 16 && vpr <= 32 && rows64 <= cus * 32 && (keep_waves < kWavesPerBlock || upto2))
      shape = nnz <= rows64 * 24 ? 1622 : 1624, keep_waves = kWavesPerBlock;
    else if (vpr > 32 && vpr <= 64 && rows64 <= cus * 16) shape = 3224;
    const bool over24 = nnz > rows64 * 24;
    const bool by_workgroup = rows64 <= cus * 2 ? (vpr <= 64 ? !upto12 : vpr <= 128 ? !upto6 : !upto12 && sizeof(E) == 4)
                                                : rows64 <= cus * 4 && vpr > 16 && vpr <= 128 && !upto12;
    const bool by_wave = vpr <= 16 ? rows64 <= cus * 16 && (over24 || (!upto12 && rows64 <= cus * 8 && (vpr <= 8 || sizeof(E) == 2)))
                                   : vpr <= 32 && rows64 <= cus * 8 && over24;
    if (by_workgroup) shape = kBlock * 100, keep_waves = kWavesPerBlock;
    else if (by_wave) shape = kWave * 100, keep_waves = kWavesPerBlock;
  }
  if (const char *forced = getenv("UGK_POOL_LPR")) {  // for sweeps; a weighted mean's last bits may vary with it
    const int v = atoi(forced);
    if (!clip && (v == 8 || v == 32 || v == 64) && vpr <= (uint32_t)v * kPoolChunks)
      shape = v * 100 + 42, keep_waves = kWavesPerBlock;
  }
  // Output rows per lane group and pass: one, but four as one list (extract_pool_rows_kernel) for samples of mostly one
  // id without a flat table (see there), as long as the launch still has wavefronts for every CU.  Without any table that
  // is for two-byte elements of more than 64 bytes (two of 256 bytes: 127 us one by one, 107 as a list), and for fp32 rows
  // of whole lines up to 384 bytes.  The other fp32 rows are faster one by one, 800,000 samples (400,000 from 640 bytes
  // on) uniform and Zipf 1.05, list / one by one: 64 bytes 54 / 37 and 48 / 31, 160 bytes 95 / 81 and 81 / 72, 400 bytes
  // 239 / 165 and 186 / 167, 512 bytes 179 / 169 and 169 / 162, 1 KB 184 / 165 and 183 / 164, 2 KB 329 / 322 and 318 / 318.
  // (an output that does not fit the memory-side cache is not written through: 131,072 samples of one id of 2 KB 120 -> 122 us;
  // nor does the list kernel below leave words: the choice of stores where it writes a row cost it a quarter of its speed)
  const uint64_t polled_nnz = n_rows * (size_t)vpr * 16 <= kMemorySideCacheBytes ? nnz : ~0ull;
  int rows = 1;
  if constexpr (KIND != 1) {
    const int lanes = vpr <= 32 ? 8 : vpr <= 128 ? 32 : 64;
    const int groups = kWave / lanes;
    const bool lists = KIND != 0 || (vpr > 4 && (sizeof(E) == 2 || vpr <= 8 || (vpr < 32 && vpr % 8 == 0)));
    if (n_rows && nnz <= rows64 + rows64 / 2 && lists) rows = 4;
    const size_t enough_waves = (size_t)cu_count() * 8;
    while (rows > 1 && n_rows / ((size_t)rows * groups) < enough_waves) rows /= 2;
    if (const char *forced = getenv("UGK_POOL_ROWS")) {  // for sweeps, like the one above
      const int v = atoi(forced);
      if (v >= 1 && v <= kPoolMaxRows) rows = v;
    }
    if (nnz >= ((uint64_t)1 << 28) || clip) rows = 1;  // the list is counted in 32 bits; clipping lives in the other kernel
    if (rows > 1) {
      const size_t rows_per_block = (size_t)rows * groups * kWavesPerBlock;
      const unsigned grid = clamp_grid((n_rows + rows_per_block - 1) / rows_per_block, 0);
      if (num_groups) *num_groups = grid;
      // (256 bytes uniform and Zipf 1.05, before / without the hint / one wavefront of four without: 90 / 101 / 91 and
      // 102 / 91 / 91)
      constexpr bool kMixed = KIND == 0 && sizeof(E) == 4;
      const uint32_t keep = kMixed && vpr % 8 == 0 ? 1 : kWavesPerBlock;
#define UGK_POOL_ROWS_GO(L)                                                                                            \
  hipLaunchKernelGGL((extract_pool_rows_kernel<K, KIND, L, E, kMixed>), dim3(grid), dim3(kBlock), 0, st, t, ids,       \
                     seg_off, weights, n_rows, (long long)nnz, rows, (const u32x4 *)cache, cache_rows,                 \
                     (const u32x4 *)host, host_rows, (u32x4 *)out, vpr, combiner, bf16, status, host_mirror,           \
                     reinterpret_cast<unsigned long long *>(counts), keep)
      if (lanes == 8) UGK_POOL_ROWS_GO(8);
      else if (lanes == 32) UGK_POOL_ROWS_GO(32);
      else UGK_POOL_ROWS_GO(64);
#undef UGK_POOL_ROWS_GO
      UGK_HIP(hipGetLastError());
      return 0;
    }
  }
  const size_t rows_per_block = (size_t)kBlock / (shape / 100);
  const unsigned grid = clamp_grid((n_rows + rows_per_block - 1) / rows_per_block, 0);
  // Samples of one or two ids write about as much as they read, and where that is much more than the L2s hold written-through
  // rows cost more than a ticket kernel behind the launch.  us, launch to end of poll, ticket / words, all rows in one place, one
  // id per sample: 512 bytes 31 MB 22.7 / 22.9, 64 MB 33.6 / 34.7, 120 MB 51.5 / 54.3; 1 KB 48 MB 27.7 / 26.9, 64 MB 33.3 / 33.4,
  // 120 MB 51.8 / 62.2; 2 KB 48 MB 10 % sooner, 123 MB 53.0 / 55.6; two ids 1 KB 67 MB 42.1 / 42.0, 134 MB 77.6 / 86.2; four ids 4 KB
  // 134 MB 121.0 / 118.4.  (Behind a table, half of 262,144 rows of 512 bytes over the link, 353 / 344.)
  const Telling words =
      KIND != 0 || !upto2 || n_rows * (size_t)vpr * 16 <= (size_t)64 << 20 ? Telling::kSooner : Telling::kTooLate;
  DoneWords done = request.take(grid, words, polled_nnz);
  if (!done.tag) done.words = reinterpret_cast<unsigned long long *>(counts);
  if (num_groups) *num_groups = done.tag ? 0 : grid;
  const bool mixed = keep_waves < kWavesPerBlock;
  bool launched = false;
#define UGK_POOL_GO(L, CH, U, CLIP, MIXED, STORE)                                                                      \
  hipLaunchKernelGGL((extract_pool_kernel<K, KIND, L, CH, U, E, CLIP, MIXED, STORE>), dim3(grid), dim3(kBlock), 0, st, t, \
                     ids, seg_off, weights, n_rows, (long long)nnz, (const u32x4 *)cache, cache_rows,                  \
                     (const u32x4 *)host, host_rows, (u32x4 *)out, vpr, combiner, bf16, max_norm, status, host_mirror, \
                     Ending<STORE>(done), keep_waves)
#define UGK_POOL(L, CH, U, CLIP, MIXED)                                                                                \
  if (shape == L * 100 + CH * 10 + U && clip == CLIP && mixed == MIXED) {                                              \
    launched = true;                                                                                                   \
    if (done.tag) UGK_POOL_GO(L, CH, U, CLIP, MIXED, kThrough);                                                        \
    else UGK_POOL_GO(L, CH, U, CLIP, MIXED, kOrdinary);                                                                \
  }
  UGK_POOL(kBlock, 0, 0, false, false)
  UGK_POOL(kWave, 0, 0, false, false)
  UGK_POOL(4, 1, 2, false, false)
  UGK_POOL(4, 1, 4, false, false)
  UGK_POOL(8, 1, 4, false, false)
  UGK_POOL(8, 2, 2, false, false)
  if constexpr (KIND == 0 && sizeof(E) == 2) {
    UGK_POOL(16, 1, 2, false, false)
  } else {
    UGK_POOL(16, 1, 4, false, false)
  }
  UGK_POOL(16, 2, 4, false, false)
  UGK_POOL(8, 4, 4, true, false)
  UGK_POOL(32, 4, 4, true, false)
  UGK_POOL(64, 4, 4, true, false)
  UGK_POOL(8, 4, 2, false, false)
  UGK_POOL(16, 2, 2, false, false)
  UGK_POOL(16, 4, 2, false, false)
  UGK_POOL(32, 2, 4, false, false)
  UGK_POOL(32, 4, 2, false, false)
  UGK_POOL(64, 4, 2, false, false)
  if constexpr (KIND == 0) {
    UGK_POOL(8, 4, 2, false, true)
    if constexpr (sizeof(E) == 4) {
      UGK_POOL(16, 2, 2, false, true)
    }
  }
#undef UGK_POOL
#undef UGK_POOL_GO
  UGK_REQUIRE(launched, "ugk_extract_pool: no kernel of shape %d", shape);
  UGK_HIP(hipGetLastError());
  return 0;
}

template <typename K>
int extract_pool(ugk_table_t t, const K *ids, const int64_t *seg_off, const float *weights, size_t n_rows, uint64_t nnz,
                 int combiner, int elem_bytes, const void *cache, uint64_t cache_rows, const void *host,
                 uint64_t host_rows, void *out, size_t row_bytes, float max_norm, uint32_t *status,
                 uint32_t *host_mirror, uint64_t *counts, uint32_t *num_groups, void *stream) {
  DoneRequest request;
  if (num_groups) *num_groups = 0;
  if (n_rows == 0) return 0;
  UGK_REQUIRE(!request.counted(), "ugk_extract_pool: the count of ids comes from the host");
  UGK_REQUIRE(seg_off && out && status, "ugk_extract_pool: null offsets, output or status");
  UGK_REQUIRE(max_norm >= 0.f, "ugk_extract_pool: max_norm %g is not a norm (0 = no clipping)", (double)max_norm);
  UGK_REQUIRE(nnz == 0 || ids, "ugk_extract_pool: null ids");
  UGK_REQUIRE(nnz <= (uint64_t)INT64_MAX, "ugk_extract_pool: %llu ids", (unsigned long long)nnz);
  UGK_REQUIRE((uintptr_t)counts % 8 == 0, "ugk_extract_pool: the count words must be 8-byte aligned");
  UGK_REQUIRE(combiner >= 0 && combiner <= 2, "ugk_extract_pool: combiner %d is not sum(0), mean(1) or sqrtn(2)", combiner);
  UGK_REQUIRE(elem_bytes == 4 || elem_bytes == 2 || elem_bytes == UGK_ELEM_BF16,
              "ugk_extract_pool: element code %d is not fp32 (4), fp16 (2) or bfloat16 (UGK_ELEM_BF16)", elem_bytes);
  const bool bf16 = elem_bytes == UGK_ELEM_BF16;
  UGK_REQUIRE(t.kind >= 0 && t.kind <= 3, "ugk_extract_pool: table kind %d", t.kind);
  if (t.kind != 0) UGK_REQUIRE(t.table && t.size, "ugk_extract_pool: empty table");
  if (t.kind >= 2)
    UGK_REQUIRE(t.size % (t.kind == 2 ? 8 : 16) == 0 && (uintptr_t)t.table % 128 == 0,
                "ugk_extract_pool: hash table must be 128-byte aligned with whole 128-byte lines of buckets");
  UGK_REQUIRE(cache_rows == 0 || cache, "ugk_extract_pool: null cache with %llu rows", (unsigned long long)cache_rows);
  UGK_REQUIRE(host_rows == 0 || host, "ugk_extract_pool: null host table with %llu rows", (unsigned long long)host_rows);
  const uintptr_t align = (uintptr_t)cache | (uintptr_t)host | (uintptr_t)out | (uintptr_t)row_bytes;
  UGK_REQUIRE(row_bytes > 0 && align % 16 == 0,
              "ugk_extract_pool: rows and buffers must be multiples of 16 bytes (row_bytes=%zu)", row_bytes);
  const uint32_t vpr = (uint32_t)(row_bytes / 16);
  UGK_REQUIRE(vpr <= (uint32_t)kWave * kPoolChunks, "ugk_extract_pool: rows of %zu bytes exceed %d", row_bytes,
              kWave * kPoolChunks * 16);
  const long long *so = reinterpret_cast<const long long *>(seg_off);
  hipStream_t st = as_stream(stream);
#define UGK_POOL_KIND(KIND)                                                                                          \
  (elem_bytes == 4 ? extract_pool_lpr<K, KIND, float>(t, ids, so, weights, n_rows, cache, cache_rows, host, host_rows, \
                                                      out, vpr, nnz, combiner, false, max_norm, status, host_mirror,  \
                                                      counts, num_groups, request, st)                                      \
                   : extract_pool_lpr<K, KIND, __half>(t, ids, so, weights, n_rows, cache, cache_rows, host,          \
                                                       host_rows, out, vpr, nnz, combiner, bf16, max_norm, status,    \
                                                       host_mirror, counts, num_groups, request, st))
  if (t.kind == 0) return UGK_POOL_KIND(0);
  if (t.kind == 1) return UGK_POOL_KIND(1);
  if (t.kind == 2) return UGK_POOL_KIND(2);
  return UGK_POOL_KIND(3);
#undef UGK_POOL_KIND
}

}  // namespace
}  // namespace ugk
