// Row gather kernels for gfx950: out[dst(i), :] = src[srcrow(i), :].
//
// This is pure HBM (or host-link) traffic, so the kernel is built around 16-byte lanes and many rows in
// flight rather than around arithmetic:
//   * a row of V 16-byte vectors is copied by LPR = min(64, pow2ceil(V)) adjacent lanes, so one wavefront
//     instruction moves 64/LPR whole rows as fully coalesced segments (512-B rows: 2 rows, 128-B rows: 8);
//   * every lane keeps UNROLL = 2 independent rows in flight (both loads issued before the first store) and the
//     launch uses many small workgroups of one pass each (gather_kernel has the figures of one, four and eight rows);
//   * three wavefronts of four load with the non-temporal hint (most rows of a table are touched once), the fourth
//     without it for the rows that a batch repeats (keep_waves_for has the figures and the exceptions); stores are
//     ordinary write-back stores while the output fits the 256 MiB memory-side cache, so the consumer finds it there, and
//     non-temporal beyond that or when the caller says its outputs do not stay there (ugk_set_output_hint);
//   * the grid has one workgroup per pass of rows, or is capped by the caller so a host-link gather occupies
//     only a few CUs while the HBM gather runs next to it (then the workgroups stride over the batch);
//   * rows of other lengths have two more kernels: gather_flat_kernel (any multiple of 4 bytes, see flat_copy) and
//     gather_stream_kernel (long ones that come out in the order of the keys);
//   * keys / index records are range-checked against the source's row count: a bad key sets a status bit
//     and its row is skipped instead of faulting.
#include <algorithm>
#include <cstdlib>
#include <type_traits>

#include "ugk_internal.h"
#include "ugk_mix.cuh"
#include "ugk_table.cuh"

namespace ugk {
namespace {

constexpr uint64_t kNoLimit = ~0ull;

// ---- index functors (what the reference calls IdxStore*) -------------------------------------------
struct DirectU32 {
  static constexpr bool kDense = true;  // row i goes to output row i
  typedef uint32_t key_t;
  const uint32_t *keys;
  __device__ __forceinline__ void get(size_t i, uint64_t &s, uint64_t &d) const {
    s = keys[i];
    d = i;
  }
};
struct DirectI64 {
  static constexpr bool kDense = true;
  typedef int64_t key_t;
  const int64_t *keys;
  __device__ __forceinline__ void get(size_t i, uint64_t &s, uint64_t &d) const {
    s = (uint64_t)keys[i];  // negative keys become huge and fail the range check
    d = i;
  }
};
struct ScatterU32 {
  static constexpr bool kDense = false;
  const uint32_t *keys;
  const uint32_t *dst;
  __device__ __forceinline__ void get(size_t i, uint64_t &s, uint64_t &d) const {
    s = keys[i];
    d = dst[i];
  }
};
struct ScatterI64 {
  static constexpr bool kDense = false;
  const int64_t *keys;
  const uint32_t *dst;
  __device__ __forceinline__ void get(size_t i, uint64_t &s, uint64_t &d) const {
    s = (uint64_t)keys[i];
    d = dst[i];
  }
};
struct IdxList {
  static constexpr bool kDense = false;
  const ugk_idx_t *idx;
  __device__ __forceinline__ void get(size_t i, uint64_t &s, uint64_t &d) const {
    const uint2 e = *reinterpret_cast<const uint2 *>(idx + i);  // one 8-byte load
    d = e.x;
    s = e.y;
  }
};

// which wavefronts load rows the ordinary way (keep_waves_for): a launch argument says, or, for a launch that is polled for and is over
// sooner without the code of both, all of them or none
enum Loads { kByWave, kPast, kKept };
template <Loads LOADS>
__device__ __forceinline__ bool keeps(uint32_t keep_waves) {
  return LOADS == kKept || (LOADS == kByWave && wave_in_block() < keep_waves);
}
template <bool KEEP, typename V>
__device__ __forceinline__ V ld_row(const V *p) {
  if constexpr (KEEP) return *p;
  else return __builtin_nontemporal_load(p);
}
template <typename V>
__device__ __forceinline__ void st_stream(V *p, V v) {
  __builtin_nontemporal_store(v, p);
}

// Bound by HBM.  Where the launch is more than one round of workgroups (many_groups), or a lane has several vectors of a
// row, a wavefront whose rows are all there and all good, which is every one but the batch's last, copies them without a
// branch: behind one each load waits for the one before.  Rows out of 5 GiB, us per launch with the branch / without:
// 512 bytes x 65,536 15.5 / 14.7, x 262,144 45.5 / 44.8 (6.0 TB/s); 1 KB x 32,768 15.5 / 14.7, x 262,144 83.1 / 81.5; 4 KB x 2,048
// 6.8 / 6.4, x 8,192 15.5 / 14.1, x 131,072 193 / 188; 128 bytes x 196,608 13.4 / 12.2.  A launch that is all on the chip at
// once is no faster for it and up to 5 % slower near that size: 512 bytes x 16,384 5.8 / 5.7, x 32,768 8.5 / 9.0, x 36,000
// 10.5 / 10.3, 64 bytes x 262,144 11.3 / 11.7, 128 bytes x 131,072 8.7 / 9.1.  (Of the rows of several vectors per lane 2 KB x
// 7,812 with skewed keys and 8 KB x 7,812, about half of one round, lose: 7.1 / 7.5 and 24.4 / 25.8.)  Rows in flight per lane, one / two / four /
// eight, all without: 512 bytes x 65,536 15.9 / 14.7 / 15.1 / 15.5, x 524,288 91.1 / 82.4 / 82.5 / 83.5; 4 KB x 32,768 43.4 /
// 43.4 / 51.9 / 48.4; 16 bytes x 32,768 3.8 / 4.5 / 5.8 / 9.0.
template <typename V, int LPR, int UNROLL, Store STORE, Loads LOADS, typename Idx>
__global__ __launch_bounds__(kBlock) void gather_kernel(Idx ix, const V *__restrict__ src, uint64_t src_rows,
                                                        V *__restrict__ out, uint64_t out_rows, uint32_t vpr,
                                                        const uint32_t *__restrict__ counts, uint32_t group,
                                                        bool many_groups, uint8_t keep_waves, size_t n, uint32_t *status, uint32_t *host_mirror, Ending<STORE> done) {
  size_t begin = 0, count = Idx::kDense ? launch_count(done, n) : n;
  if (counts) {
    const uint32_t c = counts[group];
    count = c;
    begin = (group == UGK_LOC_LOCAL) ? 0 : n - c;
    if (host_mirror && blockIdx.x == 0 && threadIdx.x == 0) tell_host(host_mirror + 1 + group, c);
  }
  constexpr int RPB = kBlock / LPR;  // rows copied by one block instruction
  const uint32_t lane = threadIdx.x % LPR;
  const uint32_t rib = threadIdx.x / LPR;
  constexpr size_t kPerIter = (size_t)RPB * UNROLL;

  for (size_t base = (size_t)blockIdx.x * kPerIter; base < count; base += (size_t)gridDim.x * kPerIter) {
    // the index words of all rows of the pass first, in flight together (a row past the end takes the last one's),
    // then the checks: a check between two of them would make the second wait for the first
    uint64_t s[UNROLL], d[UNROLL];
    bool ok[UNROLL];
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      const size_t r = base + (size_t)u * RPB + rib;
      ok[u] = r < count;
      ix.get(begin + (ok[u] ? r : count - 1), s[u], d[u]);
    }
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      if (ok[u] && (s[u] >= src_rows || d[u] >= out_rows)) {
        ok[u] = false;
        if (lane == 0) {
          atomicOr(status, UGK_ST_KEY_OUT_OF_RANGE);
          if (host_mirror) tell_host<uint32_t>(host_mirror, UGK_ST_KEY_OUT_OF_RANGE);
        }
      }
    }
    bool whole = true;
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) whole = whole && ok[u];
    // (rows of up to 64 bytes gain nothing and stay as they were)
    const bool no_branch = LPR >= 8 && (many_groups || vpr > LPR) && __ballot(!whole) == 0ull;
    // (a loop of its own for each way: in one loop the compiler makes one last store of the two arms' and lets it wait for
    // the others, 5 % of a launch)
    auto copy = [&](auto keep, auto branch) {
      constexpr bool KEEP = decltype(keep)::value, BRANCH = decltype(branch)::value;
      for (uint32_t c0 = 0; c0 < vpr; c0 += LPR) {
        const uint32_t col = c0 + lane;
        if (col < vpr) {
          V v[UNROLL];
#pragma unroll
          for (int u = 0; u < UNROLL; ++u)
            if (!BRANCH || ok[u]) v[u] = ld_row<KEEP>(src + s[u] * vpr + col);
          if constexpr (BRANCH || STORE == kThrough) arrived(v);
#pragma unroll
          for (int u = 0; u < UNROLL; ++u) {
            if (BRANCH && !ok[u]) continue;
            V *to = out + d[u] * vpr + col;
            if constexpr (STORE == kThrough) store_through(reinterpret_cast<uint64_t>(to), v[u]);
            else if constexpr (STORE == kStreaming) st_stream(to, v[u]);
            else *to = v[u];
          }
        }
      }
    };
    if (keeps<LOADS>(keep_waves)) {
      if (no_branch) copy(std::true_type{}, std::false_type{});
      else copy(std::true_type{}, std::true_type{});
    } else {
      if (no_branch) copy(std::false_type{}, std::false_type{});
      else copy(std::false_type{}, std::true_type{});
    }
    if constexpr (Idx::kDense && STORE == kThrough) {
      if (base < done.num_keys)
        for (size_t i = base + threadIdx.x; i < min(base + kPerIter, count); i += kBlock)
          copy_key_along(done, i, ix.keys[i]);
    }
  }
  if constexpr (STORE == kThrough) leave_done(done, nullptr);
}

// The same for rows the lanes of gather_kernel do not fit (see flat_copy): a wavefront takes f.tile rows, one index
// word per lane, and copies their vectors numbered through.
template <Store STORE, Loads LOADS, typename Idx>
__global__ __launch_bounds__(kBlock) void gather_flat_kernel(Idx ix, const char *__restrict__ src, uint64_t src_rows,
                                                             char *__restrict__ out, uint64_t out_rows, FlatRow f,
                                                             const uint32_t *__restrict__ counts, uint32_t group,
                                                             uint8_t keep_waves, size_t n, uint32_t *status,
                                                             uint32_t *host_mirror, Ending<STORE> done) {
  size_t begin = 0, count = Idx::kDense ? launch_count(done, n) : n;
  if (counts) {
    const uint32_t c = counts[group];
    count = c;
    begin = (group == UGK_LOC_LOCAL) ? 0 : n - c;
    if (host_mirror && blockIdx.x == 0 && threadIdx.x == 0) tell_host(host_mirror + 1 + group, c);
  }
  const size_t wave = (size_t)blockIdx.x * kWavesPerBlock + wave_in_block();
  const size_t stride = (size_t)gridDim.x * kWavesPerBlock * f.tile;
  for (size_t base = wave * f.tile; base < count; base += stride) {
    const uint32_t rows = (uint32_t)min((size_t)f.tile, count - base);
    uint64_t s = 0, d = 0;
    bool ok = lane_id() < rows;
    if (ok) ix.get(begin + base + lane_id(), s, d);
    if (ok && (s >= src_rows || d >= out_rows)) {
      ok = false;
      atomicOr(status, UGK_ST_KEY_OUT_OF_RANGE);
      if (host_mirror) tell_host<uint32_t>(host_mirror, UGK_ST_KEY_OUT_OF_RANGE);
    }
    const unsigned long long good = __ballot(ok);
    if (good != 0ull) {
      // a row that is skipped is read where the tile's first good row is
      const uint64_t at = reinterpret_cast<uint64_t>(src) + s * f.row_bytes;
      const uint64_t dummy = shfl64(at, __ffsll(good) - 1);
      const uint64_t bits = ok ? at : dummy | kNoRowBit;
      if (keeps<LOADS>(keep_waves))
        flat_copy<Idx::kDense, STORE == kThrough, true>(bits, (uint32_t)d, out, base, 0, rows, f);
      else
        flat_copy<Idx::kDense, STORE == kThrough, false>(bits, (uint32_t)d, out, base, 0, rows, f);
    }
    if constexpr (Idx::kDense && STORE == kThrough) {
      if (lane_id() < rows) copy_key_along(done, base + lane_id(), (typename Idx::key_t)s);
    }
  }
  if constexpr (STORE == kThrough) leave_done(done, nullptr);
}

// ... and with the output dealt out instead of the rows, for batches whose row i becomes output row i: a wavefront owns
// kStreamPart aligned bytes of it, whichever rows those are.  Its stores are whole aligned vectors and lines, where the
// edges of flat_copy's rows are lines written in two pieces; a vector that two rows share (SHARE: rows that are no
// multiple of 16 bytes) is put together from the last vector of the one and the first vector of the other.  Bound by
// HBM: 262,144 rows of 1204 bytes 122 us (231.6 us with 4-byte lanes) for 664 MB of lines read and rows written.
constexpr uint32_t kStreamPart = kWave * 16 * 4;  // 4 vectors per lane
constexpr uint32_t kStreamMinBytes = 256;         // a part is in at most 17 rows then

struct StreamRow {
  uint32_t row_bytes;
  uint32_t magic;  // floor(2^32 / row_bytes) + 1 for rows below kStreamPart: x / row_bytes = mulhi(x, magic) for
                   // x < row_bytes + kStreamPart; 0 for longer ones, of which a part is in two at most
  uint64_t total;  // bytes of the output
};
StreamRow stream_row(size_t row_bytes, size_t n) {
  return StreamRow{(uint32_t)row_bytes, row_bytes < kStreamPart ? (uint32_t)(0x100000000ull / row_bytes) + 1u : 0u,
                   (uint64_t)n * row_bytes};
}

template <Store STORE, Loads LOADS, bool SHARE, typename Idx>
__global__ __launch_bounds__(kBlock) void gather_stream_kernel(Idx ix, const char *__restrict__ src, uint64_t src_rows,
                                                               char *__restrict__ out, StreamRow f, uint32_t *status,
                                                               uint32_t *host_mirror, Ending<STORE> done,
                                                               uint8_t keep_waves) {
  static_assert(Idx::kDense, "row i goes to output row i");
  typedef __attribute__((address_space(1))) uint32_t *gword_t;
  constexpr int U = (int)(kStreamPart / (kWave * 16));
  auto put = [](auto *q, auto w) {
    if constexpr (STORE == kThrough) store_through(reinterpret_cast<uint64_t>(q), w);
    else *q = w;
  };
  const uint32_t lane = lane_id();
  const uint64_t total = STORE == kThrough ? launch_count(done, f.total / f.row_bytes) * f.row_bytes : f.total;
  const uint64_t stride = (uint64_t)gridDim.x * kWavesPerBlock * kStreamPart;
  for (uint64_t begin = ((uint64_t)blockIdx.x * kWavesPerBlock + wave_in_block()) * kStreamPart; begin < total;
       begin += stride) {
    const uint64_t row0 = begin / f.row_bytes;
    const uint32_t off0 = (uint32_t)(begin - row0 * f.row_bytes);  // the part begins at byte off0 of row row0
    const uint32_t bytes = (uint32_t)min((uint64_t)kStreamPart, total - begin);
    const uint64_t to = reinterpret_cast<uint64_t>(out) + begin;
    // lane l: where row row0 + l is read
    uint64_t s = 0, d = 0;
    const bool active = (uint64_t)lane * f.row_bytes < (uint64_t)off0 + bytes;
    bool ok = active;
    if (ok) ix.get(row0 + lane, s, d);
    if (ok && s >= src_rows) {
      ok = false;
      atomicOr(status, UGK_ST_KEY_OUT_OF_RANGE);
      if (host_mirror) tell_host<uint32_t>(host_mirror, UGK_ST_KEY_OUT_OF_RANGE);
    }
    const unsigned long long good = __ballot(ok);
    if (good == 0ull) {
      if constexpr (STORE == kThrough) {
        if (active) copy_key_along(done, row0 + lane, (typename Idx::key_t)s);
      }
      continue;
    }
    // a row that is skipped is read where the first good one is (all lanes take part in the shuffle)
    const uint64_t mine = reinterpret_cast<uint64_t>(src) + s * f.row_bytes;
    const uint64_t dummy = shfl64(mine, __ffsll(good) - 1);
    const uint64_t at = ok ? mine : dummy;
    const uint32_t lo = (uint32_t)at | (ok ? 0u : kNoRowBit), hi = (uint32_t)(at >> 32);
    auto part = [&](auto keep) {
      constexpr bool KEEP = decltype(keep)::value;
      // the vector that row l shares with the next one is lane l's: `end` is where row l ends in the part, its last `head`
      // bytes lie in that vector (no branch around the two loads: the ones that follow would wait for them at its end)
      u32x4 sa{}, sb{};
      uint32_t head = 0, end = 0, nlo = kNoRowBit;
      if constexpr (SHARE) {
        nlo = __shfl_down(lo, 1);
        const uint32_t nhi = __shfl_down(hi, 1);
        end = (lane + 1) * f.row_bytes - off0;
        if (active && end < bytes) head = end % 16;
        sa = __builtin_nontemporal_load(reinterpret_cast<grow_by4_t>(at + f.row_bytes - 16));
        sb = __builtin_nontemporal_load(reinterpret_cast<grow_by4_t>(((uint64_t)nhi << 32) | (nlo & ~kNoRowBit)));
      }
      u32x4 v[U];
      bool copy[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint32_t i = (u * kWave + lane) * 16;
        const bool in = i + 16 <= bytes;
        const uint32_t x = off0 + (in ? i : 0u);  // a lane past the end reads the part's first vector
        const uint32_t r = max(__umulhi(x, f.magic), x >= f.row_bytes ? 1u : 0u);
        const uint32_t off = x - r * f.row_bytes;
        const uint32_t rlo = __shfl(lo, (int)r), rhi = __shfl(hi, (int)r);
        copy[u] = in && (rlo & kNoRowBit) == 0 && (!SHARE || off + 16 <= f.row_bytes);
        const grow_by4_t p = reinterpret_cast<grow_by4_t>((((uint64_t)rhi << 32) | (rlo & ~kNoRowBit)) +
                                                          (SHARE ? min(off, f.row_bytes - 16) : off));
        if constexpr (KEEP) v[u] = *p;
        else v[u] = __builtin_nontemporal_load(p);
      }
      if constexpr (STORE == kThrough) arrived(v);
      if constexpr (STORE == kThrough && SHARE) arrived(sa), arrived(sb);
      if constexpr (SHARE) {
        if (head) {
          const gout_t q = reinterpret_cast<gout_t>(to + end - head);
          const bool row_a = (lo & kNoRowBit) == 0, row_b = (nlo & kNoRowBit) == 0;
          u32x4 w;  // the last words of sa, then the first of sb
          w.x = head == 12 ? sa.y : head == 8 ? sa.z : sa.w;
          w.y = head == 12 ? sa.z : head == 8 ? sa.w : sb.x;
          w.z = head == 12 ? sa.w : head == 8 ? sb.x : sb.y;
          w.w = head == 12 ? sb.x : head == 8 ? sb.y : sb.z;
          if (row_a && row_b) {
            if constexpr (STORE == kStreaming) __builtin_nontemporal_store(w, q);
            else put(q, w);
          } else {  // a skipped row leaves its words of the output alone
            const gword_t q1 = reinterpret_cast<gword_t>(q);
            if (row_a) put(q1, (uint32_t)w.x);
            if (head > 4 ? row_a : row_b) put(q1 + 1, (uint32_t)w.y);
            if (head > 8 ? row_a : row_b) put(q1 + 2, (uint32_t)w.z);
            if (row_b) put(q1 + 3, (uint32_t)w.w);
          }
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (copy[u]) {
          const gout_t q = reinterpret_cast<gout_t>(to + (u * kWave + lane) * 16);
          if constexpr (STORE == kStreaming) __builtin_nontemporal_store(v[u], q);
          else put(q, v[u]);
        }
    };
    if (keeps<LOADS>(keep_waves)) {
      // (for the compiler alone, which makes one of two loads that differ in the hint, and that without it)
      asm volatile("" ::: "memory");
      part(std::true_type{});
      asm volatile("" ::: "memory");
    } else {
      part(std::false_type{});
    }
    if constexpr (SHARE) {
      const uint32_t rest = bytes % 16;  // the words behind the last whole vector of the output: the end of its last row
      if (rest) {
        const uint32_t r = (uint32_t)((total - 1) / f.row_bytes - row0);
        const uint32_t rlo = __shfl(lo, (int)r), rhi = __shfl(hi, (int)r);
        if (lane < rest / 4 && (rlo & kNoRowBit) == 0) {
          const uint64_t from = (((uint64_t)rhi << 32) | rlo) + f.row_bytes - rest;
          put(reinterpret_cast<gword_t>(to + bytes - rest) + lane, (uint32_t)reinterpret_cast<gword_t>(from)[lane]);
        }
      }
    }
    if constexpr (STORE == kThrough) {
      if (active) copy_key_along(done, row0 + lane, (typename Idx::key_t)s);  // a row in two parts: twice the same key
    }
  }
  if constexpr (STORE == kThrough) leave_done(done, nullptr);
}

// Re-expansion of duplicates inside one buffer: row i takes the bytes of its representative row.  Source and
// destination are the same allocation but never the same row, so the pointers are deliberately not __restrict__.
template <typename V, int LPR>
__global__ __launch_bounds__(kBlock) void replicate_kernel(V *out, uint32_t vpr, const uint32_t *__restrict__ inverse,
                                                           const uint32_t *__restrict__ rep, size_t n) {
  constexpr int RPB = kBlock / LPR;
  const uint32_t lane = threadIdx.x % LPR, rib = threadIdx.x / LPR;
  for (size_t base = (size_t)blockIdx.x * RPB; base < n; base += (size_t)gridDim.x * RPB) {
    const size_t i = base + rib;
    if (i >= n) continue;
    const size_t r = rep[inverse[i]];
    if (r == i) continue;
    for (uint32_t col = lane; col < vpr; col += LPR) out[i * vpr + col] = out[r * vpr + col];
  }
}

constexpr int kStagedUnroll = 8;  // rows a lane group keeps in flight in gather_staged_kernel
// Rows out of the host table, or out of the stage where it holds them (refresh inserts: most of the rows a refresh
// brings in were missed by the last few lookups and are filed there).  Lanes per row chosen at run time: this runs at
// refresh time, on some hundred thousand rows.
__global__ __launch_bounds__(kBlock) void gather_staged_kernel(const u32x4 *__restrict__ host, uint64_t host_rows,
                                                               const uint32_t *__restrict__ rows,
                                                               const uint32_t *__restrict__ dst, size_t n,
                                                               u32x4 *__restrict__ out, uint64_t out_rows, uint32_t vpr,
                                                               uint32_t lpr, ugk_stage_t stage, uint32_t *status,
                                                               uint32_t *staged, uint32_t *rest_rows,
                                                               uint32_t *rest_dst, uint32_t *rest_count,
                                                               uint32_t *done_count) {
  constexpr int UNROLL = kStagedUnroll;
  __shared__ uint32_t block_staged;
  if (threadIdx.x == 0) block_staged = 0;
  __syncthreads();
  const uint32_t lane = threadIdx.x % lpr, rib = threadIdx.x / lpr, rpb = kBlock / lpr;
  const size_t per_iter = (size_t)rpb * UNROLL;
  const u32x4 *stage_rows = reinterpret_cast<const u32x4 *>(stage.rows_dev);
  uint32_t mine = 0;
  for (size_t base = (size_t)blockIdx.x * per_iter; base < n; base += (size_t)gridDim.x * per_iter) {
    // three rounds of reads, each for all rows of the pass before the next: list entries, owner words, rows.  (A check or an
    // owner word between the entries of two rows made the second row's wait for the first's: 72,000 rows of 128 bytes 19.0
    // us, 16.3 this way, with eight rows in flight as with four; 21.5 with two.)
    const u32x4 *src[UNROLL];
    uint64_t s_of[UNROLL], d[UNROLL], h_of[UNROLL];
    unsigned long long owner[UNROLL];
    bool ok[UNROLL];
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      const size_t r = base + (size_t)u * rpb + rib;
      ok[u] = r < n;
      s_of[u] = rows[ok[u] ? r : n - 1];
      d[u] = dst[ok[u] ? r : n - 1];
    }
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      h_of[u] = fmix64(s_of[u]) & stage.mask;
      owner[u] = stage.owner_dev[h_of[u]];
    }
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      const uint64_t s = s_of[u], h = h_of[u];
      if (ok[u] && (s >= host_rows || d[u] >= out_rows)) {
        ok[u] = false;
        if (lane == 0) atomicOr(status, UGK_ST_KEY_OUT_OF_RANGE);
      }
      const bool filed = ok[u] && (owner[u] >> 32) != 0 && (uint32_t)owner[u] == (uint32_t)s;
      if (rest_count) {
        // Rows the stage does not hold are left for the caller's own (throttled) copy over the host link: listed, not
        // copied.  With done_count the rows that are copied here are listed too, from the back of the same lists, for
        // a caller that publishes rows as they arrive.  One atomic per wavefront and list: the first lane of every
        // row that goes on a list takes its place from a ballot.
        const bool lead = lane == 0 && ok[u];
        const unsigned long long to_rest = __ballot(lead && !filed);
        const unsigned long long to_done = __ballot(lead && filed && done_count != nullptr);
        const unsigned long long below = (1ull << lane_id()) - 1ull;
        uint32_t rest_base = 0, done_base = 0;
        if (lane_id() == 0) {
          if (to_rest) rest_base = atomicAdd(rest_count, (uint32_t)__popcll(to_rest));
          if (to_done) done_base = atomicAdd(done_count, (uint32_t)__popcll(to_done));
        }
        rest_base = __shfl(rest_base, 0);
        done_base = __shfl(done_base, 0);
        if (lead && !filed) {
          const uint32_t at = rest_base + (uint32_t)__popcll(to_rest & below);
          rest_rows[at] = (uint32_t)s;
          rest_dst[at] = (uint32_t)d[u];
        } else if (lead && filed && done_count) {
          const uint32_t at = (uint32_t)n - 1u - (done_base + (uint32_t)__popcll(to_done & below));
          rest_rows[at] = (uint32_t)s;
          rest_dst[at] = (uint32_t)d[u];
        }
        if (!filed) ok[u] = false;
      }
      src[u] = !ok[u] ? reinterpret_cast<const u32x4 *>(out) : filed ? stage_rows + h * vpr : host + s * vpr;
      if (filed && lane == 0) ++mine;
    }
    for (uint32_t c0 = 0; c0 < vpr; c0 += lpr) {
      const uint32_t col = c0 + lane;
      if (col < vpr) {
        u32x4 v[UNROLL];
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) v[u] = ld_row<false>(src[u] + col);
#pragma unroll
        for (int u = 0; u < UNROLL; ++u)
          if (ok[u]) out[d[u] * vpr + col] = v[u];
      }
    }
  }
  if (staged == nullptr) return;
  if (mine) atomicAdd(&block_staged, mine);
  __syncthreads();
  if (threadIdx.x == 0 && block_staged) atomicAdd(staged, block_staged);
}

// A launch that may fill the chip (max_blocks == 0) gets one workgroup per pass of rows, however many that makes:
// workgroups start in order, so the rows being written at any moment form one window that moves through the output,
// which the memory side turns into far better write bursts than the same workgroups striding over the whole output
// (2 M keys of 512 bytes: 360 us against 377 us with 16,384 grid-striding workgroups; 1 M keys: 181 against 187 us).
unsigned gather_grid(size_t passes, unsigned max_blocks) {
  if (max_blocks) return clamp_grid(passes, max_blocks);
  if (passes == 0) passes = 1;
  return (unsigned)(passes > 0x7fffffffull ? 0x7fffffffull : passes);
}

// A caller caps the launch for rows that come over a link, and the groups other than the local one are peers and the host.
bool over_link(const uint32_t *counts, uint32_t group, unsigned max_blocks) {
  return max_blocks != 0 || (counts && group != UGK_LOC_LOCAL);
}

// How many of a workgroup's four wavefronts load rows the ordinary way, the others past the caches.  What a wavefront
// loads past the caches keeps their room for the output, but a row that the batch repeats (keys are skewed, and a line
// holds several short rows) is fetched as often as it is asked for, through the channel where its line lives.  One
// wavefront of four is enough for the rows that come often to be found in the caches by all four, and leaves three
// quarters of the room alone.  us, 512-byte rows in HBM, none / one / four of the wavefronts, keys uniform and
// zipf 0.8 and 1.05: 8 MB 5.1 / 5.0 / 5.3 and 5.1 / 4.9 / 5.0 and 4.8 / 4.7 / 4.4; 64 MB 25.6 / 24.6 / 25.3 and
// 24.9 / 24.2 / 23.7 and 25.4 / 22.4 / 19.2; 128 MB 44.8 / 43.8 / 44.7 and 45.5 / 42.7 / 42.1 and 48.8 / 41.0 / 39.0;
// 200 MB 65.9 / 65.9 / 84.6 and 66.5 / 63.3 / 72.7; streaming stores, 290 MB 103 / 98 / 106 and 104 / 92 / 91 and
// 96 / 87 / 86.
//   * The output and the share of the lines that is kept have to fit the memory-side cache, or the lines push the output
//     out (250 MB, uniform keys: 80 none, 99 one of four); a launch with streaming stores has left it to the lines.
//   * Rows under 48 bytes, of which a line holds several: all four, at every size (32 bytes, 128 MB, uniform 113 / 108 / 106,
//     zipf 1.05 90 / 71 / 62; 4 bytes, 64 MB 371 / 312 / 317 and 248 / 180 / 136; 40 bytes, 200 MB 182 / 199 / 173).
//     Except that lines that come to about what the L2s hold, 32 MB, push the output out of there, for rows of 16 bytes and
//     more: one of four, by which uniform keys lose nothing and skewed ones gain half.  Keys that were not looked up before,
//     16 bytes, uniform, zipf 0.8 and 1.05: 131,072 5.4 / 5.4 / 5.4, 5.2 / 5.0 / 4.8 and 4.6 / 4.3 / 4.2; 180,224 6.8 / 6.9 / 6.6, 6.6 /
//     6.2 / 6.1 and 5.5 / 5.2 / 4.6; 262,144 8.2 / 8.3 / 8.6, 7.8 / 7.6 / 7.7 and 6.1 / 5.9 / 5.4; 393,216 10.9 / 11.2 / 11.4, 10.3 / 9.9 /
//     10.5 and 7.6 / 7.0 / 6.4; 458,752 12.9 / 13.0 / 13.1, 12.1 / 12.2 / 12.1 and 9.0 / 8.1 / 7.5; 700,000 19.0 / 18.7 / 18.1, 17.9 / 17.1 /
//     16.4 and 13.0 / 11.7 / 10.4.  32 bytes: 180,224 6.8 / 6.7 / 7.0 and 6.6 / 6.6 / 6.4; 262,144 9.1 / 8.9 / 9.4 and 8.6 / 8.4 / 8.8; 320,000
//     10.3 / 10.2 / 10.7 and 9.7 / 9.6 / 10.0; 458,752 14.5 / 14.1 / 13.9 and 13.2 / 13.2 / 12.6.  20 bytes (flat): 180,224 7.1 / 7.0 / 7.0;
//     262,144 8.9 / 8.9 / 9.4; 393,216 12.3 / 12.7 / 12.4; 458,752 14.3 / 14.2 / 14.0.  12 bytes: 262,144 8.1 / 8.1 / 8.4, 458,752 13.4 /
//     13.3 / 12.9.
//   * Stores that are written through need no room in the L2s, and what one wavefront of four keeps there the others, reading past
//     it, drop again: all four or none.  us, launch to end of poll, keys that were not looked up before, none / all, uniform, zipf
//     0.8, 1.05 and 1.2: 512 bytes 64 KB 9.4 / 9.5, 9.5 / 9.4, 9.5 / 9.3 and 9.4 / 9.3; 1 MB 10.1 / 10.2, 10.1 / 10.2, 10.0 / 9.9 and 10.0 /
//     9.7; 8 MB 12.7 / 12.9, 12.7 / 12.6, 12.2 / 11.8 and 12.2 / 11.0; 16 MB 15.3 / 15.5, 15.3 / 15.2, 14.7 / 14.2 and 14.6 / 12.7; 128 bytes
//     8 MB 13.4 / 13.4, 13.3 / 13.1, 12.8 / 12.5 and 12.8 / 11.6; 4 KB 64 KB 9.9 / 10.3, 10.2 / 10.0, 10.1 / 9.6 and 10.0 / 10.1; 2 MB 12.4 / 12.5,
//     12.5 / 12.5, 12.3 / 12.2 and 12.1 / 11.3.  (Uniform keys pay 1 %.)  Beyond 16 MB uniform keys pay 2 to 3 %, 32 MB 20.7 / 21.2: none
//     there; up to 10 MB for rows that begin inside a line (200 bytes, 10 MB 15.8 / 15.9, 15.7 / 15.5, 14.8 / 14.5 and 14.5 / 13.3).  Short
//     rows: 16 bytes x 262,144 16.2 / 16.3, 15.9 / 15.7 and 14.1 / 13.0, x 1,048,576 31.9 / 32.0 and, zipf 1.05, 23.8 / 20.0; 32 bytes x
//     262,144 17.1 / 17.3, 16.6 / 16.7 and 15.2 / 14.3; 36 bytes x 466,033 24.8 / 24.9 and 21.1 / 19.3, but x 5,688,888 194 / 201.
//   * Rows over a link: none, as nothing that the chip's caches do shows beside the link (that of an uncapped gather out of
//     host memory, which cannot be told from one out of HBM here: 16 to 1204 bytes x 0.25 to 8 MB 0.98 to 1.2 times as fast).
constexpr size_t kMemorySideCache = 256ull << 20;
uint8_t keep_waves_for(size_t n, size_t row_bytes, Store store, bool over_link) {
  constexpr size_t kLine = 128;
  if (over_link) return 0;
  // bytes of the lines that a row touches, on the average over where it can begin
  const size_t lines = kLine % row_bytes == 0      ? kLine
                       : row_bytes % kLine == 0    ? row_bytes
                       : row_bytes % 16 == 0       ? row_bytes + kLine - 16
                                                   : row_bytes + kLine - 4;
  if (store == kThrough) {
    const bool all = row_bytes >= 48 ? n * row_bytes <= (size_t)(row_bytes % 64 == 0 ? 16 : 10) << 20
                                     : row_bytes <= 32 || n * (row_bytes + lines) <= kMemorySideCache;
    return all ? kWavesPerBlock : 0;
  }
  const bool as_l2 = n > (22ull << 20) / kLine && n <= (56ull << 20) / kLine;
  if (row_bytes < 48) return !as_l2 || row_bytes < 16 ? kWavesPerBlock : 1;
  return store == kStreaming || n * (row_bytes + lines / kWavesPerBlock) <= kMemorySideCache ? 1 : 0;
}

// Words (ugk_leave_done_words) come sooner than a ticket kernel behind the launch would, but for rows of single bytes or pairs: a
// line that is written through does not come together in L2.  us, launch to end of poll, ticket / words, rows in HBM: 97 bytes 1 MB
// 9.9 / 10.2, 8 MB 22.8 / 27.5, 32 MB 62 / 84; 1001 bytes 1 MB 15.8 / 19.6, 8 MB 18.7 / 23.8, 32 MB 36 / 54.
// Long rows, of more than two vectors per lane, whose next loads come back behind the stores of the last: keys that were not looked
// up before, uniform: 4 KB x 1 11.4 / 9.5, x 16 11.8 / 10.8, x 512 13.1 / 12.5, x 8,192 21.7 / 20.8; 8 KB x 8 12.8 / 12.7, x 64 14.8 / 13.9, x
// 1,024 17.1 / 16.2; 16 KB x 4 15.6 / 15.7, x 64 18.9 / 18.1; 32 KB x 2 20.6 / 21.3, x 8 26.0 / 26.0, x 64 27.2 / 26.9, x 1,024 35.1 / 33.3;
// zipf 1.05 sooner by 3 to 15 %.  (Lookups of such rows through the library, 32 KB to 16 MB of them, all in HBM, 0.6 of them and none:
// 4 to 31, 1 to 19 and 1 to 12 % sooner than with a ticket, which batches that were looked up before had seemed to favour.)
// (Outputs of 6 to 10 MB, about what the wavefronts of one round copy and all written at once, are 0.1 to 0.6 us later too where
// a launch costs the host 3 us, and 0.9 us sooner where it costs 4: words there.)
template <typename V, int LPR, int UNROLL, typename Idx>
int launch_unrolled(Idx ix, const void *src, uint64_t src_rows, void *out, uint64_t out_rows, uint32_t vpr,
                    const uint32_t *counts, uint32_t group, size_t n, unsigned max_blocks, uint32_t *status,
                    uint32_t *host_mirror, bool nt, DoneRequest &request, hipStream_t stream) {
  constexpr size_t kPerIter = (size_t)(kBlock / LPR) * UNROLL;
  const unsigned grid = request.grid(gather_grid((n + kPerIter - 1) / kPerIter, max_blocks));
  const bool many_groups = grid > (unsigned)cu_count() * 8u;  // more than 32 wavefronts per CU
  DoneWords done{};
  if constexpr (Idx::kDense) {
    if (!nt) done = request.take(grid, sizeof(V) < 4 ? Telling::kTooLate : Telling::kSooner);
    UGK_REQUIRE(!request.counted(), "gather: a launch that leaves no words cannot take its count from the device");
  }
  const uint8_t keep_waves = keep_waves_for(n, (size_t)vpr * sizeof(V), done.tag ? kThrough : nt ? kStreaming : kOrdinary,
                                            over_link(counts, group, max_blocks));
#define UGK_GO(STORE, LOADS)                                                                                           \
  hipLaunchKernelGGL((gather_kernel<V, LPR, UNROLL, STORE, LOADS, Idx>), dim3(grid), dim3(kBlock), 0, stream, ix,     \
                     reinterpret_cast<const V *>(src), src_rows, reinterpret_cast<V *>(out), out_rows, vpr, counts,   \
                     group, many_groups, keep_waves, n, status, host_mirror, Ending<STORE>(done))
  if constexpr (Idx::kDense) {
    if (done.tag) {
      if (keep_waves) UGK_GO(kThrough, kKept);
      else UGK_GO(kThrough, kPast);
      UGK_HIP(hipGetLastError());
      return 0;
    }
  }
  if (nt) UGK_GO(kStreaming, kByWave);
  else UGK_GO(kOrdinary, kByWave);
#undef UGK_GO
  UGK_HIP(hipGetLastError());
  return 0;
}

template <typename V, int LPR, typename Idx>
int launch_one(Idx ix, const void *src, uint64_t src_rows, void *out, uint64_t out_rows, uint32_t vpr,
               const uint32_t *counts, uint32_t group, size_t n, unsigned max_blocks, uint32_t *status,
               uint32_t *host_mirror, DoneRequest &request, hipStream_t stream) {
  // two rows in flight per lane; one was measured with streaming stores and is no better (262,144 keys of 512 bytes
  // into rotating outputs 49.3 us against 47.9 us, 1 M keys 184 against 180 us)
  return launch_unrolled<V, LPR, 2, Idx>(ix, src, src_rows, out, out_rows, vpr, counts, group, n, max_blocks, status,
                                         host_mirror, !request.counted() && nt_store_for(n * (size_t)vpr * sizeof(V)), request,
                                         stream);
}

template <typename V, typename Idx>
int launch_vec(Idx ix, const void *src, uint64_t src_rows, void *out, uint64_t out_rows, size_t row_bytes,
               const uint32_t *counts, uint32_t group, size_t n, unsigned max_blocks, uint32_t *status,
               uint32_t *host_mirror, DoneRequest &request, hipStream_t stream) {
  const uint32_t vpr = (uint32_t)(row_bytes / sizeof(V));
#define UGK_GO(L) \
  return launch_one<V, L, Idx>(ix, src, src_rows, out, out_rows, vpr, counts, group, n, max_blocks, status, host_mirror, \
                               request, stream)
  if constexpr (sizeof(V) == 16) {
    if (vpr <= 1) UGK_GO(1);
    if (vpr <= 2) UGK_GO(2);
    if (vpr <= 4) UGK_GO(4);
    if (vpr <= 8) UGK_GO(8);
    if (vpr <= 16) UGK_GO(16);
    if (vpr <= 32) UGK_GO(32);
    UGK_GO(64);
  } else if constexpr (sizeof(V) == 8) {  // rows of 8 bytes (see launch_gather)
    UGK_GO(1);
  } else if constexpr (sizeof(V) == 4) {  // rows of up to 16 bytes, longer ones in small launches (see launch_gather)
    if (vpr <= 1) UGK_GO(1);
    if (vpr <= 4) UGK_GO(4);
    if (vpr <= 16) UGK_GO(16);
    UGK_GO(64);
  } else {
    if (vpr <= 1) UGK_GO(1);
    if (vpr <= 16) UGK_GO(16);
    UGK_GO(64);
  }
#undef UGK_GO
}

// Rows per wavefront of a flat copy: the fewest that fill nine tenths of the last round of 4 vectors per lane, or the
// number that fills it best.  Few, because wavefronts that start in order keep the rows being written in one window
// (see gather_grid).  A small launch is a wavefront's own time, not bandwidth: up to 65,536 rows and 8 MiB are spread over
// more wavefronts of half a round, at most 16 rows (100 bytes x 2,048 3.8 -> 3.4 us, 252 bytes x 2,048 3.6 -> 3.4, 600 bytes x
// 2,048 4.8 -> 3.7, x 16,384 7.6 -> 6.6; 4-byte or 8-byte lanes, which the flat copy replaces, 3.3, 3.3, 4.1 and 7.6).
uint32_t flat_tile(size_t row_bytes, size_t n) {
  const size_t chunks = (row_bytes + 15) / 16, round = 4 * kWave;
  if (n <= 65536 && n * row_bytes <= (size_t)8 << 20)
    return (uint32_t)std::min<size_t>(std::max<size_t>(round / 2 / chunks, 1), 16);
  uint32_t best = 1;
  double best_fill = 0;
  for (uint32_t t = 1; t <= (uint32_t)kWave && t * chunks <= 4 * round; ++t) {
    const double fill = (double)(t * chunks) / (double)((t * chunks + round - 1) / round * round);
    if (fill > best_fill) best = t, best_fill = fill;
    if (fill >= 0.9) break;
  }
  return best;
}

// Which dense gathers deal the output out instead of the rows.  Measured, us per launch, rows out of HBM:
//   rows of whole vectors, against gather_kernel's 2^k lanes per row, which idle unless the row is 2^k vectors; by
//   wavefronts of that kernel (four rows of up to 64 vectors each, eight of up to 32), lanes -> this: 272 bytes 3,855 6.3 ->
//   6.8, 5,782 9.2 -> 8.4, 30,840 32.6 -> 30.4; 400 bytes 3,932 7.6 -> 8.1, 5,243 10.5 -> 9.6, 20,971 30.4 -> 28.9; 528 bytes
//   3,972 6.0 -> 6.6, 5,958 8.8 -> 8.0, 31,775 30.1 -> 28.2; 912 bytes 3,449 7.3 -> 7.9, 4,599 9.7 -> 9.3, 18,396 28.3 ->
//   27.0.  Up to four wavefronts per SIMD the lanes are the faster ones, beyond that this.  Rows of more than 64 vectors,
//   by bytes of output, 1 / 8 / 12 / 64 MiB: 1200 bytes 3.9 / 6.4 / 8.1 / 30.0 -> 3.7 / 6.4 / 7.8 / 26.8; 1616 bytes 3.9 / 6.0 /
//   7.7 / 27.2 -> 3.7 / 6.4 / 7.8 / 26.4; 2064 bytes 4.3 / 6.5 / 8.3 / 29.1 -> 3.7 / 6.4 / 7.7 / 26.2; 9008 bytes 8.3 / 10.4 /
//   11.2 / 26.9 -> 3.7 / 6.2 / 7.7 / 25.7.  Rows of 160 bytes and rows of 2^k vectors are level or slower at any size
//   other rows, against gather_flat_kernel: 404 bytes: 65,536 keys 13.4 -> 14.4, 262,144 keys 42.5 -> 44.6; 804 bytes: 21.9
//     -> 22.3, 71.6 -> 74.3; 1204 bytes: 32.3 -> 30.5, 137.6 -> 124.4; 2404 bytes: 55.1 -> 52.3; 3000 bytes: 66.1 -> 62.6
//     (the vectors that two rows share cost two loads and a store per row, which short rows have too many of)
// Over the host link a row is better asked for by one instruction: 24 MiB of 272 bytes with 32 / 128 workgroups 654 / 654 ->
// 675 / 697, 800 bytes 508 / 508 -> 524 / 519, 1600 bytes 475 / 476 -> 491 / 479, 2404 bytes (flat) 493 / 482 -> 503 / 481.  A
// launch whose grid the caller caps is one of those.
bool stream_pays(uintptr_t align, const void *out, size_t row_bytes, size_t n, unsigned max_blocks) {
  if (max_blocks) return false;
  if (align % 16 != 0) return align % 4 == 0 && (uintptr_t)out % 16 == 0 && row_bytes >= 1024;
  if (row_bytes < kStreamMinBytes || (row_bytes & (row_bytes - 1)) == 0) return false;
  if (row_bytes > 1024) return row_bytes >= 2048 || n * row_bytes >= (size_t)10 << 20;
  const size_t rows_per_wave = row_bytes > 512 ? 4 : 8;
  return n / rows_per_wave > (size_t)cu_count() * 16;
}

template <typename Idx>
int launch_flat(Idx ix, const void *src, uint64_t src_rows, void *out, uint64_t out_rows, size_t row_bytes,
                const uint32_t *counts, uint32_t group, size_t n, unsigned max_blocks, uint32_t *status,
                uint32_t *host_mirror, DoneRequest &request, hipStream_t stream) {
  const FlatRow f = flat_row(row_bytes, flat_tile(row_bytes, n));
  const size_t per_block = (size_t)f.tile * kWavesPerBlock;
  const unsigned grid = request.grid(gather_grid((n + per_block - 1) / per_block, max_blocks));
  const bool far = over_link(counts, group, max_blocks);
#define UGK_GO(STORE, LOADS, KEEP, DONE)                                                                               \
  hipLaunchKernelGGL((gather_flat_kernel<STORE, LOADS, Idx>), dim3(grid), dim3(kBlock), 0, stream, ix,                 \
                     (const char *)src, src_rows, (char *)out, out_rows, f, counts, group, KEEP, n, status, host_mirror, \
                     Ending<STORE>(DONE))
  if constexpr (Idx::kDense) {
    const DoneWords done = request.take(grid, Telling::kSooner);
    if (done.tag) {
      if (keep_waves_for(n, row_bytes, kThrough, far)) UGK_GO(kThrough, kKept, kWavesPerBlock, done);
      else UGK_GO(kThrough, kPast, 0, done);
      UGK_HIP(hipGetLastError());
      return 0;
    }
    UGK_REQUIRE(!request.counted(), "gather: a launch that leaves no words cannot take its count from the device");
  }
  UGK_GO(kOrdinary, kByWave, keep_waves_for(n, row_bytes, kOrdinary, far), DoneWords{});
#undef UGK_GO
  UGK_HIP(hipGetLastError());
  return 0;
}

template <typename Idx>
int launch_stream(Idx ix, const void *src, uint64_t src_rows, void *out, size_t row_bytes, size_t n,
                  unsigned max_blocks, uint32_t *status, uint32_t *host_mirror, DoneRequest &request, hipStream_t stream) {
  const StreamRow f = stream_row(row_bytes, n);
  const uint64_t per_block = (uint64_t)kStreamPart * kWavesPerBlock;
  const unsigned grid = request.grid(gather_grid((f.total + per_block - 1) / per_block, max_blocks));
  const bool nt = !request.counted() && nt_store_for(n * row_bytes);
  const DoneWords done = nt ? DoneWords{} : request.take(grid, Telling::kSooner);
  UGK_REQUIRE(!request.counted(), "gather: a launch that leaves no words cannot take its count from the device");
  const uint8_t keep_waves = keep_waves_for(n, row_bytes, done.tag ? kThrough : nt ? kStreaming : kOrdinary,
                                            over_link(nullptr, 0, max_blocks));
#define UGK_GO2(STORE, LOADS, SHARE)                                                                                  \
  hipLaunchKernelGGL((gather_stream_kernel<STORE, LOADS, SHARE, Idx>), dim3(grid), dim3(kBlock), 0, stream, ix,      \
                     (const char *)src, src_rows, (char *)out, f, status, host_mirror, Ending<STORE>(done), keep_waves)
#define UGK_GO(STORE, LOADS)                  \
  do {                                        \
    if (share) UGK_GO2(STORE, LOADS, true);   \
    else UGK_GO2(STORE, LOADS, false);        \
  } while (0)
  const bool share = row_bytes % 16 != 0;
  if (done.tag && keep_waves) UGK_GO(kThrough, kKept);
  else if (done.tag) UGK_GO(kThrough, kPast);
  else if (nt) UGK_GO(kStreaming, kByWave);
  else UGK_GO(kOrdinary, kByWave);
#undef UGK_GO2
#undef UGK_GO
  UGK_HIP(hipGetLastError());
  return 0;
}

template <typename Idx>
int launch_gather(Idx ix, const void *src, uint64_t src_rows, void *out, uint64_t out_rows, size_t row_bytes,
                  const uint32_t *counts, uint32_t group, size_t n, unsigned max_blocks, uint32_t *status,
                  uint32_t *host_mirror, void *stream) {
  DoneRequest request;  // (of which only gathers whose row i is output row i make use)
  if (n == 0) return 0;
  UGK_REQUIRE(src && out, "gather: null source or output");
  UGK_REQUIRE(status, "gather: null status word");
  UGK_REQUIRE(row_bytes > 0 && row_bytes <= (1u << 30), "gather: row_bytes %zu out of range", row_bytes);
  UGK_REQUIRE(n <= 0xffffffffull, "gather: batch of %zu rows exceeds 2^32", n);
  UGK_REQUIRE(Idx::kDense || !request.counted(), "gather: only ugk_gather_direct_* takes its count from the device");
  const uintptr_t align = (uintptr_t)src | (uintptr_t)out | (uintptr_t)row_bytes;
  hipStream_t st = as_stream(stream);
#define UGK_VEC(V)                                                                                                  \
  return launch_vec<V, Idx>(ix, src, src_rows, out, out_rows, row_bytes, counts, group, n, max_blocks, status,      \
                            host_mirror, request, st)
  if constexpr (Idx::kDense) {
    if (stream_pays(align, out, row_bytes, n, max_blocks))
      return launch_stream<Idx>(ix, src, src_rows, out, row_bytes, n, max_blocks, status, host_mirror, request,
                                st);
  }
  if (align % 16 == 0) UGK_VEC(u32x4);
  // short rows in small launches: 16 lanes of 4 bytes have less to do before their first load than the flat copy (36 bytes x
  // 2,048 3.2 / 3.8 us, x 65,536 5.0 / 5.3, x 262,144 14.6 / 10.6; 52 bytes x 8,192 3.3 / 4.0, x 65,536 5.4 / 6.1)
  if (align % 4 == 0 && row_bytes <= 64 && n <= 65536) UGK_VEC(uint32_t);
  // the host group of a batch, with no cap on the grid: so many requests at once the link answers better where each is one
  // instruction of 4-byte lanes (16 MiB of 100 / 148 / 200 / 252 / 300 bytes 753 / 587 / 497 / 455 / 459 us, flat 815 / 661 /
  // 571 / 519 / 485; 404 bytes 436 and 433); behind a cap the flat copy is the faster one (32 workgroups, 200 bytes 663 and
  // 522 us)
  if (align % 4 == 0 && counts && group == UGK_LOC_HOST && max_blocks == 0 && row_bytes <= 320) UGK_VEC(uint32_t);
  if (flat_row_ok(align, row_bytes))
    return launch_flat<Idx>(ix, src, src_rows, out, out_rows, row_bytes, counts, group, n, max_blocks, status,
                            host_mirror, request, st);
  // rows of 8 bytes: one lane of 8 bytes each in large launches, where four of 4 bytes, two of them idle, are too many (us:
  // 2 M rows 49.4 / 51.6, 262,144 rows 8.5 / 8.6, 8,192 rows 4.0 / 3.2)
  if (row_bytes == 8 && align % 8 == 0 && n > 262144) UGK_VEC(unsigned long long);
  if (align % 4 == 0) UGK_VEC(uint32_t);
  if (align % 2 == 0) UGK_VEC(uint16_t);
  UGK_VEC(uint8_t);
#undef UGK_VEC
}

}  // namespace

namespace {
thread_local int g_output_hint = 0;
}
bool nt_store_for(size_t out_bytes) {
  static int forced = [] {
    const char *e = getenv("UGK_GATHER_NT_STORE");
    return e ? atoi(e) : -1;
  }();
  if (forced >= 0) return forced != 0;
  if (g_output_hint == UGK_OUTPUT_STREAMS) return true;
  if (g_output_hint == UGK_OUTPUT_STAYS) return false;
  return out_bytes > kMemorySideCacheBytes;
}
// an empty launch: what it costs is the load of this file's code object onto the device (see ugk_preload_kernels)
namespace {
__global__ void preload_gather_kernel() {}
}  // namespace
void preload_gather(hipStream_t stream) { hipLaunchKernelGGL(preload_gather_kernel, dim3(1), dim3(1), 0, stream); }
}  // namespace ugk

using namespace ugk;

extern "C" {

int ugk_set_output_hint(int hint) {
  UGK_REQUIRE(hint == UGK_OUTPUT_AUTO || hint == UGK_OUTPUT_STREAMS || hint == UGK_OUTPUT_STAYS,
              "ugk_set_output_hint: unknown hint %d", hint);
  g_output_hint = hint;
  return 0;
}

int ugk_gather_direct_u32(const void *src_dev, uint64_t src_rows, const uint32_t *keys_dev, size_t n, void *out_dev,
                          size_t row_bytes, unsigned max_blocks, uint32_t *status_dev, uint32_t *host_mirror,
                          void *stream) {
  UGK_REQUIRE(n == 0 || keys_dev, "ugk_gather_direct_u32: null keys");
  return launch_gather(DirectU32{keys_dev}, src_dev, src_rows, out_dev, kNoLimit, row_bytes, nullptr, 0, n,
                       max_blocks, status_dev, host_mirror, stream);
}

int ugk_gather_direct_i64(const void *src_dev, uint64_t src_rows, const int64_t *keys_dev, size_t n, void *out_dev,
                          size_t row_bytes, unsigned max_blocks, uint32_t *status_dev, uint32_t *host_mirror,
                          void *stream) {
  UGK_REQUIRE(n == 0 || keys_dev, "ugk_gather_direct_i64: null keys");
  return launch_gather(DirectI64{keys_dev}, src_dev, src_rows, out_dev, kNoLimit, row_bytes, nullptr, 0, n,
                       max_blocks, status_dev, host_mirror, stream);
}

int ugk_gather_scatter_u32(const void *src_dev, uint64_t src_rows, const uint32_t *keys_dev,
                           const uint32_t *dst_off_dev, size_t n, void *out_dev, uint64_t out_rows, size_t row_bytes,
                           unsigned max_blocks, uint32_t *status_dev, uint32_t *host_mirror, void *stream) {
  UGK_REQUIRE(n == 0 || (keys_dev && dst_off_dev), "ugk_gather_scatter_u32: null keys or destinations");
  return launch_gather(ScatterU32{keys_dev, dst_off_dev}, src_dev, src_rows, out_dev, out_rows, row_bytes, nullptr, 0,
                       n, max_blocks, status_dev, host_mirror, stream);
}

int ugk_gather_scatter_i64(const void *src_dev, uint64_t src_rows, const int64_t *keys_dev,
                           const uint32_t *dst_off_dev, size_t n, void *out_dev, uint64_t out_rows, size_t row_bytes,
                           unsigned max_blocks, uint32_t *status_dev, uint32_t *host_mirror, void *stream) {
  UGK_REQUIRE(n == 0 || (keys_dev && dst_off_dev), "ugk_gather_scatter_i64: null keys or destinations");
  return launch_gather(ScatterI64{keys_dev, dst_off_dev}, src_dev, src_rows, out_dev, out_rows, row_bytes, nullptr, 0,
                       n, max_blocks, status_dev, host_mirror, stream);
}

int ugk_gather_scatter_staged_u32(const void *host_dev, uint64_t host_rows, const uint32_t *rows_dev,
                                  const uint32_t *dst_off_dev, size_t n, void *out_dev, uint64_t out_rows,
                                  size_t row_bytes, ugk_stage_t stage, unsigned max_blocks, uint32_t *status_dev,
                                  uint32_t *staged_dev, uint32_t *rest_rows_dev, uint32_t *rest_dst_dev,
                                  uint32_t *rest_count_dev, uint32_t *done_count_dev, void *stream) {
  DoneRequest request;
  if (n == 0) return 0;
  UGK_REQUIRE(rest_count_dev == nullptr || (rest_rows_dev && rest_dst_dev),
              "ugk_gather_scatter_staged_u32: a rest count without the two rest lists");
  UGK_REQUIRE(done_count_dev == nullptr || rest_count_dev, "ugk_gather_scatter_staged_u32: a done count without rest lists");
  UGK_REQUIRE(n <= 0xffffffffull, "ugk_gather_scatter_staged_u32: %zu rows do not fit 32-bit list positions", n);
  UGK_REQUIRE(host_dev && rows_dev && dst_off_dev && out_dev && status_dev, "ugk_gather_scatter_staged_u32: null pointer");
  UGK_REQUIRE(stage.rows_dev && stage.owner_dev && ((stage.mask + 1) & stage.mask) == 0,
              "ugk_gather_scatter_staged_u32: the stage needs buffers and a power of two of entries");
  const uintptr_t align = (uintptr_t)host_dev | (uintptr_t)out_dev | (uintptr_t)stage.rows_dev | (uintptr_t)row_bytes;
  UGK_REQUIRE(row_bytes > 0 && align % 16 == 0,
              "ugk_gather_scatter_staged_u32: rows and buffers must be multiples of 16 bytes (row_bytes=%zu)", row_bytes);
  UGK_REQUIRE(host_rows <= 0x100000000ull, "ugk_gather_scatter_staged_u32: host rows must fit 32 bits");
  const uint32_t vpr = (uint32_t)(row_bytes / 16);
  uint32_t lpr = 1;
  while (lpr < vpr && lpr < 64) lpr <<= 1;
  const size_t per_iter = (size_t)(kBlock / lpr) * kStagedUnroll;
  const unsigned grid = clamp_grid((n + per_iter - 1) / per_iter, max_blocks);
  hipLaunchKernelGGL(gather_staged_kernel, dim3(grid), dim3(kBlock), 0, as_stream(stream),
                     reinterpret_cast<const u32x4 *>(host_dev), host_rows, rows_dev, dst_off_dev, n,
                     reinterpret_cast<u32x4 *>(out_dev), out_rows, vpr, lpr, stage, status_dev, staged_dev,
                     rest_rows_dev, rest_dst_dev, rest_count_dev, done_count_dev);
  UGK_HIP(hipGetLastError());
  return 0;
}

int ugk_gather_group(const void *src_dev, uint64_t src_rows, const ugk_idx_t *idx_dev, const uint32_t *counts_dev,
                     uint32_t group, size_t n, void *out_dev, uint64_t out_rows, size_t row_bytes,
                     unsigned max_blocks, uint32_t *status_dev, uint32_t *host_mirror, void *stream) {
  UGK_REQUIRE(n == 0 || (idx_dev && counts_dev), "ugk_gather_group: null index list or counts");
  UGK_REQUIRE(group == UGK_LOC_LOCAL || group == UGK_LOC_HOST, "ugk_gather_group: group %u is not local/host", group);
  return launch_gather(IdxList{idx_dev}, src_dev, src_rows, out_dev, out_rows, row_bytes, counts_dev, group, n, max_blocks,
                       status_dev, host_mirror, stream);
}

int ugk_replicate_rows(void *out_dev, size_t row_bytes, const uint32_t *inverse_dev, const uint32_t *rep_dev, size_t n,
                       void *stream) {
  if (n == 0) return 0;
  UGK_REQUIRE(out_dev && inverse_dev && rep_dev, "ugk_replicate_rows: null pointer");
  UGK_REQUIRE(row_bytes > 0, "ugk_replicate_rows: empty rows");
  hipStream_t st = as_stream(stream);
  if (((uintptr_t)out_dev | row_bytes) % 16 == 0) {
    const uint32_t vpr = (uint32_t)(row_bytes / 16);
    if (vpr <= 8) {
      const unsigned grid = clamp_grid((n + kBlock / 8 - 1) / (kBlock / 8), 0);
      hipLaunchKernelGGL((replicate_kernel<u32x4, 8>), dim3(grid), dim3(kBlock), 0, st, (u32x4 *)out_dev, vpr,
                         inverse_dev, rep_dev, n);
    } else {
      const unsigned grid = clamp_grid((n + kBlock / 32 - 1) / (kBlock / 32), 0);
      hipLaunchKernelGGL((replicate_kernel<u32x4, 32>), dim3(grid), dim3(kBlock), 0, st, (u32x4 *)out_dev, vpr,
                         inverse_dev, rep_dev, n);
    }
  } else {
    const unsigned grid = clamp_grid((n + kBlock / 32 - 1) / (kBlock / 32), 0);
    hipLaunchKernelGGL((replicate_kernel<uint8_t, 32>), dim3(grid), dim3(kBlock), 0, st, (uint8_t *)out_dev,
                       (uint32_t)row_bytes, inverse_dev, rep_dev, n);
  }
  UGK_HIP(hipGetLastError());
  return 0;
}

int ugk_gather_idx(const void *src_dev, uint64_t src_rows, const ugk_idx_t *idx_dev, size_t count, void *out_dev,
                   size_t row_bytes, unsigned max_blocks, uint32_t *status_dev, void *stream) {
  UGK_REQUIRE(count == 0 || idx_dev, "ugk_gather_idx: null index list");
  return launch_gather(IdxList{idx_dev}, src_dev, src_rows, out_dev, kNoLimit, row_bytes, nullptr, 0, count,
                       max_blocks, status_dev, nullptr, stream);
}

}  // extern "C"
