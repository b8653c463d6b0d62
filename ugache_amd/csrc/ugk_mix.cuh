// What the kernels that look a key up and read its row in one go have in common (the fused extraction and the pooled
// one): where a key's row lives, and how a launch hands its per-source row counts to the host.  And the copy of rows
// that are no power of two of 16-byte vectors, or start at 4-byte boundaries only, which the gathers share with the
// fused extraction.
#pragma once

#include "ugk_internal.h"
#include "ugk_table.cuh"

namespace ugk {
namespace {

constexpr int kWavesPerBlock = kBlock / kWave;

typedef const __attribute__((address_space(1))) u32x4 *grow_t;  // a row in global memory (HBM, or mapped host memory)
typedef __attribute__((address_space(1))) u32x4 *gout_t;

// ---- the end of a launch a host polls for --------------------------------------------------------------------------
// Stores that are written through the caches (system scope): once such a store has been acknowledged its bytes are in
// memory, and not in the L2 of an XCD that is written back when the kernel has ended.  In assembler, for the language has
// no such stores of 16 bytes.  The s_nop: gfx940 and later want two wait states between a store of more than 8 bytes and a
// vector instruction that overwrites its data, and the compiler, which sees to that elsewhere, does not look into assembler.
template <typename V>
__device__ __forceinline__ void store_through(uint64_t to, V v) {
  typedef __attribute__((address_space(1))) char *gbyte_t;
  const gbyte_t p = reinterpret_cast<gbyte_t>(to);
  if constexpr (sizeof(V) == 16) asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1\n\ts_nop 1" ::"v"(p), "v"(v) : "memory");
  else if constexpr (sizeof(V) == 8) asm volatile("global_store_dwordx2 %0, %1, off sc0 sc1" ::"v"(p), "v"(v) : "memory");
  else if constexpr (sizeof(V) == 4) asm volatile("global_store_dword %0, %1, off sc0 sc1" ::"v"(p), "v"(v) : "memory");
  else if constexpr (sizeof(V) == 2) asm volatile("global_store_short %0, %1, off sc0 sc1" ::"v"(p), "v"((uint32_t)v) : "memory");
  else asm volatile("global_store_byte %0, %1, off sc0 sc1" ::"v"(p), "v"((uint32_t)v) : "memory");
}

// Everything in v has arrived, before the first of it is stored.  One counter counts a wavefront's loads and stores, in the
// order they were issued, and a wait names how many may still be on their way.  Stores that are written through are not in
// the compiler's count (they are assembly), stores behind a condition may or may not have been issued: so the wait for the
// second of four loads would be one for the first store as well, until that is in memory, and a lane's stores leave one by
// one.  us, launch to end of poll, before / with this: gather 512 bytes x 1,024 10.8 / 10.2, 4 KB x 128 13.5 / 11.7, 8 KB x
// 1,024 19.3 / 15.6; lookup and gather in one kernel, 512 bytes x 4,096 13.9 / 13.3, 1 KB x 4,096 15.9 / 14.7, 2 KB x 512 17.1 /
// 14.3, 4 KB x 2,048 25.5 / 18.7; that kernel with ordinary stores and a ticket behind it 15.3 / 15.1, 16.1 / 15.6, 16.3 / 14.9,
// 22.8 / 19.8.  (Ordinary stores of the flat and the stream copy of a plain gather: 1 to 5 % either way, left as they were.)
template <typename V>
__device__ __forceinline__ void arrived(V &v) {
  if constexpr (sizeof(V) >= 4) asm volatile("" : "+v"(v));
}
template <typename V, int N>
__device__ __forceinline__ void arrived(V (&v)[N]) {
#pragma unroll
  for (int u = 0; u < N; ++u) arrived(v[u]);
}

// how a kernel stores its rows: a template parameter, not a launch argument, for with a run-time choice the optimiser merges
// an ordinary and a non-temporal store into one and the hint is lost, and the code of all of them costs a small launch
// 0.2 to 0.4 us (26,624 rows of 64 bytes 3.6 -> 4.0)
enum Store { kOrdinary, kStreaming, kThrough };

// What a kernel is told about its end: one that is polled for everything, any other where the counts of its workgroups go, if
// anywhere.  Not more than that: the arguments are in host memory, and the line of 64 bytes that the whole of DoneWords pushed
// the launch's own numbers into cost every launch of a plain gather (us, stream-ordered: 262,144 rows of 200 bytes 24.9 ->
// 25.9, of 12 bytes 7.9 -> 8.2, 16,384 rows of 512 bytes 4.3 -> 5.1).
template <Store STORE>
struct Ending {
  unsigned long long *words;
  explicit Ending(const DoneWords &done) : words(done.words) {}
  __device__ explicit Ending(unsigned long long *counts) : words(counts) {}
};
template <>
struct Ending<kThrough> : DoneWords {
  explicit Ending(const DoneWords &done) : DoneWords(done) {}
};

// how many of its n keys the launch looks up (ugk_done_t::count_dev)
template <Store STORE>
__device__ __forceinline__ size_t launch_count(const Ending<STORE> &done, size_t n) {
  if constexpr (STORE == kThrough) {
    if (done.num_keys == 0 && done.keys) return min(n, (size_t)*static_cast<const uint32_t *>(done.keys));
  }
  return n;
}

// A word for the host beside the rows (an error flag, a key).  The same kind of store: an ordinary one into host memory is
// acknowledged before it is there, and the words of leave_done, which say that all of this is complete, may overtake it
// (a lookup of four keys, one of them out of range, returned without its error that way).
template <typename T>
__device__ __forceinline__ void tell_host(T *word, T v) {
  __hip_atomic_store(word, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// key i of the launch, where the host wants a copy (a lane per key: neighbouring lanes' keys leave as one write)
template <typename K>
__device__ __forceinline__ void copy_key_along(const DoneWords &done, uint64_t i, K key) {
  if (i < done.num_keys) tell_host(static_cast<K *>(done.keys) + i, key);
}

// The last thing a workgroup does: its counts, and where a host polls the news that it has ended.  All threads call it; tot (in LDS,
// may be NULL) holds the rows taken from the cache and all others.
template <Store STORE>
__device__ __forceinline__ void leave_done(const Ending<STORE> &done, const uint32_t *tot) {
  if constexpr (STORE == kThrough) {
    // The set of counters this launch does not use is made zero for the next one, in front of the wait: once all words are
    // there that is complete, also for a launch on another stream, which does not wait for this one to end.  (A counter
    // cleared by the workgroup that finds it complete would need a wait between that and its word.)
    if (gridDim.x > kDoneDirect && blockIdx.x < kDoneFan && threadIdx.x == 0)
      __hip_atomic_store(done.counters + ((done.set ^ 1u) * kDoneFan + blockIdx.x) * 16, 0ull, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wavefront's stores have been acknowledged
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  const uint32_t local = tot ? tot[0] : 0u, others = tot ? tot[1] : 0u;
  if constexpr (STORE != kThrough) {
    done.words[blockIdx.x] = ((unsigned long long)others << 32) | local;
  } else {
    const unsigned long long tag = (unsigned long long)done.tag << 48, mine = ((unsigned long long)others << 24) | local;
    if (gridDim.x <= kDoneDirect) {
      done.words[blockIdx.x] = tag | mine;
      return;
    }
    const uint32_t g = blockIdx.x % kDoneFan, members = gridDim.x / kDoneFan + (g < gridDim.x % kDoneFan ? 1u : 0u);
    const unsigned long long add = (1ull << 48) | mine;
    unsigned long long *counter = done.counters + (done.set * kDoneFan + g) * 16;  // a line each
    const unsigned long long sum =
        __hip_atomic_fetch_add(counter, add, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + add;
    if ((uint32_t)(sum >> 48) == members) done.words[g] = tag | (sum & 0xffffffffffffull);
  }
}

// ---- flat row copy -------------------------------------------------------------------------------------------------
// Rows of any multiple of 4 bytes above 16, as 16-byte vectors all the same: a vector load or store of global memory
// needs 4-byte alignment only, and the last vector of a row is moved back so that it ends with the row (it overlaps
// the one before it; both write the same bytes).  The vectors of a wavefront's rows are numbered through and dealt
// to the 64 lanes in order, so that no lane is idle whatever the row's length.  Bound by HBM, whose unit is a line of 128
// bytes: a row of R bytes at a random multiple of 4 touches (R + 124) / 128 of them.  What it replaced were lanes of 4 or
// 8 bytes, 16 or 64 to a row; gathers of 262,144 rows out of 4 GiB of HBM, before -> after: 36 bytes 14.6 -> 10.6 us,
// 100 bytes 38.0 -> 17.0 us (5.0 TB/s of lines read and rows written), 200 bytes 44.3 -> 25.7, 404 bytes 64.3 -> 42.7,
// 804 bytes 137.8 -> 71.6.  The stores are ordinary ones whatever the size of the output and whatever ugk_set_output_hint says:
// rows that end inside a line leave it in two pieces, which non-temporal stores write out apart.  us per launch, ordinary /
// non-temporal: 804 bytes, one buffer of 224 / 288 / 600 MiB 80 / 100, 123 / 130, 266 / 270, four of 224 MiB in turn 99.5 /
// 100; 200 bytes 99 / 119, 151 / 155, 319 / 323 and 116 / 119; 1020 bytes 78 / 100, 121 / 132, 265 / 278 and 96 / 101; only
// rows of 36 bytes are 2 % the other way beyond the memory-side cache, 317 / 312 for 288 MiB.
typedef u32x4 u32x4_by4 __attribute__((aligned(4)));
typedef const __attribute__((address_space(1))) u32x4_by4 *grow_by4_t;
typedef __attribute__((address_space(1))) u32x4_by4 *gout_by4_t;

struct FlatRow {
  uint32_t row_bytes;
  uint32_t chunks;  // 16-byte vectors of a row, the last one overlapping
  uint32_t magic;   // floor(2^32 / chunks) + 1: idx / chunks = mulhi(idx, magic) for every idx < 64 * chunks
  uint32_t tile;    // rows numbered through together, at most 64
};
constexpr uint32_t kFlatMinBytes = 20;        // shorter rows are one vector or none
constexpr uint32_t kFlatMaxBytes = 1u << 30;  // lengths and offsets in a row are counted in 32 bits
constexpr uint32_t kFlatMaxTiled = 8192;      // chunks up to which mulhi divides exactly (idx * chunks < 2^32)
constexpr uint32_t kNoRowBit = 1;             // in a row's address: nothing is copied for it

static inline bool flat_row_ok(uintptr_t align, size_t row_bytes) { return align % 4 == 0 && row_bytes >= kFlatMinBytes; }

// tile: how many rows a wavefront numbers through (a row too long to divide by is a tile of its own)
static inline FlatRow flat_row(size_t row_bytes, uint32_t tile) {
  FlatRow f;
  f.row_bytes = (uint32_t)row_bytes;
  f.chunks = (uint32_t)((row_bytes + 15) / 16);
  const bool tiled = f.chunks < kFlatMaxTiled;
  f.magic = tiled ? (uint32_t)(0x100000000ull / f.chunks) + 1u : 0u;
  f.tile = tiled ? tile : 1u;
  return f;
}

// Copies the rows r0 .. r0 + count - 1 of the wavefront, count <= f.tile: lane r holds where row r is read (kNoRowBit:
// not at all) and, with DENSE false, which output row it becomes; with DENSE row r becomes output row d0 + r.  All
// lanes call it with the same r0 and count.
template <bool DENSE, bool THROUGH, bool KEEP, bool WAIT = THROUGH>
__device__ __forceinline__ void flat_copy(uint64_t src_bits, uint32_t dst_row, char *out, size_t d0, uint32_t r0,
                                          uint32_t count, const FlatRow &f) {
  constexpr int U = 4;  // vectors in flight per lane
  const uint32_t total = count * f.chunks;
  const uint32_t tail = f.row_bytes - 16;
  for (uint32_t i0 = 0; i0 < total; i0 += kWave * U) {
    grow_by4_t p[U];
    gout_by4_t q[U];
    bool ok[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t want = i0 + u * kWave + lane_id();
      // a lane past the end reads the last vector again instead of branching around its load
      const uint32_t idx = want < total ? want : total - 1;
      const uint32_t r = __umulhi(idx, f.magic);
      const uint32_t at = min((idx - r * f.chunks) * 16, tail);
      const uint32_t lo = __shfl((uint32_t)src_bits, (int)(r0 + r)), hi = __shfl((uint32_t)(src_bits >> 32), (int)(r0 + r));
      ok[u] = want < total && (lo & kNoRowBit) == 0;
      p[u] = reinterpret_cast<grow_by4_t>((((uint64_t)hi << 32) | (lo & ~kNoRowBit)) + at);
      const size_t d = DENSE ? d0 + r0 + r : (size_t)__shfl(dst_row, (int)(r0 + r));
      q[u] = reinterpret_cast<gout_by4_t>(reinterpret_cast<uint64_t>(out) + d * f.row_bytes + at);
    }
    u32x4 v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if constexpr (KEEP) v[u] = *p[u];
      else v[u] = __builtin_nontemporal_load(p[u]);
    }
    if constexpr (WAIT) arrived(v);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (ok[u]) {
        if constexpr (THROUGH) store_through(reinterpret_cast<uint64_t>(q[u]), v[u]);
        else *q[u] = v[u];
      }
  }
}

// where a key's row lives, as an integer address (the head of the output for a key without a row, see below)
struct MixRow {
  uint64_t bits;
  uint64_t host_row;  // the row of the host table it is, ~0 for a row of the cache or no row
  bool has_row, from_cache;
};

// row_units: length of a row in units of T (a row of 16-byte vectors may be longer than 32 bits of bytes)
template <typename T>
__device__ __forceinline__ MixRow mix_resolve(const ugk_table_t &t, uint64_t key, bool active, const Found &f,
                                              const T *cache, uint64_t cache_rows, const T *host, uint64_t host_rows,
                                              const void *out, uint32_t row_units, uint32_t *status,
                                              uint32_t *host_mirror) {
  const T *rowp = nullptr;
  uint64_t host_row = ~0ull;
  if (active) {
    if (f.hit && f.loc == UGK_LOC_LOCAL && f.off < cache_rows) rowp = cache + (uint64_t)f.off * row_units;
    else if (f.hit && f.loc == UGK_LOC_HOST && f.off < host_rows) host_row = f.off;
    else if (!f.hit && fallback_row(t, key) < host_rows) host_row = fallback_row(t, key);
    else {
      atomicOr(status, UGK_ST_KEY_OUT_OF_RANGE);
      if (host_mirror) tell_host<uint32_t>(host_mirror, UGK_ST_KEY_OUT_OF_RANGE);
    }
  }
  // A key without a row copies nothing; its lanes read the head of the output instead (mapped whatever the key), so
  // that the loads of the copy carry no branch: behind a branch each of them waits for the one before.
  if (host_row != ~0ull) rowp = host + host_row * row_units;
  MixRow r;
  r.host_row = host_row;
  r.has_row = rowp != nullptr;
  r.bits = r.has_row ? reinterpret_cast<uint64_t>(rowp) : reinterpret_cast<uint64_t>(out);
  r.from_cache = r.has_row && f.hit && f.loc == UGK_LOC_LOCAL;
  return r;
}

// Group sizes for the host: every workgroup leaves its two sums in a word of its own in pinned host memory, a posted
// write nobody waits for; the host adds the words up after it has waited for the stream.  Handing them over through
// device-side atomics cost more than it looks: a 64-bit add and a dependent ticket per workgroup 16 us of a 69 us
// launch at 99 % hits (same-address atomics are performed one after the other at the memory side), one add whose
// result tells the last workgroup still 5 us (every workgroup ends by waiting for the round trip), and a device-scope
// fence per workgroup 13-49 % of a whole step (each writes back and invalidates the L2 of its XCD).
// (A launch that a host polls for waits for its stores anyway, and adds its workgroups up in a few counters: leave_done.)
template <Store STORE>
__device__ __forceinline__ void mix_leave_counts(uint32_t *block_tot, uint32_t wave_local, uint32_t wave_host,
                                                 const Ending<STORE> &done) {
  if (lane_id() == 0) {
    if (wave_local) atomicAdd(&block_tot[0], wave_local);
    if (wave_host) atomicAdd(&block_tot[1], wave_host);
  }
  leave_done(done, block_tot);
}

}  // namespace
}  // namespace ugk
