// Internal helpers shared by the gfx950 translation units behind include/ugache_hip.h.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstdint>
#include <cstdio>

#include "ugache_hip.h"

int ugk_set_error(const char *fmt, ...) __attribute__((format(printf, 1, 2)));

#define UGK_HIP(expr)                                                                                        \
  do {                                                                                                       \
    hipError_t ugk_e_ = (expr);                                                                              \
    if (ugk_e_ != hipSuccess)                                                                                \
      return ugk_set_error("%s failed: %s (%s:%d)", #expr, hipGetErrorString(ugk_e_), __FILE__, __LINE__);   \
  } while (0)

#define UGK_REQUIRE(cond, ...)                        \
  do {                                                \
    if (!(cond)) return ugk_set_error(__VA_ARGS__);   \
  } while (0)

namespace ugk {

constexpr int kBlock = 256;  // 4 wavefronts of 64 lanes
constexpr int kWave = 64;

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// Number of compute units of the current device (cached per device).
int cu_count();

// Upper bound, in workgroups per CU, of grid-stride launches that should fill the chip (default 64: many short
// workgroups balance better than few long ones on this part); UGK_BLOCKS_PER_CU overrides.
int blocks_per_cu();

static inline hipStream_t as_stream(void *s) { return reinterpret_cast<hipStream_t>(s); }

static inline unsigned clamp_grid(size_t want, unsigned max_blocks) {
  if (want == 0) want = 1;
  size_t cap = max_blocks ? (size_t)max_blocks : (size_t)cu_count() * (size_t)blocks_per_cu();
  if (want > cap) want = cap;
  return (unsigned)want;
}

// Non-temporal stores for an extraction whose output of `out_bytes` will not stay in the 256 MiB memory-side cache
// anyway; ordinary write-back stores otherwise, so that the consumer finds the rows there.  The caller's hint
// (ugk_set_output_hint) and UGK_GATHER_NT_STORE=0/1 override the size rule.  The line is the cache's size to the megabyte;
// gathers into one buffer, ordinary / non-temporal stores, us: 512-byte rows, output of 192 MiB 63.9 / 70.2, 224 MiB 72.8 /
// 81.2, 256 MiB 83.7 / 92.0, 288 MiB 112.5 / 103.4; 128-byte rows 256 MiB 89.3 / 94.0, 288 MiB 114.1 / 105.1; 1204-byte
// rows 256 MiB 89.5 / 105.5, 288 MiB 120.9 / 118.0.
constexpr size_t kMemorySideCacheBytes = (size_t)256 << 20;
bool nt_store_for(size_t out_bytes);

// What a launch leaves for a host that polls for its end (ugk_leave_done_words; leave_done in ugk_mix.cuh); tag 0: nobody
// polls, and words, if there are any, are the per-workgroup counts of ugk_extract_mix_*.
struct DoneWords {
  unsigned long long *words, *counters;
  void *keys;         // the launch leaves its first num_keys keys here (pinned host memory); where num_keys is 0 and this is
  uint64_t num_keys;  // not, it is a device word: how many of the launch's keys there are (launch_count)
  uint32_t tag;
  uint32_t set;       // which of the two sets of counters
};
// Up to kDoneDirect workgroups leave a word each.  More of them meet in kDoneFan counters, workgroup b in counter b %
// kDoneFan, and the last one of a counter leaves its word: writes into host memory cost 2 us per thousand, and a host that
// polls thousands of words falls behind.  262,144 rows of 512 bytes gathered, launch to end of poll, with 32 / 64 / 128 /
// 256 / 512 / 1024 counters 48.6 / 48.7 / 49.0 / 49.3 / 49.7 / 50.8 us, a word per workgroup (16,384) 53.0, one-lane ticket
// kernel behind the gather 52.0; 8,192 rows (512 workgroups) 8.9 / 8.8 / 9.0 / 9.3 / 9.2 / 9.2, 9.1 and 9.8; 1,664 rows 8.4 /
// 8.6 / 8.2 / 8.2 / 8.1 / 8.1, 8.0 and 9.4; 8 rows 6.3 against 8.5.
constexpr uint32_t kDoneDirect = UGK_DONE_WORDS, kDoneFan = UGK_DONE_COUNTERS / 2;

// When words are there, against a ticket kernel behind the launch (ugk_done_t::where_faster): sooner or at the same time, or later by
// more than a kernel that copies keys takes.
enum class Telling { kSooner, kTooLate };

// The request of ugk_leave_done_words, if this thread has made one: the entry points that can fulfil it take it as they
// begin, so that it never meets a later launch.
class DoneRequest {
 public:
  DoneRequest();
  // grid: workgroups of the launch; count_limit: no counter of it reaches this, 0 where none are kept
  DoneWords take(unsigned grid, Telling words, uint64_t count_limit = 0);
  // whether the number of keys is in a device word; a launch that has not taken the request then must not go ahead
  bool counted() const;
  // ... and one that has leaves workgroups without keys: not more of them than keep the chip busy
  unsigned grid(unsigned wanted) const;

 private:
  ugk_done_t *_done;
};

__device__ __forceinline__ unsigned lane_id() { return __lane_id(); }
// number of the wavefront in its workgroup, in a scalar register: what is computed from it stays scalar
__device__ __forceinline__ unsigned wave_in_block() { return __builtin_amdgcn_readfirstlane(threadIdx.x / kWave); }

// one per source file with kernels: launches an empty kernel of that file on `stream`
void preload_gather(hipStream_t stream);
void preload_hotness(hipStream_t stream);
void preload_partition(hipStream_t stream);
void preload_pool(hipStream_t stream);
void preload_pool_i64(hipStream_t stream);
void preload_refresh(hipStream_t stream);
void preload_table(hipStream_t stream);

}  // namespace ugk
