// Re-placement of the cache on the device, from the hotness counters the lookups keep there: which rows belong to
// the K best-ranked ones, which cached rows fell out, which rows come in, which cache slots are free.  The rank order
// is the one FreqRecorder::Sort + RepSolver::Solve use on the host (freq_recorder.cc:275-281,
// optimal_solver_class.cc:1869-1924): observed rows by (count << 32 | row) descending, never-observed rows behind
// them in ascending row order.
//
// place  : the K best-ranked rows as a bitmap, in two streaming passes over the counters (HBM-bound) and a few
//          launches over bitmaps:
//            1. histogram of min(count, 2047) -> the count T of the K-th best row and how many rows with count T are
//               still needed (counts of 2047 and more are rare: then three more histogram passes over the digits of
//               the count settle T exactly);
//            2. split: bit r of `gt` = count[r] > T, bit r of `eq` = count[r] == T (and the counters are reset if the
//               caller wants the next interval to start from zero);
//          When the caller keeps a bitmap of the observed rows (counter above zero) and fewer rows were observed than
//          are wanted, T is 0 without looking: gt = observed, eq = ~observed, and steps 1 and 2 are bitmap launches.
//            3. the needed rows among `eq` are its topmost set bits (T > 0: larger row first) or its lowest ones
//               (T == 0: never-observed rows in ascending order): the position of the last needed bit is found with the
//               chunk offsets of the ordered compaction below; result = gt | (eq restricted to that side of it).
// bitmap : ordered compaction of the set bits of a, ~a, a & ~b into an ascending index list (count, scan, emit), and
//          setting / clearing listed bits.  Membership of the cache and occupancy of its slots live in such bitmaps,
//          so evict = cached & ~new, insert = new & ~cached, free slots = ~used are all the same three launches.
#include "ugk_internal.h"
#include "ugk_mix.cuh"

namespace ugk {
namespace {

// sums over the wavefront by DPP (adds within rows of 16 lanes, then across them): no trip through LDS, where the six dependent
// permutes of a shuffled scan wait for each other and for those of the CU's other wavefronts
__device__ __forceinline__ uint32_t wave_incl_sum(uint32_t x) {  // of lanes 0 .. mine
  constexpr int kRowShr = 0x110, kRowBcast15 = 0x142, kRowBcast31 = 0x143;
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, kRowShr + 1, 0xf, 0xf, false);
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, kRowShr + 2, 0xf, 0xf, false);
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, kRowShr + 4, 0xf, 0xf, false);
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, kRowShr + 8, 0xf, 0xf, false);
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, kRowBcast15, 0xa, 0xf, false);
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, kRowBcast31, 0xc, 0xf, false);
  return x;
}
__device__ __forceinline__ uint32_t wave_sum(uint32_t x) {  // of all lanes, the same in each
  return (uint32_t)__builtin_amdgcn_readlane((int)wave_incl_sum(x), kWave - 1);
}

constexpr int kHistBins = 2048;        // 11-bit digits at most
constexpr uint32_t kSatCount = kHistBins - 1;
constexpr int kBmChunks = 8192;        // fixed partition of a bitmap, independent of the launch grid
constexpr int kCountPasses = 3;        // digits of a 32-bit count, most significant first
constexpr int kPassShift[kCountPasses] = {21, 10, 0};
constexpr int kPassBits[kCountPasses] = {11, 11, 10};

// A bitmap is cut twice: into kBmChunks chunks of whole 64-word blocks (what the one-workgroup scan works on), and
// into those blocks, each one wavefront load wide.  The emit pass runs one wavefront per block, so set bits that all
// sit in a few chunks (the rows a refresh evicts are often one contiguous run) are still spread over the chip.
constexpr uint64_t kBmMaxBits = 1ull << 32;
constexpr uint32_t kBmMaxBlocks = (uint32_t)(kBmMaxBits / 64 / kWave);  // 2^20
struct BmWs {
  uint32_t total;
  uint32_t scanned;              // base holds the prefix; 0: still the counts (the emit pass adds them up itself)
  uint32_t pad[2];
  uint32_t base[kBmChunks];      // per chunk: first the count, after the scan the exclusive prefix
  uint32_t block[kBmMaxBlocks];  // per 64-word block: its count
};

// The workgroups of a launch that add up two counts: each comes to one of kArriveLines lines, the last of a line to the
// top one (adds on one word are performed one after the other).  A line's first word counts arrivals above the first
// count, the second count is complete before its arrival is seen.
constexpr uint32_t kArriveLines = 32;
struct Arrivals {
  unsigned long long line[kArriveLines + 1][16];
};
// one thread of the workgroup, all of whose stores have been acknowledged; true for the last workgroup of the launch,
// which then has both sums
__device__ __forceinline__ bool arrive(Arrivals *at, uint32_t &a, uint32_t &b) {
  const uint32_t lines = min(gridDim.x, kArriveLines), mine = blockIdx.x % lines;
  uint32_t members = gridDim.x / lines + (mine < gridDim.x % lines ? 1u : 0u);
  for (int level = 0; level < 2; ++level) {
    unsigned long long *w = at->line[level ? kArriveLines : mine];
    __hip_atomic_fetch_add(w + 1, (unsigned long long)b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const unsigned long long add = (1ull << 32) | a;
    const unsigned long long sum = __hip_atomic_fetch_add(w, add, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + add;
    if ((uint32_t)(sum >> 32) != members) return false;
    a = (uint32_t)sum;
    b = (uint32_t)__hip_atomic_load(w + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    members = lines;
  }
  return true;
}

// workspace of a placement
struct RankWs {
  unsigned long long threshold;  // rank of the K-th best row (for reports)
  unsigned long long remaining;  // rows still to be found: first among all rows, in the end among those with count T
  uint32_t count_t;              // T (digits picked so far)
  uint32_t settled;              // the saturating first pass found T
  uint32_t last_row;             // the last needed row among those with count T
  uint32_t from_bitmap;          // fewer rows were observed than are wanted: T = 0, no pass over the counters
  uint32_t keep_mode;            // with a keep bitmap: 1 = the needed rows with count T all come from eq & keep,
                                 // 2 = all of eq & keep is in and the rest comes from eq & ~keep
  uint32_t last_t;               // T of the placement before this one (whatever the memory held, the first time)
  uint32_t guess_t;              // the T the first pass over the counters split by on the way (= last_t)
  uint32_t split_done;           // the guess was T: gt and eq are written, the second pass is not needed
  uint32_t scans_done;           // of bitmap_scan2_kernel behind a placement with a ticket

  uint32_t hist[kHistBins];
  Arrivals arrivals;             // of rank_combine_observed_kernel
  BmWs bm;                       // chunk offsets of `eq`
};

__device__ __forceinline__ unsigned long long rank_of(uint32_t cnt, uint32_t row) {
  return cnt ? ((unsigned long long)cnt << 32) | row : (unsigned long long)(0xffffffffu - row);
}

// mode 0: digit = min(count, 2047) of every row.  mode 1: digit (shift, bits) of the counts that match the digits
// picked so far; skipped when the first pass settled T.
__global__ __launch_bounds__(kBlock) void rank_hist_kernel(const uint32_t *__restrict__ counts, uint64_t n,
                                                           RankWs *ws, int mode, int shift, int bits) {
  if (ws->from_bitmap || (mode == 1 && ws->settled)) return;
  __shared__ uint32_t lh[kHistBins];
  const int tid = threadIdx.x;
  for (int b = tid; b < kHistBins; b += kBlock) lh[b] = 0;
  __syncthreads();
  const uint32_t hi_mask = (mode == 0 || shift + bits >= 32) ? 0u : ~0u << (shift + bits);
  const uint32_t want = ws->count_t & hi_mask;
  const uint32_t digit_mask = (1u << bits) - 1u;
  // consecutive rows mostly share a digit (the cold ones all do): a lane keeps a run and touches the LDS histogram
  // only when the digit changes
  uint32_t last = 0, run = 0;
  auto take = [&](uint32_t c) {
    uint32_t d;
    if (mode == 0) {
      d = c < kSatCount ? c : kSatCount;
    } else {
      if ((c & hi_mask) != want) return;
      d = (c >> shift) & digit_mask;
    }
    if (d == last) {
      ++run;
    } else {
      if (run) atomicAdd(&lh[last], run);
      last = d;
      run = 1;
    }
  };
  const uint64_t n_vec = n / 4;
  const u32x4 *cv = reinterpret_cast<const u32x4 *>(counts);
  for (uint64_t v = (uint64_t)blockIdx.x * kBlock + tid; v < n_vec; v += (uint64_t)gridDim.x * kBlock) {
    const u32x4 c = __builtin_nontemporal_load(cv + v);
    take(c.x);
    take(c.y);
    take(c.z);
    take(c.w);
  }
  if (blockIdx.x == 0 && tid < (int)(n - n_vec * 4)) take(counts[n_vec * 4 + tid]);  // the last n % 4 rows
  if (run) atomicAdd(&lh[last], run);
  __syncthreads();
  for (int b = tid; b < kHistBins; b += kBlock)
    if (lh[b]) atomicAdd(&ws->hist[b], lh[b]);
}

// one workgroup: the digit d with  #(bins above d) < remaining <= #(bins at or above d)
__global__ __launch_bounds__(kBlock) void rank_pick_kernel(RankWs *ws, int mode, int shift, int with_split) {
  constexpr int kPer = kHistBins / kBlock;  // 8 bins per thread
  __shared__ unsigned long long suffix[kBlock + 1];
  const int tid = threadIdx.x;
  if (ws->from_bitmap || (mode == 1 && ws->settled)) return;  // uniform: nothing was counted either
  uint32_t h[kPer];
  unsigned long long mine = 0;
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    h[j] = ws->hist[tid * kPer + j];
    mine += h[j];
  }
  suffix[tid] = mine;
  if (tid == 0) suffix[kBlock] = 0;
  __syncthreads();
  for (int s = 1; s < kBlock; s <<= 1) {  // inclusive suffix sums
    const unsigned long long add = tid + s < kBlock ? suffix[tid + s] : 0;
    __syncthreads();
    suffix[tid] += add;
    __syncthreads();
  }
  const unsigned long long need = ws->remaining;
  __syncthreads();
  if (suffix[tid] >= need && suffix[tid + 1] < need) {
    unsigned long long above = suffix[tid + 1];
#pragma unroll
    for (int j = kPer - 1; j >= 0; --j) {
      if (above + h[j] >= need) {
        const uint32_t d = (uint32_t)(tid * kPer + j);
        if (mode == 0) {
          if (d < kSatCount) {  // counts below the saturation value are exact: T is known
            ws->count_t = d;
            ws->remaining = need - above;
            ws->settled = 1;
            if (with_split) ws->split_done = d == ws->guess_t;
          }
        } else {
          ws->count_t |= d << shift;
          ws->remaining = need - above;
        }
        break;
      }
      above += h[j];
    }
  }
#pragma unroll
  for (int j = 0; j < kPer; ++j) ws->hist[tid * kPer + j] = 0;
}

__global__ void rank_init_kernel(RankWs *ws, unsigned long long remaining) {
  const int tid = threadIdx.x;
  if (tid == 0) {
    ws->threshold = 0;
    ws->remaining = remaining;
    ws->count_t = 0;
    ws->settled = 0;
    ws->last_row = 0;
    ws->from_bitmap = 0;
    ws->keep_mode = 0;
    ws->guess_t = ws->last_t;
    ws->split_done = 0;
  }
  for (int b = tid; b < kHistBins; b += blockDim.x) ws->hist[b] = 0;
}

// bit r of gt = count[r] > T, of eq = count[r] == T.  A wavefront takes 64 consecutive rows per load, so a ballot is
// a word.
constexpr int kMarkWords = 16;  // words (loads in flight) per wavefront and round
__global__ __launch_bounds__(kBlock) void rank_split_kernel(uint32_t *counts, uint64_t n, const RankWs *ws,
                                                            unsigned long long *gt, unsigned long long *eq,
                                                            int reset_counts) {
  if (ws->from_bitmap || ws->split_done) return;
  const uint32_t t = ws->count_t;
  const int lane = (int)lane_id();
  const uint64_t n_words = (n + 63) / 64;
  const uint64_t wave = ((uint64_t)blockIdx.x * kBlock + threadIdx.x) / kWave;
  const uint64_t n_waves = (uint64_t)gridDim.x * (kBlock / kWave);
  for (uint64_t w0 = wave * kMarkWords; w0 < n_words; w0 += n_waves * kMarkWords) {
    uint32_t c[kMarkWords];
#pragma unroll
    for (int k = 0; k < kMarkWords; ++k) {
      const uint64_t row = (w0 + k) * 64 + lane;
      c[k] = row < n ? __builtin_nontemporal_load(counts + row) : 0u;
    }
    // lane k keeps word k of the round; the words leave in one store per bitmap, as one run of adjacent words
    unsigned long long my_gt = 0, my_eq = 0;
#pragma unroll
    for (int k = 0; k < kMarkWords; ++k) {
      const uint64_t row = (w0 + k) * 64 + lane;
      const unsigned long long above = __ballot(row < n && c[k] > t);
      const unsigned long long equal = __ballot(row < n && c[k] == t);
      if (lane == k) {
        my_gt = above;
        my_eq = equal;
      }
      // a group of 64 counters with any of them above zero is cleared as a whole: two full lines written, where the
      // counters above zero alone would be partial writes that the memory side turns into a read and a write each
      // (500 M counters, 43 M of them above zero: the placement takes 1.13 ms this way and took 1.67 ms the other)
      const bool any_counted = __ballot(row < n && c[k] != 0) != 0ull;
      if (reset_counts && any_counted && row < n) counts[row] = 0;
    }
    if (lane < kMarkWords && w0 + lane < n_words) {
      gt[w0 + lane] = my_gt;
      eq[w0 + lane] = my_eq;
    }
  }
}

// The first pass over the counters (histogram of min(count, 2047), as rank_hist_kernel in mode 0) that also splits on
// its way by a guess of T, the T of the placement before: counters that are kept from refresh to refresh only grow, and
// the K-th best count moves slowly, so the guess is mostly right and the second pass over the counters (2 GB at
// 500 M rows) is not needed (rank_pick_kernel compares, rank_split_kernel leaves at once).  A wrong guess costs the
// two bitmaps written in vain.  Never with a reset of the counters: the second pass would find them cleared.
__global__ __launch_bounds__(kBlock) void rank_hist_split_kernel(const uint32_t *__restrict__ counts, uint64_t n,
                                                                 RankWs *ws, unsigned long long *gt,
                                                                 unsigned long long *eq) {
  if (ws->from_bitmap) return;
  __shared__ uint32_t lh[kHistBins];
  const int tid = threadIdx.x;
  for (int b = tid; b < kHistBins; b += kBlock) lh[b] = 0;
  __syncthreads();
  const uint32_t t = ws->guess_t;
  const int lane = (int)lane_id();
  const uint64_t n_words = (n + 63) / 64;
  const uint64_t wave = ((uint64_t)blockIdx.x * kBlock + tid) / kWave;
  const uint64_t n_waves = (uint64_t)gridDim.x * (kBlock / kWave);
  uint32_t last = 0, run = 0;  // a lane keeps a run of equal digits (the cold rows all share one)
  for (uint64_t w0 = wave * kMarkWords; w0 < n_words; w0 += n_waves * kMarkWords) {
    uint32_t c[kMarkWords];
#pragma unroll
    for (int k = 0; k < kMarkWords; ++k) {
      const uint64_t row = (w0 + k) * 64 + lane;
      c[k] = row < n ? __builtin_nontemporal_load(counts + row) : 0u;
    }
    unsigned long long my_gt = 0, my_eq = 0;
#pragma unroll
    for (int k = 0; k < kMarkWords; ++k) {
      const uint64_t row = (w0 + k) * 64 + lane;
      const unsigned long long above = __ballot(row < n && c[k] > t);
      const unsigned long long equal = __ballot(row < n && c[k] == t);
      if (lane == k) {
        my_gt = above;
        my_eq = equal;
      }
      if (row < n) {
        const uint32_t d = c[k] < kSatCount ? c[k] : kSatCount;
        if (d == last) {
          ++run;
        } else {
          if (run) atomicAdd(&lh[last], run);
          last = d;
          run = 1;
        }
      }
    }
    if (lane < kMarkWords && w0 + lane < n_words) {
      gt[w0 + lane] = my_gt;
      eq[w0 + lane] = my_eq;
    }
  }
  if (run) atomicAdd(&lh[last], run);
  __syncthreads();
  for (int b = tid; b < kHistBins; b += kBlock)
    if (lh[b]) atomicAdd(&ws->hist[b], lh[b]);
}

// after the observed rows were counted (ws->bm.total): fewer than wanted means every observed row is in and the rest
// comes from the never-observed ones, lowest row first
__global__ void rank_decide_kernel(RankWs *ws) {
  if (ws->bm.total < ws->remaining) {
    ws->from_bitmap = 1;
    ws->settled = 1;
    ws->count_t = 0;
    ws->remaining -= ws->bm.total;
  }
}

// the split of that case: gt = observed, eq = ~observed; counters of observed rows reset on request
__global__ __launch_bounds__(kBlock) void rank_split_bitmap_kernel(uint32_t *counts, uint64_t n, const RankWs *ws,
                                                                   const unsigned long long *observed,
                                                                   unsigned long long *gt, unsigned long long *eq,
                                                                   int reset_counts) {
  if (!ws->from_bitmap) return;
  const uint64_t n_words = (n + 63) / 64;
  for (uint64_t w = (uint64_t)blockIdx.x * kBlock + threadIdx.x; w < n_words; w += (uint64_t)gridDim.x * kBlock) {
    unsigned long long m = observed[w];
    unsigned long long rest = ~m;
    if (n - w * 64 < 64) rest &= (1ull << (n - w * 64)) - 1ull;
    gt[w] = m;
    eq[w] = rest;
    if (reset_counts)
      while (m) {
        counts[w * 64 + __builtin_ctzll(m)] = 0;
        m &= m - 1;
      }
  }
}

// with a keep bitmap, after eq & keep was counted (ws->bm.total): enough of them means the needed rows are all kept
// ones; otherwise every kept one is in and the rest is looked for among the others
__global__ void rank_keep_decide_kernel(RankWs *ws) {
  if (ws->bm.total >= ws->remaining) {
    ws->keep_mode = 1;
  } else {
    ws->keep_mode = 2;
    ws->remaining -= ws->bm.total;
  }
}

// the rows with count T among which the last needed one is looked for
__device__ __forceinline__ unsigned long long tie_word(const RankWs *ws, const unsigned long long *eq,
                                                       const unsigned long long *keep, uint64_t w) {
  unsigned long long m = eq[w];
  if (keep) m &= ws->keep_mode == 1 ? keep[w] : ~keep[w];
  return m;
}

// one workgroup: the row of the last needed bit of eq.  With T > 0 the needed rows are the `remaining` topmost set
// bits, the last of them is bit number total - remaining (counted from the bottom, from 0); with T == 0 they are the
// lowest ones, the last is number remaining - 1.
__global__ __launch_bounds__(kBlock) void rank_locate_kernel(RankWs *ws, const unsigned long long *eq,
                                                             const unsigned long long *keep, uint64_t nbits,
                                                             uint64_t per_chunk) {
  __shared__ uint32_t chunk_of;
  const int tid = threadIdx.x;
  const uint32_t total = ws->bm.total;
  const uint32_t index = ws->count_t ? total - (uint32_t)ws->remaining : (uint32_t)ws->remaining - 1u;
  if (tid == 0) ws->last_t = ws->count_t;  // the next placement's guess
  constexpr int kPer = kBmChunks / kBlock;
  for (int j = 0; j < kPer; ++j) {
    const int c = tid * kPer + j;
    const uint32_t lo = ws->bm.base[c], hi = c + 1 < kBmChunks ? ws->bm.base[c + 1] : total;
    if (lo <= index && index < hi) chunk_of = (uint32_t)c;  // exactly one chunk holds it
  }
  __syncthreads();
  if (tid >= kWave) return;
  const uint32_t c = chunk_of;
  const uint64_t n_words = (nbits + 63) / 64;
  const uint64_t begin = (uint64_t)c * per_chunk, end = min(n_words, begin + per_chunk);
  uint32_t skip = index - ws->bm.base[c];  // set bits of the chunk below the wanted one
  for (uint64_t w0 = begin; w0 < end; w0 += kWave) {
    const uint64_t w = w0 + tid;
    unsigned long long m = w < end ? tie_word(ws, eq, keep, w) : 0ull;
    const uint32_t mine = __popcll(m);
    const uint32_t incl = wave_incl_sum(mine);
    const uint32_t all = __shfl(incl, kWave - 1);
    if (skip < all) {  // in this group of words; wavefront-uniform
      if (incl - mine <= skip && skip < incl) {
        uint32_t drop = skip - (incl - mine);
        while (drop--) m &= m - 1;
        const uint32_t row = (uint32_t)(w * 64 + __builtin_ctzll(m));
        ws->last_row = row;
        ws->threshold = rank_of(ws->count_t, row);
      }
      return;
    }
    skip -= all;
  }
}

// in_new = gt | (eq on the needed side of last_row); gt is in_new itself.  With a keep bitmap the side is taken of
// eq & keep (mode 1) or of eq & ~keep on top of all of eq & keep (mode 2).
__global__ __launch_bounds__(kBlock) void rank_combine_kernel(const RankWs *ws, unsigned long long *in_new,
                                                              const unsigned long long *eq,
                                                              const unsigned long long *keep, uint64_t n_words,
                                                              unsigned long long *observed_to_clear) {
  const uint64_t wl = ws->last_row >> 6;
  const unsigned bl = ws->last_row & 63u;
  const bool upward = ws->count_t != 0;  // rows at and above last_row, or at and below it
  for (uint64_t w = (uint64_t)blockIdx.x * kBlock + threadIdx.x; w < n_words; w += (uint64_t)gridDim.x * kBlock) {
    unsigned long long mask;
    if (upward) mask = w > wl ? ~0ull : (w == wl ? ~0ull << bl : 0ull);
    else mask = w < wl ? ~0ull : (w == wl ? (bl == 63 ? ~0ull : (1ull << (bl + 1)) - 1ull) : 0ull);
    unsigned long long add = tie_word(ws, eq, keep, w) & mask;
    if (keep && ws->keep_mode == 2) add |= eq[w] & keep[w];
    in_new[w] |= add;
    if (observed_to_clear) observed_to_clear[w] = 0;  // the counters were reset: no row is observed any more
  }
}

// The counts of all chunks scanned by one workgroup of kScanBlock threads, eight neighbouring chunks a thread, in registers:
// pre[j] = counts in front of chunk 8 * tid + j, total = all of them.  (With 256 threads, a scan in LDS and the counts read
// from memory twice rank_locate_unobserved_kernel took 13.5 us; 5.7 this way.)
constexpr int kScanBlock = kBmChunks / 8;
__device__ __forceinline__ void scan_chunks(const uint32_t *counts, uint32_t (&pre)[8], uint32_t &total) {
  constexpr int kWaves = kScanBlock / kWave;
  __shared__ uint32_t wave_sum[kWaves];
  const int tid = threadIdx.x, lane = tid % kWave;
  // (a workspace is 8-byte aligned)
  const u32x4_by4 *c4 = reinterpret_cast<const u32x4_by4 *>(counts) + 2 * tid;
  const u32x4 lo = c4[0], hi = c4[1];
  const uint32_t c[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
  uint32_t sum = 0;
#pragma unroll
  for (int j = 0; j < 8; ++j) pre[j] = sum, sum += c[j];
  const uint32_t incl = wave_incl_sum(sum);
  if (lane == kWave - 1) wave_sum[tid / kWave] = incl;
  __syncthreads();
  uint32_t before = incl - sum;
  total = 0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    if (w < tid / kWave) before += wave_sum[w];
    total += wave_sum[w];
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) pre[j] += before;
}

// ---- the placement when the caller knows that fewer rows were observed than are wanted ----------------------------
// One workgroup, after `observed` was counted into ws->bm: scans the chunk counts, checks the caller's promise and
// finds the last needed never-observed row, the (want - observed rows - 1)-th clear bit of `observed`, ascending (clear
// bits in front of chunk c = its first bit number - set bits in front of it).  Three dependent reads: the chunk counts,
// the block counts of the one chunk, the 64 words of the one block.
__global__ __launch_bounds__(kScanBlock) void rank_locate_unobserved_kernel(RankWs *ws, const unsigned long long *observed,
                                                                            uint64_t nbits, uint64_t per_chunk,
                                                                            unsigned long long want, uint32_t *status,
                                                                            uint32_t *observed_host) {
  __shared__ uint32_t chunk_of;
  __shared__ uint64_t skip_of;
  const int tid = threadIdx.x;
  if (tid == 0) {  // what rank_init_kernel sets, for the readers of a placement (the histogram is not used here)
    ws->threshold = 0;
    ws->remaining = want;
    ws->count_t = 0;
    ws->settled = 0;
    ws->last_row = 0;
    ws->from_bitmap = 0;
    ws->keep_mode = 0;
    ws->scans_done = 0;
  }
  for (uint32_t i = tid; i < (kArriveLines + 1) * 16; i += kScanBlock) (&ws->arrivals.line[0][0])[i] = 0ull;
  uint32_t pre[8], total;
  scan_chunks(ws->bm.base, pre, total);
  if (tid == 0) ws->bm.total = total;
  if (tid == 0 && observed_host) *observed_host = total;
  if (total >= want) {  // uniform: the promise does not hold, nothing is placed
    if (tid == 0) atomicOr(status, UGK_ST_PLACE_PROMISE);
    return;
  }
  const uint64_t index = want - total - 1;  // among the clear bits, from 0
  const uint64_t chunk_bits = per_chunk * 64;
  // the last chunk with no more than `index` clear bits in front of it holds the bit, and it is the one whose clear bits
  // reach beyond: exactly one chunk
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const uint64_t c = (uint64_t)tid * 8 + j;
    const uint64_t first = min(c * chunk_bits, nbits), behind = min((c + 1) * chunk_bits, nbits);
    const uint64_t lo = first - pre[j];
    // set bits up to the chunk's end: the next one's prefix, which the last of a thread's eight finds from its count
    const uint32_t upto = j < 7 ? pre[j < 7 ? j + 1 : 7] : pre[7] + ws->bm.base[c];
    if (lo <= index && index < behind - upto) chunk_of = (uint32_t)c, skip_of = index - lo;
  }
  __syncthreads();
  if (tid >= kWave) return;
  const uint32_t c = chunk_of;
  const uint64_t n_words = (nbits + 63) / 64;
  const uint64_t n_blocks = (n_words + kWave - 1) / kWave;
  const uint64_t blocks_per_chunk = per_chunk / kWave, first_blk = (uint64_t)c * blocks_per_chunk;
  constexpr uint64_t kBlockBits = (uint64_t)kWave * 64;
  uint64_t skip = skip_of;  // clear bits of the chunk below the wanted one
  // the block: a lane per block of the chunk
  uint64_t blk = 0;
  bool found = false;
  for (uint64_t b0 = 0; b0 < blocks_per_chunk && !found; b0 += kWave) {
    const uint64_t b = first_blk + b0 + tid;
    uint32_t mine = 0;
    if (b0 + tid < blocks_per_chunk && b < n_blocks) {
      const uint64_t bits = min(nbits - b * kBlockBits, kBlockBits);
      mine = (uint32_t)bits - ws->bm.block[b];
    }
    const uint32_t incl = wave_incl_sum(mine);
    const uint32_t all = __shfl(incl, kWave - 1);
    if (skip < all) {  // wavefront-uniform
      const unsigned long long holds = __ballot(incl - mine <= skip && skip < incl);
      const int src = __builtin_ctzll(holds);
      blk = first_blk + b0 + src;
      skip -= __shfl(incl - mine, src);
      found = true;
    } else {
      skip -= all;
    }
  }
  if (!found) return;  // cannot be: the chunk holds the bit
  // the word and the bit: a lane per word of the block
  const uint64_t w = blk * kWave + tid;
  unsigned long long m = 0ull;
  if (w < n_words) {
    m = ~observed[w];
    if (nbits - w * 64 < 64) m &= (1ull << (nbits - w * 64)) - 1ull;
  }
  const uint32_t mine = __popcll(m);
  const uint32_t incl = wave_incl_sum(mine);
  if (incl - mine <= skip && skip < incl) {
    uint32_t drop = (uint32_t)skip - (incl - mine);
    while (drop--) m &= m - 1;
    const uint32_t row = (uint32_t)(w * 64 + __builtin_ctzll(m));
    ws->last_row = row;
    ws->threshold = rank_of(0u, row);
    ws->remaining = want - total;
    ws->from_bitmap = 1;
    ws->settled = 1;
  }
}

// in_new = observed | (never observed, up to last_row); with `cached`, the rows that leave (cached & ~in_new) and come
// in (in_new & ~cached) are counted per 64-word block and per chunk on the way, as bitmap_count_kernel would, and all in
// all: the last workgroup to end writes both sums to totals_host.  One wavefront per chunk.  With a ticket, which that
// workgroup writes behind the sums, a host that polls for it may go on at once, on any stream: what the refresh reads next is
// written through to memory then (leave_done has the why).  Only a launch that is the placement's last one gets a ticket.
__global__ __launch_bounds__(kBlock) void rank_combine_observed_kernel(uint32_t *counts, uint64_t nbits,
                                                                       uint64_t per_chunk, RankWs *ws,
                                                                       unsigned long long *observed,
                                                                       unsigned long long *in_new,
                                                                       const unsigned long long *cached,
                                                                       BmWs *evict_ws, BmWs *insert_ws,
                                                                       int reset_counts, uint32_t *totals_host,
                                                                       uint32_t ticket) {
  __shared__ uint32_t leaving_of[kBlock / kWave], coming_of[kBlock / kWave];
  if (!ws->from_bitmap) {  // nothing was placed
    if (cached && blockIdx.x == 0 && threadIdx.x == 0) {
      totals_host[0] = totals_host[1] = 0;
      __threadfence_system();
      if (ticket) *(volatile uint32_t *)(totals_host + 3) = ticket;
    }
    return;
  }
  const uint64_t wl = ws->last_row >> 6;
  const unsigned bl = ws->last_row & 63u;
  const int lane = (int)lane_id();
  const uint64_t n_words = (nbits + 63) / 64;
  const uint64_t wave = ((uint64_t)blockIdx.x * kBlock + threadIdx.x) / kWave;
  const uint64_t n_waves = (uint64_t)gridDim.x * (kBlock / kWave);
  auto put = [ticket](auto *to, auto v) {
    if (ticket) store_through(reinterpret_cast<uint64_t>(to), v);
    else *to = v;
  };
  if (cached && blockIdx.x == 0 && threadIdx.x == 0) put(&evict_ws->scanned, 0u), put(&insert_ws->scanned, 0u);
  uint32_t out_all = 0, in_all = 0;
  for (uint64_t chunk = wave; chunk < (uint64_t)kBmChunks; chunk += n_waves) {
    const uint64_t begin = chunk * per_chunk, end = min(n_words, begin + per_chunk);
    uint32_t out_sum = 0, in_sum = 0;
    for (uint64_t w0 = begin; w0 < end; w0 += kWave) {
      const uint64_t w = w0 + lane;
      uint32_t leaving = 0, coming = 0;
      if (w < end) {
        unsigned long long obs = observed[w];
        unsigned long long upto = w < wl ? ~0ull : (w == wl ? (bl == 63 ? ~0ull : (1ull << (bl + 1)) - 1ull) : 0ull);
        if (nbits - w * 64 < 64) upto &= (1ull << (nbits - w * 64)) - 1ull;
        const unsigned long long nw = obs | (~obs & upto);
        put(in_new + w, nw);
        if (cached) {
          const unsigned long long c = cached[w];
          leaving = __popcll(c & ~nw);
          coming = __popcll(nw & ~c);
        }
        if (reset_counts) {
          observed[w] = 0;
          while (obs) {
            counts[w * 64 + __builtin_ctzll(obs)] = 0;
            obs &= obs - 1;
          }
        }
      }
      if (cached) {  // uniform
        leaving = wave_sum(leaving);
        coming = wave_sum(coming);
        if (lane == 0) {
          put(&evict_ws->block[w0 / kWave], leaving);  // chunks begin on block boundaries
          put(&insert_ws->block[w0 / kWave], coming);
        }
        out_sum += leaving;
        in_sum += coming;
      }
    }
    if (cached && lane == 0) {
      put(&evict_ws->base[chunk], out_sum);
      put(&insert_ws->base[chunk], in_sum);
    }
    out_all += out_sum;
    in_all += in_sum;
  }
  if (!cached) return;  // uniform
  if (ticket) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wavefront's stores have been acknowledged
  if (lane == 0) leaving_of[threadIdx.x / kWave] = out_all, coming_of[threadIdx.x / kWave] = in_all;
  __syncthreads();
  if (threadIdx.x != 0) return;
  uint32_t out_wg = 0, in_wg = 0;
#pragma unroll
  for (int w = 0; w < kBlock / kWave; ++w) out_wg += leaving_of[w], in_wg += coming_of[w];
  if (!arrive(&ws->arrivals, out_wg, in_wg)) return;
  // (there before this launch has ended: where a scan behind it leaves the ticket, an ordinary store could be overtaken by that)
  tell_host(totals_host, out_wg);
  tell_host(totals_host + 1, in_wg);
  if (ticket) {
    __threadfence_system();
    *(volatile uint32_t *)(totals_host + 3) = ticket;
  }
}

// every row, or none: bitmap of n set (or clear) bits, counters reset on request
__global__ __launch_bounds__(kBlock) void rank_fill_kernel(uint32_t *counts, uint64_t n, unsigned long long *bitmap,
                                                           int all, int reset_counts, RankWs *ws,
                                                           unsigned long long *observed) {
  const uint64_t n_words = (n + 63) / 64;
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  for (uint64_t w = (uint64_t)blockIdx.x * kBlock + threadIdx.x; w < n_words; w += stride) {
    unsigned long long m = all ? ~0ull : 0ull;
    if (all && n - w * 64 < 64) m = (1ull << (n - w * 64)) - 1ull;
    bitmap[w] = m;
    if (reset_counts && observed) observed[w] = 0;
  }
  if (reset_counts)
    for (uint64_t r = (uint64_t)blockIdx.x * kBlock + threadIdx.x; r < n; r += stride) counts[r] = 0;
  if (blockIdx.x == 0 && threadIdx.x == 0) ws->threshold = all ? 0ull : ~0ull;
}

// ---- bitmaps ----------------------------------------------------------------------------------------------
constexpr int kBmInvertA = 1, kBmAndB = 2;  // flags: ~a instead of a; & b instead of & ~b
__device__ __forceinline__ unsigned long long bm_word(const unsigned long long *a, const unsigned long long *b,
                                                      int flags, uint64_t nbits, uint64_t w) {
  unsigned long long m = a[w];
  if (flags & kBmInvertA) m = ~m;
  if (b) m &= (flags & kBmAndB) ? b[w] : ~b[w];
  const uint64_t first = w * 64;
  if (nbits - first < 64) m &= (1ull << (nbits - first)) - 1ull;  // the last, partial word
  return m;
}

static inline uint64_t bm_words_per_chunk(uint64_t n_words) {
  return ((n_words + kBmChunks - 1) / kBmChunks + kWave - 1) / kWave * kWave;
}

// gate (may be NULL): the placement whose keep_mode must be 2 for the launch to do anything
__global__ __launch_bounds__(kBlock) void bitmap_count_kernel(const unsigned long long *a, const unsigned long long *b,
                                                              int flags, uint64_t nbits, uint64_t per_chunk,
                                                              BmWs *ws, const RankWs *gate) {
  if (gate && gate->keep_mode != 2) return;
  if (blockIdx.x == 0 && threadIdx.x == 0) ws->scanned = 0;
  const int lane = (int)lane_id();
  const uint64_t n_words = (nbits + 63) / 64;
  const uint64_t wave = ((uint64_t)blockIdx.x * kBlock + threadIdx.x) / kWave;
  const uint64_t n_waves = (uint64_t)gridDim.x * (kBlock / kWave);
  for (uint64_t chunk = wave; chunk < (uint64_t)kBmChunks; chunk += n_waves) {
    const uint64_t begin = chunk * per_chunk, end = min(n_words, begin + per_chunk);
    uint32_t found = 0;
    for (uint64_t w0 = begin; w0 < end; w0 += kWave) {
      const uint64_t w = w0 + lane;
      uint32_t mine = w < end ? __popcll(bm_word(a, b, flags, nbits, w)) : 0u;
      mine = wave_sum(mine);
      if (lane == 0) ws->block[w0 / kWave] = mine;  // chunks begin on block boundaries
      found += mine;
    }
    if (lane == 0) ws->base[chunk] = found;
  }
}

// bitmap_count_kernel for a & ~b and b & ~a at once: the two bitmaps are read once, both workspaces are left as two
// counts would leave them
__global__ __launch_bounds__(kBlock) void bitmap_count_diff_kernel(const unsigned long long *a,
                                                                   const unsigned long long *b, uint64_t nbits,
                                                                   uint64_t per_chunk, BmWs *ws_ab, BmWs *ws_ba) {
  const int lane = (int)lane_id();
  const uint64_t n_words = (nbits + 63) / 64;
  const uint64_t wave = ((uint64_t)blockIdx.x * kBlock + threadIdx.x) / kWave;
  const uint64_t n_waves = (uint64_t)gridDim.x * (kBlock / kWave);
  for (uint64_t chunk = wave; chunk < (uint64_t)kBmChunks; chunk += n_waves) {
    const uint64_t begin = chunk * per_chunk, end = min(n_words, begin + per_chunk);
    uint32_t sum_ab = 0, sum_ba = 0;
    for (uint64_t w0 = begin; w0 < end; w0 += kWave) {
      const uint64_t w = w0 + lane;
      uint32_t n_ab = 0, n_ba = 0;
      if (w < end) {
        unsigned long long wa = a[w], wb = b[w];
        if (nbits - w * 64 < 64) {  // the last, partial word
          const unsigned long long valid = (1ull << (nbits - w * 64)) - 1ull;
          wa &= valid;
          wb &= valid;
        }
        n_ab = __popcll(wa & ~wb);
        n_ba = __popcll(wb & ~wa);
      }
      n_ab = wave_sum(n_ab);
      n_ba = wave_sum(n_ba);
      if (lane == 0) {
        ws_ab->block[w0 / kWave] = n_ab;  // chunks begin on block boundaries
        ws_ba->block[w0 / kWave] = n_ba;
      }
      sum_ab += n_ab;
      sum_ba += n_ba;
    }
    if (lane == 0) {
      ws_ab->base[chunk] = sum_ab;
      ws_ba->base[chunk] = sum_ba;
    }
  }
}

// one workgroup of kScanBlock threads: the counts of the chunks become their prefix
template <bool THROUGH>
__device__ __forceinline__ void scan_ws(BmWs *ws, uint32_t *total_host) {
  auto put = [](uint32_t *to, auto v) {
    typedef decltype(v) __attribute__((aligned(4))) by4_t;
    if constexpr (THROUGH) store_through(reinterpret_cast<uint64_t>(to), v);
    else *reinterpret_cast<by4_t *>(to) = v;
  };
  uint32_t pre[8], total;
  scan_chunks(ws->base, pre, total);
  uint32_t *to = ws->base + 8 * threadIdx.x;
  put(to, u32x4{pre[0], pre[1], pre[2], pre[3]});
  put(to + 4, u32x4{pre[4], pre[5], pre[6], pre[7]});
  if (threadIdx.x == 0) {
    put(&ws->total, total);
    put(&ws->scanned, 1u);
    if (total_host) *total_host = total;
  }
}

__global__ __launch_bounds__(kScanBlock) void bitmap_scan_kernel(BmWs *ws, uint32_t *total_host, const RankWs *gate) {
  if (gate && gate->keep_mode != 2) return;
  scan_ws<false>(ws, total_host);
}

// two workspaces in one launch (one workgroup each), totals to totals_host[0] and [1]
__global__ __launch_bounds__(kScanBlock) void bitmap_scan2_kernel(BmWs *a, BmWs *b, uint32_t *totals_host) {
  scan_ws<false>(blockIdx.x == 0 ? a : b, totals_host ? totals_host + blockIdx.x : (uint32_t *)nullptr);
}

// The same behind a placement whose end the host polls for: the prefixes are the last of what the refresh reads next, so they
// are written through and the workgroup that finishes second leaves the ticket (a ticket left by the placement itself let
// the lists on another stream start in front of the scan).
__global__ __launch_bounds__(kScanBlock) void bitmap_scan2_ticket_kernel(BmWs *a, BmWs *b, RankWs *placed,
                                                                         uint32_t *ticket_host, uint32_t ticket) {
  if (placed->from_bitmap) scan_ws<true>(blockIdx.x == 0 ? a : b, nullptr);  // else nothing was placed or counted
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wavefront's stores have been acknowledged
  __syncthreads();
  if (threadIdx.x != 0) return;
  if (__hip_atomic_fetch_add(&placed->scans_done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 1u) return;
  __threadfence_system();
  *(volatile uint32_t *)ticket_host = ticket;
}

// The set bits of one 64-word block, a lane per word on entry (m), to out[pos0 ...] in ascending order; n_set: how
// many there are (wavefront-uniform).  A block with few bits: every lane walks the bits of its own word (a step or
// two).  A block with many: the wavefront takes the non-zero words one at a time, a lane per bit, one store of
// consecutive positions per word and at most 64 of them (a lane per word would store at 64 scattered places per step,
// 64 steps for a block of all ones: a contiguous run of rows that leave the cache kept a handful of wavefronts busy
// long after the rest had finished; for blocks with a few bits the word-at-a-time form is the slower one, 51 against
// 37 us over 122 k blocks with four bits each).
constexpr uint32_t kEmitDense = 2 * kWave;
__device__ __forceinline__ uint32_t set_bits_upto(unsigned long long m) {  // in the words of this lane and the ones below
  return wave_incl_sum(__popcll(m));
}
__device__ __forceinline__ uint64_t uniform64(uint64_t x) {  // a value that all lanes have, in scalar registers
  return ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(x >> 32)) << 32) |
         (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)x);
}
__device__ __forceinline__ void emit_word(unsigned long long m, uint32_t incl, uint32_t n_set, uint64_t pos0, uint64_t w,
                                          int lane, uint32_t *out, uint64_t max_out) {
  const uint32_t excl = incl - __popcll(m);
  if (n_set <= kEmitDense) {
    uint64_t pos = pos0 + excl;
    while (m) {
      const int bit = __builtin_ctzll(m);
      m &= m - 1;
      if (pos < max_out) out[pos] = (uint32_t)(w * 64 + bit);
      ++pos;
    }
    return;
  }
  if (pos0 >= max_out) return;
  // What is the same in all lanes is in scalar registers, so that a word is two bit counts, the value and the store, and the
  // positions of four words are worked out before the first of them is stored (unrolled further the code of a block no longer
  // stays in the instruction cache beside the rest: lists of scattered bits 1.5 us longer).
  const uint64_t blk_pos = uniform64(pos0), room64 = max_out - blk_pos;
  const uint32_t room = room64 < n_set ? (uint32_t)room64 : n_set;  // entries of the block that the list has room for
  const uint32_t w_first = (uint32_t)uniform64(w - (uint64_t)lane);
  uint32_t *const to = out + blk_pos;
  const unsigned long long todo = __ballot(m != 0ull);
  constexpr int kAtOnce = 4;
#pragma unroll 1
  for (int src = 0; src < kWave; src += kAtOnce) {  // wavefront-uniform
    if (((todo >> src) & ((1u << kAtOnce) - 1u)) == 0) continue;
    unsigned long long word[kAtOnce];
    uint32_t pos[kAtOnce];
#pragma unroll
    for (int u = 0; u < kAtOnce; ++u) {
      const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)m, src + u);
      const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(m >> 32), src + u);
      const uint32_t before = (uint32_t)__builtin_amdgcn_readlane((int)excl, src + u);
      word[u] = ((unsigned long long)hi << 32) | lo;
      pos[u] = __builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, before));
    }
#pragma unroll
    for (int u = 0; u < kAtOnce; ++u)
      if (__builtin_amdgcn_inverse_ballot_w64(word[u]) && pos[u] < room)
        to[pos[u]] = (w_first + (uint32_t)(src + u)) * 64 + (uint32_t)lane;
  }
}

__global__ __launch_bounds__(kBlock) void bitmap_emit_kernel(const unsigned long long *a, const unsigned long long *b,
                                                             int flags, uint64_t nbits, uint64_t per_chunk,
                                                             const BmWs *ws, uint32_t *out, uint64_t max_out,
                                                             uint32_t *total_host) {
  if (total_host && blockIdx.x == 0 && threadIdx.x == 0) *total_host = ws->total;
  const int lane = (int)lane_id();
  const uint64_t n_words = (nbits + 63) / 64;
  const uint64_t n_blocks = (n_words + kWave - 1) / kWave;
  const uint64_t wave = ((uint64_t)blockIdx.x * kBlock + threadIdx.x) / kWave;
  const uint64_t n_waves = (uint64_t)gridDim.x * (kBlock / kWave);
  const uint64_t blocks_per_chunk = per_chunk / kWave;
  for (uint64_t blk = wave; blk < n_blocks; blk += n_waves) {
    const uint32_t n_here = ws->block[blk];
    if (n_here == 0) continue;  // wavefront-uniform
    // where the block's elements go: its chunk's offset plus the counts of the chunk's earlier blocks
    const uint64_t chunk = blk / blocks_per_chunk, first = chunk * blocks_per_chunk;
    uint32_t before = 0;
    for (uint64_t q = first + lane; q < blk; q += kWave) before += ws->block[q];
    before = wave_sum(before);
    const uint64_t pos0 = (uint64_t)ws->base[chunk] + before;
    if (pos0 >= max_out) continue;
    const uint64_t w = blk * kWave + lane;
    unsigned long long m = w < n_words ? bm_word(a, b, flags, nbits, w) : 0ull;
    emit_word(m, set_bits_upto(m), n_here, pos0, w, lane, out, max_out);
  }
}

// Both differences of two bitmaps in one pass, a & ~b -> out_ab and b & ~a -> out_ba, each list as bitmap_emit_kernel
// writes it from its own counts (ws_ab, ws_ba).  The small arrays of counts are read before it is known whether the
// block holds anything, the two words of the bitmaps only when it does: two dependent reads per block.
constexpr int kDiffBlocks = 1;  // consecutive blocks per wavefront and round
__global__ __launch_bounds__(kBlock) void bitmap_emit_diff_kernel(const unsigned long long *a,
                                                                  const unsigned long long *b, uint64_t nbits,
                                                                  uint64_t per_chunk, const BmWs *ws_ab,
                                                                  const BmWs *ws_ba, uint32_t *out_ab, uint64_t max_ab,
                                                                  uint32_t *out_ba, uint64_t max_ba) {
  const int lane = (int)lane_id();
  const uint64_t n_words = (nbits + 63) / 64;
  const uint64_t n_blocks = (n_words + kWave - 1) / kWave;
  const uint64_t n_groups = (n_blocks + kDiffBlocks - 1) / kDiffBlocks;
  const uint64_t wave = ((uint64_t)blockIdx.x * kBlock + threadIdx.x) / kWave;
  const uint64_t n_waves = (uint64_t)gridDim.x * (kBlock / kWave);
  const uint64_t blocks_per_chunk = per_chunk / kWave;
  for (uint64_t grp = wave; grp < n_groups; grp += n_waves) {
    const uint64_t blk0 = grp * kDiffBlocks;
    // first round, all of it asked for at once: the counts of the group's blocks, the counts in front of its first
    // block inside that block's chunk, the chunk offsets
    uint32_t n_ab[kDiffBlocks], n_ba[kDiffBlocks];
    uint64_t base_ab[kDiffBlocks], base_ba[kDiffBlocks];
#pragma unroll
    for (int j = 0; j < kDiffBlocks; ++j) {
      const uint64_t blk = min(blk0 + j, n_blocks - 1);
      const bool valid = blk0 + j < n_blocks;
      n_ab[j] = valid ? ws_ab->block[blk] : 0u;
      n_ba[j] = valid ? ws_ba->block[blk] : 0u;
      base_ab[j] = ws_ab->base[blk / blocks_per_chunk];
      base_ba[j] = ws_ba->base[blk / blocks_per_chunk];
    }
    uint32_t before_ab = 0, before_ba = 0;
    for (uint64_t q = blk0 / blocks_per_chunk * blocks_per_chunk + lane; q < blk0; q += kWave) {
      before_ab += ws_ab->block[q];
      before_ba += ws_ba->block[q];
    }
    uint32_t any = 0;
#pragma unroll
    for (int j = 0; j < kDiffBlocks; ++j) any |= n_ab[j] | n_ba[j];
    if (any == 0) continue;  // wavefront-uniform
    before_ab = wave_sum(before_ab);
    before_ba = wave_sum(before_ba);
    // where each block's elements go: its chunk's offset plus the counts of the chunk's earlier blocks
    uint64_t pos_ab[kDiffBlocks], pos_ba[kDiffBlocks];
#pragma unroll
    for (int j = 0; j < kDiffBlocks; ++j) {
      if (j > 0) {
        const bool new_chunk = (blk0 + j) % blocks_per_chunk == 0;
        before_ab = new_chunk ? 0u : before_ab + n_ab[j - 1];
        before_ba = new_chunk ? 0u : before_ba + n_ba[j - 1];
      }
      pos_ab[j] = base_ab[j] + before_ab;
      pos_ba[j] = base_ba[j] + before_ba;
    }
    // second round: the words of the blocks that hold anything that is still wanted
    unsigned long long wa[kDiffBlocks], wb[kDiffBlocks];
    bool do_ab[kDiffBlocks], do_ba[kDiffBlocks];
#pragma unroll
    for (int j = 0; j < kDiffBlocks; ++j) {
      do_ab[j] = n_ab[j] != 0 && pos_ab[j] < max_ab;
      do_ba[j] = n_ba[j] != 0 && pos_ba[j] < max_ba;
      const uint64_t w = (blk0 + j) * kWave + lane;
      wa[j] = wb[j] = 0ull;
      if ((do_ab[j] || do_ba[j]) && w < n_words) {
        wa[j] = a[w];
        wb[j] = b[w];
        if (nbits - w * 64 < 64) {  // the last, partial word
          const unsigned long long valid = (1ull << (nbits - w * 64)) - 1ull;
          wa[j] &= valid;
          wb[j] &= valid;
        }
      }
    }
#pragma unroll
    for (int j = 0; j < kDiffBlocks; ++j) {
      const uint64_t w = (blk0 + j) * kWave + lane;
      const unsigned long long ab = wa[j] & ~wb[j], ba = wb[j] & ~wa[j];
      if (do_ab[j]) emit_word(ab, set_bits_upto(ab), n_ab[j], pos_ab[j], w, lane, out_ab, max_ab);
      if (do_ba[j]) emit_word(ba, set_bits_upto(ba), n_ba[j], pos_ba[j], w, lane, out_ba, max_ba);
    }
  }
}

// The emit pass over a bitmap of up to kSmallBits bits, whose chunks are at most kSmallBlocks blocks long: a wavefront per chunk, which
// asks for its words together with the counts it needs to know its place, where no scan has run: one round of reads, and
// no one-workgroup launch between the count and this one.  Longer chunks would make a wavefront of a dense one work long after
// the others.
// Wavefront v of workgroup b takes chunk v * grid + b, so that neighbouring chunks, which are dense together where rows or slots are
// set in one run, are on different CUs, and adds up the counts of its strip of the chunks, v * grid and on: all of
// them for the other wavefronts of the workgroup, those in front of its own chunk for itself.
// us, the list alone / a scan and a wavefront per 64-word block (what it replaces) / a workgroup taking neighbouring chunks, one word at a
// time with its positions in 64-bit vector registers: 50.5 M bits, 461,000 of them in one run 10.6 / 5.0 + 8.8 / 24.0, scattered 5.5 /
// 5.0 + 6.3 / 5.5, 5 M in one run 15.0 / 5.0 + 12.1 / 26.0; 4 M bits, 72,000 in one run 6.2 / 5.0 + 8.0 / 10.8, scattered 4.0 / 5.0 + 3.9 /
// 4.0, all 9.1 / 5.0 + 10.4 / 15.4; 100,000 bits, all 6.1 / 5.0 + 8.2 / 12.8; two lists out of 40 M bits, 72,000 each, scattered 6.2 /
// 5.0 + 6.6 / 6.6, one of them a run 10.9 / 5.0 + 8.5 / 14.7, 60 M bits and 461,000 each 13.8 / 5.0 + 9.3 / 25.2.
constexpr uint64_t kSmallBlocks = 2, kSmallBits = (uint64_t)kBmChunks * kSmallBlocks * kWave * 64;
constexpr uint32_t kSmallStrip = 512, kSmallWaves = kBmChunks / kSmallStrip;
struct SmallGrid {
  unsigned groups, threads;
  SmallGrid(uint64_t nbits, uint64_t per_chunk) {
    const uint32_t chunks = (uint32_t)(((nbits + 63) / 64 + per_chunk - 1) / per_chunk);  // that hold any word
    const uint32_t waves = (chunks + kSmallStrip - 1) / kSmallStrip;
    groups = (chunks + waves - 1) / waves;
    threads = waves * kWave;
  }
};
struct BmList {
  const BmWs *ws;
  uint32_t *out;
  uint64_t max_out;
};
// sets S of one (LISTS == 1: bm_word's of a and b) or two lists (a & ~b, b & ~a); total_host (LISTS == 1): |S|
template <int LISTS>
__global__ __launch_bounds__(kSmallWaves * kWave) void bitmap_emit_small_kernel(const unsigned long long *a,
                                                                                const unsigned long long *b, int flags,
                                                                                uint64_t nbits, uint64_t per_chunk,
                                                                                BmList first, BmList second,
                                                                                uint32_t *total_host) {
  __shared__ uint32_t part[LISTS][kSmallWaves];
  const BmList list[2] = {first, second};
  const int lane = (int)lane_id(), wv = (int)wave_in_block(), waves = (int)(blockDim.x / kWave);
  const uint64_t n_words = (nbits + 63) / 64;
  const uint32_t strip = (uint32_t)wv * gridDim.x, chunk = strip + blockIdx.x;  // below kBmChunks
  const uint64_t w_first = (uint64_t)chunk * per_chunk + lane;
  unsigned long long m[LISTS][kSmallBlocks];
#pragma unroll
  for (uint64_t j = 0; j < kSmallBlocks; ++j) {
    const uint64_t w = w_first + j * kWave;
    const bool in = j * kWave < per_chunk && w < n_words;
    const uint64_t at = in ? w : 0;  // no branch around the loads
    if constexpr (LISTS == 1) {
      m[0][j] = in ? bm_word(a, b, flags, nbits, at) : 0ull;
    } else {
      const unsigned long long valid = !in ? 0ull : nbits - at * 64 < 64 ? (1ull << (nbits - at * 64)) - 1ull : ~0ull;
      const unsigned long long wa = a[at], wb = b[at];
      m[0][j] = wa & ~wb & valid;
      m[1][j] = wb & ~wa & valid;
    }
  }
  // (a chunk behind the last word has a count of zero)
  uint32_t front[LISTS], sum[LISTS], own[LISTS], scanned[LISTS], all[LISTS];
#pragma unroll
  for (int l = 0; l < LISTS; ++l) {
    const uint32_t *counts = list[l].ws->base;
    scanned[l] = list[l].ws->scanned;
    all[l] = list[l].ws->total;
    own[l] = counts[chunk];
    front[l] = sum[l] = 0;
#pragma unroll
    for (uint32_t q = 0; q < kSmallStrip / kWave; ++q) {
      const uint32_t c = q * kWave + lane;
      const uint32_t n = counts[strip + min(c, gridDim.x - 1)];
      if (c < gridDim.x) sum[l] += n;
      if (c < blockIdx.x) front[l] += n;
    }
  }
#pragma unroll
  for (int l = 0; l < LISTS; ++l) {
    front[l] = wave_sum(front[l]);
    sum[l] = wave_sum(sum[l]);
    if (lane == 0) part[l][wv] = sum[l];
  }
  __syncthreads();
#pragma unroll
  for (int l = 0; l < LISTS; ++l) {
    const uint32_t others = lane < waves ? part[l][lane] : 0u;
    uint32_t pos = front[l] + wave_sum(lane < wv ? others : 0u);
    if (scanned[l]) pos = own[l];
    if (LISTS == 1 && total_host && blockIdx.x == 0 && wv == 0) {
      const uint32_t total = scanned[l] ? all[l] : wave_sum(others);
      if (lane == 0) *total_host = total;
    }
#pragma unroll
    for (uint64_t j = 0; j < kSmallBlocks; ++j) {
      if (__ballot(m[l][j] != 0ull) == 0ull) continue;
      const uint32_t incl = set_bits_upto(m[l][j]);
      const uint32_t n_set = (uint32_t)__builtin_amdgcn_readlane((int)incl, kWave - 1);
      if (pos < list[l].max_out)
        emit_word(m[l][j], incl, n_set, pos, w_first + j * kWave, lane, list[l].out, list[l].max_out);
      pos += n_set;
    }
  }
}

__global__ __launch_bounds__(kBlock) void bitmap_update_kernel(unsigned long long *bitmap, uint64_t nbits,
                                                               const uint32_t *idx, size_t n, int set,
                                                               uint32_t *status) {
  for (size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (size_t)gridDim.x * kBlock) {
    const uint32_t p = idx[i];
    if (p >= nbits) {
      atomicOr(status, UGK_ST_KEY_OUT_OF_RANGE);
      continue;
    }
    const unsigned long long bit = 1ull << (p & 63);
    if (set) atomicOr(bitmap + (p >> 6), bit);
    else atomicAnd(bitmap + (p >> 6), ~bit);
  }
}

// every bit up to and including position *last_pos: what taking the lowest free slots, the last of them *last_pos,
// does to the slot bitmap, as a pass over the bitmap instead of one atomic per slot on words 64 neighbours share
__global__ __launch_bounds__(kBlock) void bitmap_set_through_kernel(unsigned long long *bitmap, uint64_t nbits,
                                                                    const uint32_t *last_pos, uint32_t *status) {
  const uint64_t last = *last_pos;
  if (last >= nbits) {
    if (blockIdx.x == 0 && threadIdx.x == 0) atomicOr(status, UGK_ST_KEY_OUT_OF_RANGE);
    return;
  }
  const uint64_t wl = last >> 6;
  for (uint64_t w = (uint64_t)blockIdx.x * kBlock + threadIdx.x; w <= wl; w += (uint64_t)gridDim.x * kBlock) {
    if (w < wl) bitmap[w] = ~0ull;
    else bitmap[w] |= (last & 63) == 63 ? ~0ull : (1ull << ((last & 63) + 1)) - 1ull;
  }
}

__global__ __launch_bounds__(kBlock) void rows_to_keys_kernel(const uint32_t *rows, size_t n, uint64_t mul,
                                                              uint64_t mask, long long *keys) {
  for (size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (size_t)gridDim.x * kBlock)
    keys[i] = (long long)(((uint64_t)rows[i] * mul) & mask);
}

}  // namespace
// an empty launch: what it costs is the load of this file's code object onto the device (see ugk_preload_kernels)
namespace {
__global__ void preload_refresh_kernel() {}
}  // namespace
void preload_refresh(hipStream_t stream) { hipLaunchKernelGGL(preload_refresh_kernel, dim3(1), dim3(1), 0, stream); }
}  // namespace ugk

using namespace ugk;

extern "C" {

size_t ugk_rank_workspace_bytes(void) { return sizeof(RankWs); }

int ugk_rank_place(uint32_t *counts_dev, uint64_t num_rows, uint64_t k, void *ws_dev, uint64_t *in_new_dev,
                   uint64_t *scratch_bitmap_dev, uint64_t *observed_dev, int reset_counts, void *stream) {
  return ugk_rank_place_keep(counts_dev, num_rows, k, ws_dev, in_new_dev, scratch_bitmap_dev, observed_dev, nullptr,
                             reset_counts, stream);
}

int ugk_rank_place_keep(uint32_t *counts_dev, uint64_t num_rows, uint64_t k, void *ws_dev, uint64_t *in_new_dev,
                        uint64_t *scratch_bitmap_dev, uint64_t *observed_dev, const uint64_t *keep_dev,
                        int reset_counts, void *stream) {
  UGK_REQUIRE(counts_dev && ws_dev && in_new_dev && scratch_bitmap_dev, "ugk_rank_place: null pointer");
  UGK_REQUIRE(keep_dev != in_new_dev && keep_dev != scratch_bitmap_dev,
              "ugk_rank_place_keep: the keep bitmap is one of the output bitmaps");
  UGK_REQUIRE(num_rows > 0 && num_rows < 0xffffffffull, "ugk_rank_place: %llu rows do not fit 32 bits",
              (unsigned long long)num_rows);
  UGK_REQUIRE((uintptr_t)counts_dev % 16 == 0 && (uintptr_t)ws_dev % 8 == 0, "ugk_rank_place: misaligned buffer");
  RankWs *ws = static_cast<RankWs *>(ws_dev);
  hipStream_t st = as_stream(stream);
  unsigned long long *in_new = reinterpret_cast<unsigned long long *>(in_new_dev);
  unsigned long long *eq = reinterpret_cast<unsigned long long *>(scratch_bitmap_dev);
  unsigned long long *observed = reinterpret_cast<unsigned long long *>(observed_dev);
  const unsigned long long *keep = reinterpret_cast<const unsigned long long *>(keep_dev);
  const unsigned long long *none = nullptr;
  const RankWs *no_gate = nullptr;
  const uint64_t n_words = (num_rows + 63) / 64;
  if (k == 0 || k >= num_rows) {  // no row, or every row
    const unsigned grid = clamp_grid(((reset_counts ? num_rows : n_words) + kBlock - 1) / kBlock, 0);
    hipLaunchKernelGGL(rank_fill_kernel, dim3(grid), dim3(kBlock), 0, st, counts_dev, num_rows, in_new,
                       k == 0 ? 0 : 1, reset_counts, ws, observed);
    UGK_HIP(hipGetLastError());
    return 0;
  }
  hipLaunchKernelGGL(rank_init_kernel, dim3(1), dim3(kBlock), 0, st, ws, (unsigned long long)k);
  const uint64_t per_chunk = bm_words_per_chunk(n_words);
  const unsigned bm_grid = clamp_grid((kBmChunks + (kBlock / kWave) - 1) / (kBlock / kWave), (unsigned)cu_count() * 8u);
  const unsigned word_grid = clamp_grid((n_words + kBlock - 1) / kBlock, 0);
  if (observed) {
    hipLaunchKernelGGL(bitmap_count_kernel, dim3(bm_grid), dim3(kBlock), 0, st, observed, none, 0, num_rows, per_chunk,
                       &ws->bm, no_gate);
    hipLaunchKernelGGL(bitmap_scan_kernel, dim3(1), dim3(kScanBlock), 0, st, &ws->bm, (uint32_t *)nullptr, no_gate);
    hipLaunchKernelGGL(rank_decide_kernel, dim3(1), dim3(1), 0, st, ws);
    hipLaunchKernelGGL(rank_split_bitmap_kernel, dim3(word_grid), dim3(kBlock), 0, st, counts_dev, num_rows, ws,
                       observed, in_new, eq, reset_counts);
  }
  // a few long workgroups: every workgroup ends with a flush of its histogram into the shared one
  const unsigned hist_grid = clamp_grid((num_rows / 4 + kBlock - 1) / kBlock, (unsigned)cu_count() * 8u);
  // counters that are kept: the first pass splits by the last placement's T on its way (see rank_hist_split_kernel)
  const int with_split = reset_counts ? 0 : 1;
  if (with_split) {
    // twice the workgroups of the plain histogram pass: 474 against 508 us per placement at 500 M rows (557 with half,
    // 487 with eight times as many)
    const unsigned grid = clamp_grid((num_rows / 4 + kBlock - 1) / kBlock, (unsigned)cu_count() * 16u);
    hipLaunchKernelGGL(rank_hist_split_kernel, dim3(grid), dim3(kBlock), 0, st, counts_dev, num_rows, ws, in_new, eq);
  }
  else
    hipLaunchKernelGGL(rank_hist_kernel, dim3(hist_grid), dim3(kBlock), 0, st, counts_dev, num_rows, ws, 0, 0, 11);
  hipLaunchKernelGGL(rank_pick_kernel, dim3(1), dim3(kBlock), 0, st, ws, 0, 0, with_split);
  for (int p = 0; p < kCountPasses; ++p) {  // leave at once when the first pass settled T
    hipLaunchKernelGGL(rank_hist_kernel, dim3(hist_grid), dim3(kBlock), 0, st, counts_dev, num_rows, ws, 1,
                       kPassShift[p], kPassBits[p]);
    hipLaunchKernelGGL(rank_pick_kernel, dim3(1), dim3(kBlock), 0, st, ws, 1, kPassShift[p], 0);
  }
  const unsigned split_grid =
      clamp_grid((n_words + kMarkWords * (kBlock / kWave) - 1) / (kMarkWords * (kBlock / kWave)), 0);
  hipLaunchKernelGGL(rank_split_kernel, dim3(split_grid), dim3(kBlock), 0, st, counts_dev, num_rows, ws, in_new, eq,
                     reset_counts);
  if (keep) {
    // rows that tie at the K-th count: the kept ones first.  The second count runs only when they do not suffice.
    hipLaunchKernelGGL(bitmap_count_kernel, dim3(bm_grid), dim3(kBlock), 0, st, eq, keep, kBmAndB, num_rows, per_chunk,
                       &ws->bm, no_gate);
    hipLaunchKernelGGL(bitmap_scan_kernel, dim3(1), dim3(kScanBlock), 0, st, &ws->bm, (uint32_t *)nullptr, no_gate);
    hipLaunchKernelGGL(rank_keep_decide_kernel, dim3(1), dim3(1), 0, st, ws);
    hipLaunchKernelGGL(bitmap_count_kernel, dim3(bm_grid), dim3(kBlock), 0, st, eq, keep, 0, num_rows, per_chunk,
                       &ws->bm, (const RankWs *)ws);
    hipLaunchKernelGGL(bitmap_scan_kernel, dim3(1), dim3(kScanBlock), 0, st, &ws->bm, (uint32_t *)nullptr,
                       (const RankWs *)ws);
  } else {
    hipLaunchKernelGGL(bitmap_count_kernel, dim3(bm_grid), dim3(kBlock), 0, st, eq, none, 0, num_rows, per_chunk,
                       &ws->bm, no_gate);
    hipLaunchKernelGGL(bitmap_scan_kernel, dim3(1), dim3(kScanBlock), 0, st, &ws->bm, (uint32_t *)nullptr, no_gate);
  }
  hipLaunchKernelGGL(rank_locate_kernel, dim3(1), dim3(kBlock), 0, st, ws, eq, keep, num_rows, per_chunk);
  hipLaunchKernelGGL(rank_combine_kernel, dim3(word_grid), dim3(kBlock), 0, st, ws, in_new, eq, keep, n_words,
                     reset_counts ? observed : (unsigned long long *)nullptr);
  UGK_HIP(hipGetLastError());
  return 0;
}

int ugk_rank_place_observed(uint32_t *counts_dev, uint64_t num_rows, uint64_t k, void *ws_dev, uint64_t *in_new_dev,
                            uint64_t *observed_dev, int reset_counts, const uint64_t *cached_dev, void *evict_ws_dev,
                            void *insert_ws_dev, uint32_t *totals_host, uint32_t *status_dev, void *stream) {
  return ugk_rank_place_observed_ticket(counts_dev, num_rows, k, ws_dev, in_new_dev, observed_dev, reset_counts, cached_dev,
                                        evict_ws_dev, insert_ws_dev, totals_host, status_dev, 0, stream);
}

int ugk_rank_place_observed_ticket(uint32_t *counts_dev, uint64_t num_rows, uint64_t k, void *ws_dev,
                                   uint64_t *in_new_dev, uint64_t *observed_dev, int reset_counts,
                                   const uint64_t *cached_dev, void *evict_ws_dev, void *insert_ws_dev,
                                   uint32_t *totals_host, uint32_t *status_dev, uint32_t ticket, void *stream) {
  UGK_REQUIRE(ticket == 0 || cached_dev, "ugk_rank_place_observed: a ticket comes with the counts of what changes");
  UGK_REQUIRE(ws_dev && in_new_dev && observed_dev && status_dev, "ugk_rank_place_observed: null pointer");
  UGK_REQUIRE(counts_dev || !reset_counts, "ugk_rank_place_observed: counters to reset, but no counters");
  UGK_REQUIRE(num_rows > 0 && num_rows < 0xffffffffull, "ugk_rank_place_observed: %llu rows do not fit 32 bits",
              (unsigned long long)num_rows);
  UGK_REQUIRE(k > 0 && k < num_rows, "ugk_rank_place_observed: k = %llu is not inside (0, %llu)",
              (unsigned long long)k, (unsigned long long)num_rows);
  UGK_REQUIRE(in_new_dev != observed_dev && cached_dev != in_new_dev,
              "ugk_rank_place_observed: the output bitmap is one of the input bitmaps");
  UGK_REQUIRE(!cached_dev || (evict_ws_dev && insert_ws_dev && totals_host && evict_ws_dev != insert_ws_dev),
              "ugk_rank_place_observed: counting what changes needs two workspaces and the host words");
  RankWs *ws = static_cast<RankWs *>(ws_dev);
  hipStream_t st = as_stream(stream);
  unsigned long long *observed = reinterpret_cast<unsigned long long *>(observed_dev);
  const unsigned long long *none = nullptr;
  const RankWs *no_gate = nullptr;
  const uint64_t n_words = (num_rows + 63) / 64;
  const uint64_t per_chunk = bm_words_per_chunk(n_words);
  const unsigned bm_grid = clamp_grid((kBmChunks + (kBlock / kWave) - 1) / (kBlock / kWave), (unsigned)cu_count() * 8u);
  hipLaunchKernelGGL(bitmap_count_kernel, dim3(bm_grid), dim3(kBlock), 0, st, observed, none, 0, num_rows, per_chunk,
                     &ws->bm, no_gate);
  hipLaunchKernelGGL(rank_locate_unobserved_kernel, dim3(1), dim3(kScanBlock), 0, st, ws, observed, num_rows, per_chunk,
                     (unsigned long long)k, status_dev, totals_host ? totals_host + 2 : (uint32_t *)nullptr);
  // the emit pass of longer bitmaps wants the chunk counts scanned; the ticket is left by whichever launch is the last one
  const bool scan = cached_dev && num_rows > kSmallBits;
  BmWs *evict_ws = static_cast<BmWs *>(evict_ws_dev), *insert_ws = static_cast<BmWs *>(insert_ws_dev);
  hipLaunchKernelGGL(rank_combine_observed_kernel, dim3(bm_grid), dim3(kBlock), 0, st, counts_dev, num_rows, per_chunk,
                     ws, observed, reinterpret_cast<unsigned long long *>(in_new_dev),
                     reinterpret_cast<const unsigned long long *>(cached_dev), evict_ws, insert_ws, reset_counts,
                     totals_host, scan ? 0u : ticket);
  if (scan && ticket)
    hipLaunchKernelGGL(bitmap_scan2_ticket_kernel, dim3(2), dim3(kScanBlock), 0, st, evict_ws, insert_ws, ws,
                       totals_host + 3, ticket);
  else if (scan)
    hipLaunchKernelGGL(bitmap_scan2_kernel, dim3(2), dim3(kScanBlock), 0, st, evict_ws, insert_ws, (uint32_t *)nullptr);
  UGK_HIP(hipGetLastError());
  return 0;
}

int ugk_rank_threshold(const void *ws_dev, uint64_t *threshold_host, void *stream) {
  UGK_REQUIRE(ws_dev && threshold_host, "ugk_rank_threshold: null pointer");
  UGK_HIP(hipMemcpyAsync(threshold_host, ws_dev, sizeof(uint64_t), hipMemcpyDeviceToHost, as_stream(stream)));
  UGK_HIP(hipStreamSynchronize(as_stream(stream)));
  return 0;
}

size_t ugk_bitmap_workspace_bytes(void) { return sizeof(BmWs); }

int ugk_bitmap_count(const uint64_t *a_dev, const uint64_t *b_dev, int invert_a, uint64_t nbits, void *ws_dev,
                     uint32_t *total_host, void *stream) {
  UGK_REQUIRE(a_dev && ws_dev, "ugk_bitmap_count: null pointer");
  UGK_REQUIRE(nbits > 0 && nbits <= 0xffffffffull, "ugk_bitmap_count: %llu bits do not fit 32-bit positions",
              (unsigned long long)nbits);
  const uint64_t n_words = (nbits + 63) / 64;
  const uint64_t per_chunk = bm_words_per_chunk(n_words);
  // every chunk slot is written (the empty ones with zero), so the scan needs no clearing in front of it
  const unsigned grid = clamp_grid((kBmChunks + (kBlock / kWave) - 1) / (kBlock / kWave), (unsigned)cu_count() * 8u);
  hipLaunchKernelGGL(bitmap_count_kernel, dim3(grid), dim3(kBlock), 0, as_stream(stream),
                     reinterpret_cast<const unsigned long long *>(a_dev),
                     reinterpret_cast<const unsigned long long *>(b_dev), invert_a ? kBmInvertA : 0, nbits,
                     per_chunk, static_cast<BmWs *>(ws_dev), (const RankWs *)nullptr);
  if (total_host || nbits > kSmallBits)
    hipLaunchKernelGGL(bitmap_scan_kernel, dim3(1), dim3(kScanBlock), 0, as_stream(stream), static_cast<BmWs *>(ws_dev),
                       total_host, (const RankWs *)nullptr);
  UGK_HIP(hipGetLastError());
  return 0;
}

int ugk_bitmap_count_diff(const uint64_t *a_dev, const uint64_t *b_dev, uint64_t nbits, void *ws_ab_dev,
                          void *ws_ba_dev, uint32_t *totals_host, void *stream) {
  UGK_REQUIRE(a_dev && b_dev && ws_ab_dev && ws_ba_dev && ws_ab_dev != ws_ba_dev,
              "ugk_bitmap_count_diff: null pointer, or one workspace for both counts");
  UGK_REQUIRE(nbits > 0 && nbits <= 0xffffffffull, "ugk_bitmap_count_diff: %llu bits do not fit 32-bit positions",
              (unsigned long long)nbits);
  const uint64_t per_chunk = bm_words_per_chunk((nbits + 63) / 64);
  const unsigned grid = clamp_grid((kBmChunks + (kBlock / kWave) - 1) / (kBlock / kWave), (unsigned)cu_count() * 8u);
  hipLaunchKernelGGL(bitmap_count_diff_kernel, dim3(grid), dim3(kBlock), 0, as_stream(stream),
                     reinterpret_cast<const unsigned long long *>(a_dev),
                     reinterpret_cast<const unsigned long long *>(b_dev), nbits, per_chunk,
                     static_cast<BmWs *>(ws_ab_dev), static_cast<BmWs *>(ws_ba_dev));
  hipLaunchKernelGGL(bitmap_scan2_kernel, dim3(2), dim3(kScanBlock), 0, as_stream(stream), static_cast<BmWs *>(ws_ab_dev),
                     static_cast<BmWs *>(ws_ba_dev), totals_host);
  UGK_HIP(hipGetLastError());
  return 0;
}

int ugk_bitmap_emit(const uint64_t *a_dev, const uint64_t *b_dev, int invert_a, uint64_t nbits, const void *ws_dev,
                    uint32_t *out_dev, uint64_t max_out, void *stream) {
  return ugk_bitmap_emit_counted(a_dev, b_dev, invert_a, nbits, ws_dev, out_dev, max_out, nullptr, stream);
}

int ugk_bitmap_emit_counted(const uint64_t *a_dev, const uint64_t *b_dev, int invert_a, uint64_t nbits, const void *ws_dev,
                            uint32_t *out_dev, uint64_t max_out, uint32_t *total_host, void *stream) {
  UGK_REQUIRE(a_dev && ws_dev, "ugk_bitmap_emit: null pointer");
  UGK_REQUIRE(nbits > 0 && nbits <= 0xffffffffull, "ugk_bitmap_emit: %llu bits do not fit 32-bit positions",
              (unsigned long long)nbits);
  if (max_out == 0 && !total_host) return 0;
  UGK_REQUIRE(out_dev || max_out == 0, "ugk_bitmap_emit: null output list");
  const uint64_t n_words = (nbits + 63) / 64;
  const uint64_t per_chunk = bm_words_per_chunk(n_words);
  if (nbits <= kSmallBits) {
    const SmallGrid grid(nbits, per_chunk);
    hipLaunchKernelGGL((bitmap_emit_small_kernel<1>), dim3(grid.groups), dim3(grid.threads), 0, as_stream(stream),
                       reinterpret_cast<const unsigned long long *>(a_dev),
                       reinterpret_cast<const unsigned long long *>(b_dev), invert_a ? kBmInvertA : 0, nbits, per_chunk,
                       BmList{static_cast<const BmWs *>(ws_dev), out_dev, max_out}, BmList{nullptr, nullptr, 0}, total_host);
    UGK_HIP(hipGetLastError());
    return 0;
  }
  const uint64_t n_blocks = (n_words + kWave - 1) / kWave;
  const unsigned grid = clamp_grid((n_blocks + (kBlock / kWave) - 1) / (kBlock / kWave), 0);
  hipLaunchKernelGGL(bitmap_emit_kernel, dim3(grid), dim3(kBlock), 0, as_stream(stream),
                     reinterpret_cast<const unsigned long long *>(a_dev),
                     reinterpret_cast<const unsigned long long *>(b_dev), invert_a ? kBmInvertA : 0, nbits,
                     per_chunk, static_cast<const BmWs *>(ws_dev), out_dev, max_out, total_host);
  UGK_HIP(hipGetLastError());
  return 0;
}

int ugk_bitmap_emit_diff(const uint64_t *a_dev, const uint64_t *b_dev, uint64_t nbits, const void *ws_ab_dev,
                         const void *ws_ba_dev, uint32_t *out_ab_dev, uint64_t max_ab, uint32_t *out_ba_dev,
                         uint64_t max_ba, void *stream) {
  UGK_REQUIRE(a_dev && b_dev && ws_ab_dev && ws_ba_dev, "ugk_bitmap_emit_diff: null pointer");
  UGK_REQUIRE(nbits > 0 && nbits <= 0xffffffffull, "ugk_bitmap_emit_diff: %llu bits do not fit 32-bit positions",
              (unsigned long long)nbits);
  if (max_ab == 0 && max_ba == 0) return 0;
  UGK_REQUIRE((out_ab_dev || max_ab == 0) && (out_ba_dev || max_ba == 0), "ugk_bitmap_emit_diff: null output list");
  const uint64_t n_words = (nbits + 63) / 64;
  const uint64_t per_chunk = bm_words_per_chunk(n_words);
  if (nbits <= kSmallBits) {
    const SmallGrid grid(nbits, per_chunk);
    hipLaunchKernelGGL((bitmap_emit_small_kernel<2>), dim3(grid.groups), dim3(grid.threads), 0, as_stream(stream),
                       reinterpret_cast<const unsigned long long *>(a_dev),
                       reinterpret_cast<const unsigned long long *>(b_dev), 0, nbits, per_chunk,
                       BmList{static_cast<const BmWs *>(ws_ab_dev), out_ab_dev, max_ab},
                       BmList{static_cast<const BmWs *>(ws_ba_dev), out_ba_dev, max_ba}, (uint32_t *)nullptr);
    UGK_HIP(hipGetLastError());
    return 0;
  }
  const uint64_t n_groups = ((n_words + kWave - 1) / kWave + kDiffBlocks - 1) / kDiffBlocks;
  const unsigned grid = clamp_grid((n_groups + (kBlock / kWave) - 1) / (kBlock / kWave), 0);
  hipLaunchKernelGGL(bitmap_emit_diff_kernel, dim3(grid), dim3(kBlock), 0, as_stream(stream),
                     reinterpret_cast<const unsigned long long *>(a_dev),
                     reinterpret_cast<const unsigned long long *>(b_dev), nbits, per_chunk,
                     static_cast<const BmWs *>(ws_ab_dev), static_cast<const BmWs *>(ws_ba_dev), out_ab_dev, max_ab,
                     out_ba_dev, max_ba);
  UGK_HIP(hipGetLastError());
  return 0;
}

int ugk_bitmap_update(uint64_t *bitmap_dev, uint64_t nbits, const uint32_t *idx_dev, size_t n, int set,
                      uint32_t *status_dev, void *stream) {
  if (n == 0) return 0;
  UGK_REQUIRE(bitmap_dev && idx_dev && status_dev, "ugk_bitmap_update: null pointer");
  const unsigned grid = clamp_grid((n + kBlock - 1) / kBlock, 0);
  hipLaunchKernelGGL(bitmap_update_kernel, dim3(grid), dim3(kBlock), 0, as_stream(stream),
                     reinterpret_cast<unsigned long long *>(bitmap_dev), nbits, idx_dev, n, set, status_dev);
  UGK_HIP(hipGetLastError());
  return 0;
}

int ugk_bitmap_set_through(uint64_t *bitmap_dev, uint64_t nbits, const uint32_t *last_pos_dev, uint32_t *status_dev,
                           void *stream) {
  UGK_REQUIRE(bitmap_dev && last_pos_dev && status_dev, "ugk_bitmap_set_through: null pointer");
  UGK_REQUIRE(nbits > 0, "ugk_bitmap_set_through: empty bitmap");
  const unsigned grid = clamp_grid(((nbits + 63) / 64 + kBlock - 1) / kBlock, 0);
  hipLaunchKernelGGL(bitmap_set_through_kernel, dim3(grid), dim3(kBlock), 0, as_stream(stream),
                     reinterpret_cast<unsigned long long *>(bitmap_dev), nbits, last_pos_dev, status_dev);
  UGK_HIP(hipGetLastError());
  return 0;
}

int ugk_rows_to_keys(const uint32_t *rows_dev, size_t n, uint64_t mul, uint64_t mask, int64_t *keys_out_dev,
                     void *stream) {
  if (n == 0) return 0;
  UGK_REQUIRE(rows_dev && keys_out_dev, "ugk_rows_to_keys: null pointer");
  UGK_REQUIRE(mul & 1ull, "ugk_rows_to_keys: the key multiplier must be odd");
  const unsigned grid = clamp_grid((n + kBlock - 1) / kBlock, 0);
  hipLaunchKernelGGL(rows_to_keys_kernel, dim3(grid), dim3(kBlock), 0, as_stream(stream), rows_dev, n, mul, mask,
                     reinterpret_cast<long long *>(keys_out_dev));
  UGK_HIP(hipGetLastError());
  return 0;
}

}  // extern "C"
